"""The k rows that the element loads of tg_gemm_dl and tg_gemm_dl64s read from
B stay inside it in a last, partial k-tile.  The kernels overwrite what such
rows bring, so no result shows a row past the end: the row rule
(csrc/tg_elem_rows.hpp, which both kernels use) is replayed on the host."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "tropical-gemm_amd", "csrc")

# One wave of a k-tile: `loads` instructions from its first row, `per_row` of
# them per row.
REPLAY = r"""
#include <cstdio>
#include "tg_elem_rows.hpp"

static int replay(const char* kernel, int bk, int waves, int loads, int per_row) {
    int bad = 0;
    for (int left = 1; left <= bk; ++left)
        for (int wave = 0; wave < waves; ++wave) {
            const int ins0 = wave * loads;
            int row = tg::elem_first_row(ins0 / per_row, left);
            for (int q = 0; q < loads; ++q) {
                const int own = (ins0 + q) / per_row;  // the row this load fills
                if (row < 0 || row >= left || (own < left && row != own)) {
                    std::printf("%s: left %d wave %d load %d reads row %d\n", kernel, left, wave, q, row);
                    ++bad;
                }
                if (q % per_row == per_row - 1 && tg::elem_steps(own, left)) ++row;
            }
        }
    return bad;
}

int main() {
    // 64 columns: a 32-bit row is one instruction of 64 lanes, a 64-bit row two.
    return replay("tg_gemm_dl", 32, 4, 8, 1) + replay("tg_gemm_dl64s", 16, 4, 8, 2) ? 1 : 0;
}
"""


def test_element_loads_read_rows_of_b_only(tmp_path):
    src, exe = tmp_path / "replay.cpp", tmp_path / "replay"
    src.write_text(REPLAY)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-I", CSRC, "-o", exe, src], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


def test_both_kernels_use_the_rule():
    for name in ("tg_gemm_dl.hpp", "tg_gemm_dl64s.hpp"):
        text = open(os.path.join(CSRC, name)).read()
        assert "elem_first_row(" in text and "elem_steps(" in text, name
