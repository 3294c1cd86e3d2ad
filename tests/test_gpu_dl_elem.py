"""The direct-to-LDS kernel with element loads (32-bit problems whose rows or
operands are not whole 16-byte vectors), at the edges of its tiles, k-tiles
and resolve windows, against the oracle bit for bit."""
import numpy as np
import pytest

from oracle import oracle
from tests import tg_cases as tc
from tests.test_gpu_nan import assert_nan_exact, nan_inputs
from tests.test_gpu_parity import _strided_batched, assert_exact, gpu_gemm

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# (m, n, k): a last k-tile of 1, 2, 3, 31 and 32 k, a last chunk of 1, 2, 3
# and 5 k (windows that shift back over K), one row or column past a tile,
# a last column group of 1, 2 and 3 columns; K slices of unequal length (17
# and 18 k-tiles) and a fourth slice left empty (9 k-tiles).
SHAPES = [(513, 511, 97), (449, 577, 130), (640, 450, 99), (576, 514, 255), (511, 513, 160),
          (577, 449, 197), (512, 515, 511), (515, 512, 514), (513, 513, 549), (513, 512, 257),
          (512, 577, 288), (449, 451, 1027), (512, 512, 260)]


@pytest.mark.parametrize("dt", ["f32", "i32"])
@pytest.mark.parametrize("m,n,k", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
def test_element_loads_edges(dt, m, n, k):
    from tropical_gemm import _native as nat

    rng = np.random.default_rng(m + 3 * n + 7 * k)
    dtype = tc.NP_DTYPES[dt]
    for sr in tc.SEMIRINGS:
        # Up to 256 tiles, K from 256 runs in two (1024: four) slices, value-only in
        # four.
        cut = k >= 256
        keys = dt == "i32" and sr != "maxmul" and k <= 160  # tg_gemm_kresg
        assert nat.gemm_plan(sr, dt, m, n, k, True) == (
            "kresg" if keys else "dl_elem_cl8" + (" slices 4" if k >= 1024 else " slices 2" if cut else ""))
        assert nat.gemm_plan(sr, dt, m, n, k, False) == "dl_elem" + (" slices 4" if cut else "")
        # Ties across k, and winners in the last, partial window.
        lo, hi = (1, 50) if sr == "maxmul" else (-50, 50)
        a = rng.integers(lo, hi, size=(m, k))
        b = rng.integers(lo, hi, size=(k, n))
        a[::3, k - 1] = 60 if sr != "minplus" else -60
        b[k - 1, ::5] = 60 if sr != "minplus" else -60
        a[1::7, k - 2] = a[1::7, k - 1]
        b[k - 6, ::2] += 6
        a, b = a.astype(dtype), b.astype(dtype)
        print(f"[case] element loads {sr} {dt} {m}x{n}x{k}", flush=True)
        c_ref, am_ref = oracle.gemm(sr, a, b)
        c, am = gpu_gemm(sr, a, b, True)
        assert_exact(c, am, c_ref, am_ref)
        c, _ = gpu_gemm(sr, a, b, False)
        np.testing.assert_array_equal(c, c_ref)


@pytest.mark.parametrize("sr,m,n,k,with_argmax,plan", [
    ("maxplus", 1473, 1501, 517, True, "dl_elem_cl16"),
    ("minplus", 1090, 1201, 515, True, "dl_elem_cl8 slices 2"),
    ("maxplus", 1090, 1200, 515, False, "dl_elem slices 2"),
    ("maxmul", 1200, 1200, 700, True, "dl_elem_cl8 slices 2"),  # aligned
    ("minplus", 2100, 2101, 259, False, "dl_elem"),
])
def test_element_loads_more_tiles(sr, m, n, k, with_argmax, plan):
    from tropical_gemm import _native as nat

    rng = np.random.default_rng(m + k)
    a = rng.integers(1, 60, size=(m, k)).astype(np.float32)
    b = rng.integers(1, 60, size=(k, n)).astype(np.float32)
    rows = np.unique(np.concatenate([np.arange(0, m, 41), [63, 64, m - 1]]))
    c_ref, am_ref = oracle.gemm(sr, a[rows], b)
    assert nat.gemm_plan(sr, "f32", m, n, k, with_argmax) == plan
    print(f"[case] element loads {plan} {sr} {m}x{n}x{k}", flush=True)
    c, am = gpu_gemm(sr, a, b, with_argmax)
    assert_exact(c[rows], am[rows] if with_argmax else None, c_ref, am_ref if with_argmax else None)


@pytest.mark.parametrize("k", [131, 515])
@pytest.mark.parametrize("sr", tc.SEMIRINGS)
def test_element_loads_nan_rule_and_layouts(sr, k):
    m, n = 513, 515
    a, b = nan_inputs(sr, np.float32, m, n, k, seed=3)
    c_ref, am_ref = oracle.gemm(sr, a, b)
    for layout in ("row", "col"):
        for with_argmax in (True, False):
            print(f"[case] element loads NaN {sr} {layout} argmax={with_argmax}", flush=True)
            c, am = gpu_gemm(sr, a, b, with_argmax, layout=layout)
            assert_nan_exact(c, am, c_ref, am_ref if with_argmax else None)


@pytest.mark.parametrize("dt", ["f32", "i32"])
def test_element_loads_misaligned_batches(dt):
    """Sizes that are whole vectors, batch strides that are not."""
    from tropical_gemm import _native as nat

    sr = "minplus" if dt == "f32" else "maxmul"  # i32 MinPlus: tg_gemm_kresg
    m, n, k = 320, 384, 160
    strides = (m * k + 1, k * n, m * n + 3)
    assert nat.gemm_plan(sr, dt, m, n, k, True, batch=3, strides=strides) == "dl_elem_cl8"
    rng = np.random.default_rng(12)
    items = [(tc.rng_matrix(rng, tc.NP_DTYPES[dt], (m, k), -1000, 1000),
              tc.rng_matrix(rng, tc.NP_DTYPES[dt], (k, n), -1000, 1000)) for _ in range(3)]
    print(f"[case] element loads misaligned batch {dt}", flush=True)
    for (x, y), (c, am) in zip(items, _strided_batched(sr, items, gap_a=1, gap_c=3)):
        assert_exact(c, am, *oracle.gemm(sr, x, y))


def test_short_k_without_workspace_keeps_the_exact_mode():
    """A workspace too small for B^T (the fixed scratch of tg_gemm_noalloc)
    leaves K up to 384 to the generic kernel's exact mode."""
    from tropical_gemm import _native as nat

    m, n, k = 513, 80001, 300
    assert nat.gemm_plan("maxplus", "f32", m, n, k, True).startswith("dl_elem_cl8")
    assert nat.gemm_plan("maxplus", "f32", m, n, k, True, workspace_bytes=64 << 20) == "tiles_exact"
