"""C ABI checks that need no GPU: the library loads, exports every symbol the
header declares, and rejects bad arguments before touching the device."""
import ctypes
import os
import re

import pytest

from tropical_gemm import _native as nat

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "tropical_gemm_hip.h")


def header_symbols():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(tg_[a-z0-9_]+)\s*\(", text)))


def test_library_built():
    assert os.path.exists(nat.library_path()), "run __graft_entry__.build() first"


def test_every_declared_symbol_is_exported_and_bound():
    lib = nat.load()
    declared = header_symbols()
    assert len(declared) >= 20
    for name in declared:
        assert hasattr(lib, name), f"{name} declared in the header but not exported"
    assert sorted(nat.SIGNATURES) == declared, "ctypes signatures out of sync with the header"


def test_version_and_status_strings():
    lib = nat.load()
    assert lib.tg_version() == 1
    assert lib.tg_status_string(nat.TG_ERR_DIMENSION_MISMATCH) == b"dimension mismatch"
    assert lib.tg_status_string(999) == b"unknown status"


def _gemm(**kw):
    args = dict(device=0, sr=0, dt=0, layout=0, A=1, B=1, C=1, argmax=None, m=4, n=4, k=4)
    args.update(kw)
    lib = nat.load()
    p = lambda v: None if v is None else ctypes.c_void_p(v)  # noqa: E731
    return lib.tg_gemm(args["device"], args["sr"], args["dt"], args["layout"], p(args["A"]),
                       p(args["B"]), p(args["C"]), p(args["argmax"]), args["m"], args["n"],
                       args["k"], None)


@pytest.mark.parametrize("kw,status,needle", [
    (dict(sr=7), nat.TG_ERR_INVALID_ARGUMENT, "unknown semiring"),
    (dict(dt=9), nat.TG_ERR_INVALID_ARGUMENT, "unknown dtype"),
    (dict(layout=3), nat.TG_ERR_INVALID_ARGUMENT, "unknown layout"),
    (dict(m=-1), nat.TG_ERR_DIMENSION_MISMATCH, "negative dimension"),
    (dict(k=2**31), nat.TG_ERR_DIMENSION_MISMATCH, "2^31-1"),
    (dict(C=None), nat.TG_ERR_INVALID_ARGUMENT, "C is NULL"),
    (dict(A=None), nat.TG_ERR_INVALID_ARGUMENT, "A or B is NULL"),
])
def test_gemm_argument_validation(kw, status, needle):
    assert _gemm(**kw) == status
    assert needle in nat.last_error()


def test_workspace_size_and_validation():
    lib = nat.load()
    assert lib.tg_gemm_workspace_size(0, 1, 64, 64, 64, 0) == 0
    need = lib.tg_gemm_workspace_size(0, 1, 100, 70, 33, 1)
    # B^T staging covers the wider of m and n: column-major calls swap the
    # operands, so the kernel's B is A (k x m).
    assert need >= 100 * 33 * 4 and need % 256 == 0
    assert lib.tg_gemm_workspace_size(0, 1, 70, 100, 33, 1) == need
    assert lib.tg_gemm_workspace_size(1, 2, 10, 10, 10, 1) >= 2 * 10 * 10 * 8
    rc = lib.tg_gemm_ws(0, 0, 0, 0, ctypes.c_void_p(16), ctypes.c_void_p(16), ctypes.c_void_p(16),
                        ctypes.c_void_p(16), 8, 8, 8, ctypes.c_void_p(256), 16, None)
    assert rc == nat.TG_ERR_INVALID_ARGUMENT and "workspace too small" in nat.last_error()


def test_batched_output_overlap_rejected():
    lib = nat.load()
    p = ctypes.c_void_p(4096)
    rc = lib.tg_gemm_strided_batched(0, 0, 0, 0, p, p, p, None, 3, 4, 4, 4, 16, 16, 8, None)
    assert rc == nat.TG_ERR_DIMENSION_MISMATCH and "overlap" in nat.last_error()


def test_backward_rejects_integer_dtype():
    lib = nat.load()
    p = ctypes.c_void_p(4096)
    rc = lib.tg_backward_a(0, nat.DTYPE["i32"], 0, p, p, p, 4, 4, 4, None)
    assert rc == nat.TG_ERR_UNSUPPORTED and "f32/f64" in nat.last_error()


def test_maxmul_backward_needs_operand():
    lib = nat.load()
    p = ctypes.c_void_p(4096)
    rc = lib.tg_maxmul_backward_a(0, 0, 0, p, p, None, p, 4, 4, 4, None)
    assert rc == nat.TG_ERR_INVALID_ARGUMENT and "other operand" in nat.last_error()


def test_hip_error_maps_reference_variants():
    e = nat.HipError(nat.TG_ERR_DIMENSION_MISMATCH, "A.cols (3) != B.rows (4)")
    assert e.kind == "DimensionMismatch" and "A.cols" in str(e)
    assert nat.HipError(nat.TG_ERR_NO_DEVICE, "x").kind == "NoDevice"


def test_python_layer_rejects_host_tensors():
    torch = pytest.importorskip("torch")
    from tropical_gemm import ops

    a = torch.zeros(2, 3)
    b = torch.zeros(3, 2)
    with pytest.raises(ValueError, match="device tensors"):
        ops.gemm("maxplus", a, b)
    with pytest.raises(ValueError, match="Expected 2D"):
        ops.gemm("maxplus", a, torch.zeros(3))
    with pytest.raises(ValueError, match="same dtype"):
        ops.gemm("maxplus", a, torch.zeros(3, 2, dtype=torch.float64))


# ---------------------------------------------------------------------------
# Dispatch and launch geometry (host logic; no device needed)
# ---------------------------------------------------------------------------

@pytest.mark.parametrize("sr,dt,m,n,k,argmax,expected", [
    ("maxplus", "f32", 4096, 4096, 4096, True, "dl_4x8_cl16"),       # P
    ("minplus", "f32", 4096, 4096, 4096, True, "dl_4x8_cl16"),       # C2
    ("maxmul", "f32", 8192, 4096, 2048, False, "dl_8x8_cl32"),       # C3
    ("maxplus", "i32", 262144, 128, 128, True, "kresw"),             # C4
    ("maxplus", "f32", 1024, 1024, 1024, True, "dl_4x4_cl8 slices 4"),  # C1
    ("maxplus", "f32", 65536, 8, 2048, True, "shortk"),              # M1 (m, k, n order below)
    ("maxplus", "f32", 67, 45, 40, True, "tiles_exact"),
    ("maxplus", "f64", 4096, 4096, 4096, True, "dl64_4x8_cl16"),
    ("maxplus", "f64", 64, 64, 640, True, "tiles_chunked"),
    ("maxplus", "f64", 4096, 4096, 4096, False, "dl64_4x8"),
    ("maxplus", "f64", 4096, 4096, 128, False, "tiles"),
    ("maxplus", "i64", 4096, 4096, 4096, True, "dl64s_4x4_cl16"),
    ("maxplus", "i64", 4096, 4096, 4096, False, "dl64s_4x4"),
    ("minplus", "i64", 4096, 4097, 48, False, "tiles"),
    ("minplus", "i64", 4096, 4096, 1 << 21, True, "tiles_chunked"),  # past the 16-bit chunk slots
    ("maxplus", "f32", 2048, 2048, 2048, False, "dl_4x8"),           # E1's GEMMs: one 64x64 round
    ("minplus", "f32", 2048, 4096, 1024, False, "dl_8x8_cl32"),      # one 128x128 round
    ("maxplus", "f32", 3072, 3072, 2048, False, "dl_4x4_cl32"),      # 1.125 rounds of 128x128
    ("maxplus", "f32", 1536, 2048, 2048, False, "dl_4x4_cl32"),      # 0.75 rounds of 64x64
])
def test_gemm_plan_names_the_configured_paths(sr, dt, m, n, k, argmax, expected):
    if expected == "shortk":
        m, n, k = 65536, 2048, 8
    assert nat.gemm_plan(sr, dt, m, n, k, argmax) == expected


def test_gemm_plan_rejects_what_the_call_rejects():
    assert nat.gemm_plan("maxplus", "f32", -1, 4, 4) == "invalid"
    assert nat.gemm_plan("maxplus", "f32", 0, 4, 4) == "none"


@pytest.mark.parametrize("dt", [0, 1])
@pytest.mark.parametrize("want_a", [1, 0])
@pytest.mark.parametrize("shape", [(1, 4096, 4096, 4096), (1, (1 << 24) + 1, 2, 3),
                                   (1, 3, (1 << 31) - 1, 3), (65535 * 4, 64, 64, 64),
                                   (1, 5, 9000, 100000), (3, 2, 2, 1 << 30)])
def test_backward_geometry_caps_every_launch_dimension(dt, want_a, shape):
    """Grid-stride kernels: whatever M, N, K and batch, the grid stays at or
    below 16384 workgroups of at most 512 threads, and LDS within the CU."""
    batch, m, n, k = shape
    lib = nat.load()
    for layout in (0, 1):
        plan = lib.tg_backward_plan(dt, layout, want_a, batch, m, n, k).decode()
        fields = dict(f.split("=") for f in plan.split()[2:])
        assert 1 <= int(fields["grid"]) <= 16384, plan
        assert 1 <= int(fields["waves"]) <= 8, plan
        assert int(fields["lds"]) <= 160 * 1024, plan
        elem = 4 if dt == 0 else 8
        if k * elem > 128 * 1024:
            assert "global" in plan, plan


def _noalloc_bytes(sr, dt, m, n, k, argmax, layout="row"):
    lib = nat.load()
    return lib.tg_gemm_noalloc_bytes(nat.SEMIRING[sr], nat.DTYPE[dt], nat.LAYOUT[layout], 256, 256,
                                     256, 256 if argmax else None, m, n, k)


def _round256(x):
    return -(-x // 256) * 256


@pytest.mark.parametrize("m,n,k,argmax", [(2048, 2048, 1024, True), (2048, 2048, 1024, False),
                                          (1024, 2048, 512, False), (2000, 4004, 544, True)])
def test_noalloc_bytes_cover_the_f64_direct_to_lds_workspace(m, n, k, argmax):
    """f64 problems on the direct-to-LDS kernel read B^T (argmax) and the
    operand classes (4 bytes per row of A and per column of B) from the
    workspace: tg_gemm_noalloc's scratch need counts both."""
    plan = nat.gemm_plan("maxplus", "f64", m, n, k, argmax, workspace_bytes=64 << 20)
    assert plan.startswith("dl64"), plan
    want = (_round256(k * n * 8) if argmax else 0) + _round256((m + n) * 4)
    assert _noalloc_bytes("maxplus", "f64", m, n, k, argmax) == want


def test_noalloc_bytes_of_other_paths():
    # 32-bit argmax on the direct-to-LDS kernel: B^T staging (row-major: k x n).
    assert nat.gemm_plan("maxplus", "f32", 4096, 4096, 4096, True) == "dl_4x8_cl16"
    assert _noalloc_bytes("maxplus", "f32", 4096, 4096, 4096, True) == 4096 * 4096 * 4
    # Split K: the value and index partials after the (here unused) B^T region.
    assert nat.gemm_plan("maxplus", "f32", 1024, 1024, 1024, True,
                         workspace_bytes=64 << 20) == "dl_4x4_cl8 slices 4"
    assert _noalloc_bytes("maxplus", "f32", 1024, 1024, 1024, True) == \
        1024 * 1024 * 4 + 2 * (2 * 1024 * 1024 * 4)
    # Paths without workspace, and empty products.
    assert _noalloc_bytes("maxplus", "f32", 4096, 4096, 4096, False) == 0
    assert _noalloc_bytes("maxplus", "i32", 262144, 128, 128, True) == 0
    assert _noalloc_bytes("maxplus", "f32", 0, 4, 4, True) == 0
    assert _noalloc_bytes("maxplus", "f32", -1, 4, 4, True) == 2**64 - 1


@pytest.mark.parametrize("dt,m,n,k,argmax", [
    ("f32", 1000, 1001, 300, True),   # element loads in tg_gemm; the exact tiles without a workspace
    ("i32", 1000, 1001, 300, True),
    ("f64", 1500, 1500, 512, True),   # 64 x 64 tiles with operand classes (and B^T)
    ("f64", 1000, 1000, 400, False),
    ("i64", 1000, 1000, 1000, True),  # 64 x 64 tiles with B^T
])
def test_noalloc_leaves_the_scratch_to_products_that_need_it(dt, m, n, k, argmax):
    """Calls that share no scratch may overlap on other streams and threads:
    a product that can run without one does."""
    assert nat.gemm_plan("maxmul", dt, m, n, k, argmax).startswith(("dl_elem", "dl64s"))
    assert _noalloc_bytes("maxmul", dt, m, n, k, argmax) == 0


def test_noalloc_scratch_where_no_kernel_is_without():
    # Argmax beyond the exact tiles' range, and value-only f64 that the 64 x 128
    # tiles (operand classes) can run.
    assert _noalloc_bytes("maxplus", "f32", 1000, 1001, 400, True) >= 1001 * 400 * 4
    assert _noalloc_bytes("maxplus", "i64", 500, 500, 2100, True) >= 500 * 2100 * 8
    assert _noalloc_bytes("maxplus", "f64", 1000, 1000, 520, True) >= 1000 * 520 * 8
    assert _noalloc_bytes("maxplus", "f64", 1024, 2048, 512, False) == (1024 + 2048) * 4


@pytest.mark.parametrize("dt,batch,m,n,k,argmax,allocates", [
    # Tiles without a workspace, where one would have to be allocated per call.
    ("f32", 16, 64, 1025, 97, True, False), ("f32", 16, 64, 1025, 300, True, True),
    ("f32", 500, 65, 65, 200, True, False), ("i32", 30, 129, 131, 255, True, False),
    ("i32", 64, 33, 65, 97, True, False), ("f64", 1, 1000, 1000, 257, False, False),
    ("f32", 1, 50000, 50, 384, True, False), ("f32", 1, 1000, 1001, 97, True, True),
    ("f64", 1, 1500, 1500, 300, True, False), ("f64", 1, 1500, 1500, 512, True, True),
    ("f64", 128, 128, 128, 512, True, False), ("f64", 1, 1000, 1000, 512, False, True),
    ("i64", 1, 1500, 1500, 188, True, False), ("i64", 1, 1500, 1500, 300, True, True),
    ("i64", 256, 64, 64, 1000, True, False), ("i64", 1, 1000, 1000, 1000, True, True),
    # Kernels that have to have one, and one that never does.
    ("f32", 1, 4096, 4096, 4096, True, True), ("f64", 4, 64, 64, 640, True, True),
    ("f32", 1, 4096, 4096, 4096, False, False),
])
def test_tg_gemm_allocates_a_workspace_where_it_pays(dt, batch, m, n, k, argmax, allocates):
    lib = nat.load()
    sr = "maxplus" if dt == "i64" else "maxmul"
    got = lib.tg_gemm_alloc_bytes(nat.SEMIRING[sr], nat.DTYPE[dt], nat.LAYOUT["row"], 256,
                                  256, 256, 256 if argmax else None, batch, m, n, k, m * k, k * n,
                                  m * n)
    full = lib.tg_gemm_workspace_size(nat.DTYPE[dt], batch, m, n, k, int(argmax))
    assert got == (full if allocates else 0)


@pytest.mark.parametrize("dt,batch,m,n,k,argmax,expected", [
    # Sizes either side of where the direct-to-LDS tiles outweigh their
    # prepasses and padding (expected: the start of the path's name).
    ("f64", 1, 1000, 1000, 300, True, "tiles_exact"), ("f64", 1, 1000, 1000, 400, True, "dl64s"),
    ("f64", 256, 64, 64, 512, True, "tiles_exact"), ("f64", 256, 64, 64, 513, True, "dl64s"),
    ("f64", 1, 8, 65536, 512, True, "tiles_exact"), ("f64", 1, 1500, 1500, 256, True, "dl64s"),
    ("f64", 64, 128, 128, 257, False, "tiles"), ("f64", 64, 128, 128, 320, False, "dl64s"),
    ("f64", 128, 128, 128, 449, True, "tiles_exact"), ("f64", 128, 128, 128, 449, False, "tiles"),
    ("f64", 128, 128, 128, 450, False, "dl64s"), ("f64", 1, 34, 47910, 321, False, "dl64s"),
    ("f64", 1, 1501, 1501, 256, True, "tiles_exact"), ("f64", 1, 1501, 1501, 257, True, "dl64s"),
    ("f64", 1, 512, 512, 256, False, "dl64s"),
    ("i64", 1, 1000, 1000, 300, True, "tiles_exact"), ("i64", 1, 1000, 1000, 513, True, "dl64s"),
    ("i64", 128, 128, 128, 256, True, "tiles_exact"), ("i64", 128, 128, 128, 257, True, "dl64s"),
    ("i64", 1, 34, 47910, 193, True, "tiles_exact"), ("i64", 1220, 64, 64, 257, True, "dl64s"),
    ("i64", 1024, 33, 33, 128, True, "tiles_exact"), ("i64", 1, 4096, 4096, 97, True, "dl64s"),
    ("i64", 1, 1500, 1500, 100, False, "tiles"), ("i64", 1, 1500, 1500, 128, False, "dl64s"),
    ("i64", 1, 1500, 1500, 129, False, "tiles"), ("i64", 1, 1500, 1500, 192, False, "dl64s"),
    ("i64", 1, 1000, 1000, 81, False, "tiles"), ("i64", 1, 1000, 1001, 64, False, "dl64s"),
    ("f32", 500, 65, 65, 97, True, "tiles_exact"), ("f32", 500, 65, 65, 200, True, "dl_elem"),
    ("f32", 1, 1000, 1001, 97, True, "dl_elem"), ("i32", 100, 100, 101, 97, True, "tiles_exact"),
    ("i32", 100, 100, 101, 130, True, "dl_elem"), ("f32", 1, 1000000, 2, 515, False, "tiles"),
    ("i32", 500, 65, 65, 100, False, "tiles"), ("i32", 1, 2001, 2001, 97, False, "tiles"),
    ("i32", 1260, 85, 31, 131, False, "tiles"), ("f32", 53, 214, 388, 115, True, "tiles_exact"), ("i32", 1, 700, 701, 100, False, "dl_elem"),
    ("f32", 1, 3, 100000, 97, True, "dl_elem"),
])
def test_gemm_plan_either_side_of_the_64x64_tiles(dt, batch, m, n, k, argmax, expected):
    # i32 by MaxMul (MaxPlus argmax runs on keys there), i64 by MaxPlus (MaxMul has
    # lines of its own).
    sr = "maxplus" if dt == "i64" else "maxmul"
    strides = (m * k, k * n, m * n)
    assert nat.gemm_plan(sr, dt, m, n, k, argmax, batch=batch, strides=strides).startswith(expected)


@pytest.mark.parametrize("batch,m,n,k,expected", [
    (1, 1500, 1500, 300, "tiles_exact"), (1, 1500, 1500, 301, "dl64s"),
    (1, 34, 47910, 1500, "tiles_exact"), (1, 34, 47910, 1502, "dl64s"),
    (1, 34, 47910, 1501, "tiles_exact"), (1, 100, 16383, 2500, "tiles_chunked"),
    (1, 1378, 1379, 400, "tiles_exact"), (1, 1378, 1379, 513, "dl64s"),
    (1, 1000, 1001, 512, "tiles_exact"), (1, 1000, 1001, 513, "dl64s"),
])
def test_gemm_plan_of_i64_maxmul_argmax(batch, m, n, k, expected):
    assert nat.gemm_plan("maxmul", "i64", m, n, k, True, batch=batch).startswith(expected)


def test_aligned_products_of_two_rounds_of_tiles():
    for dt, k, argmax, expected in (("f32", 256, True, "dl_elem"), ("i32", 256, True, "dl_4x4"),
                                    ("i32", 320, True, "dl_elem"), ("f32", 288, False, "dl_4x4"),
                                    ("f32", 320, False, "dl_elem")):
        assert nat.gemm_plan("maxplus", dt, 1408, 1408, k, argmax).startswith(expected)


def test_element_load_tiles_of_one_launch():
    # 2^24 tiles of 256 threads are 2^32, one more than a launch's dimension holds.
    m = 1 << 30
    assert nat.gemm_plan("maxplus", "f32", m, 5, 48, False) == "tiles"
    assert nat.gemm_plan("maxplus", "f32", m - 64, 5, 48, False) == "dl_elem"


def test_gemm_plan_of_unaligned_short_k_keys():
    for m, n, k, expected in ((524288, 33, 12, "tiles_exact"), (524288, 33, 20, "kresg"),
                              (65536, 33, 12, "kresg"), (524288, 48, 12, "kresg")):
        assert nat.gemm_plan("maxplus", "i32", m, n, k, True) == expected


@pytest.mark.parametrize("sr,dt,batch,m,n,k,argmax,few", [
    # Long K of few outputs: 32-bit K that splits over the whole chip goes there.
    ("maxplus", "f32", 1, 256, 256, 4096, False, True), ("maxplus", "f32", 1, 256, 256, 8192, False, False),
    ("maxplus", "f32", 1, 256, 256, 4096, True, True), ("maxplus", "i32", 1, 256, 256, 8192, True, False),
    ("maxplus", "f32", 1, 700, 700, 1024, False, False), ("maxplus", "f32", 1, 700, 700, 1024, True, True),
    ("maxplus", "f32", 1, 64, 64, 1 << 20, False, False), ("maxplus", "f32", 1, 64, 64, 32768, False, True),
    ("maxplus", "i32", 1, 64, 64, 65536, False, False), ("maxplus", "f32", 1, 64, 64, 65536, True, True),
    ("maxplus", "f32", 1, 16, 256, 32768, False, True), ("maxplus", "f32", 1, 16, 256, 65536, False, False),
    ("maxplus", "f32", 1, 16, 16, 65536, True, True), ("maxplus", "f32", 1, 16, 16, 262144, True, False),
    ("maxplus", "f32", 1, 64, 64, (1 << 20) - 1, False, True),  # K that does not split
    ("maxplus", "f64", 1, 64, 64, 1 << 20, True, True),
    ("maxplus", "f64", 256, 64, 64, 300, True, False), ("maxplus", "f64", 256, 65, 65, 300, True, True),
    ("maxplus", "f64", 1, 1000, 1000, 300, True, False), ("maxplus", "f64", 1, 700, 700, 300, True, True),
    ("maxplus", "f64", 1, 300, 5000, 300, False, False), ("maxplus", "f64", 64, 128, 128, 300, False, True),
    ("maxplus", "f32", 1, 47500, 40, 33, True, False), ("maxplus", "f32", 1, 30000, 40, 33, True, True),
    ("maxmul", "i32", 1, 100, 15000, 64, True, False), ("maxplus", "f64", 475, 41, 41, 33, True, False),
    ("maxplus", "f64", 475, 41, 41, 200, True, True), ("maxplus", "f64", 1784, 41, 41, 128, True, False),
    ("maxplus", "f64", 1, 100, 15000, 64, False, False), ("maxplus", "i64", 1, 15000, 40, 33, True, False),
    ("maxplus", "i64", 1, 15000, 40, 64, True, True), ("maxmul", "i64", 1220, 64, 64, 161, True, False),
    ("maxmul", "i64", 1, 100, 50000, 200, True, True), ("maxplus", "i64", 732, 64, 64, 400, False, False),
    ("maxplus", "i64", 1, 2047, 2049, 1025, False, True), ("maxplus", "i64", 128, 128, 128, 129, False, False),
    ("maxplus", "f32", 256, 48, 48, 512, True, False), ("maxplus", "f32", 64, 48, 48, 512, True, True),
    # Up to 64 columns at short K.
    ("maxplus", "f32", 1, 524288, 64, 2, True, False), ("maxplus", "f32", 1, 524288, 64, 12, True, True),
    ("maxplus", "f32", 1, 524288, 32, 2, True, True), ("maxplus", "f32", 1, 524288, 33, 32, True, False),
    ("maxplus", "f32", 1, 524288, 3, 2, True, False), ("maxplus", "f32", 1, 524288, 3, 12, True, True),
    ("maxplus", "f64", 1, 524288, 33, 24, True, False), ("maxplus", "f64", 1, 65536, 30, 12, True, True),
    ("maxplus", "f32", 1, 524288, 33, 32, False, False), ("maxplus", "f64", 1, 524288, 50, 12, False, True),
    ("maxplus", "f32", 5000, 48, 48, 8, False, False), ("maxplus", "f32", 5000, 48, 48, 16, False, True),
    ("maxplus", "f32", 1, 4096, 33, 32, True, True),
    ("maxplus", "f32", 1, 3, 524288, 36, False, False), ("maxplus", "f32", 1, 524288, 8, 36, False, True),
])
def test_few_output_kernel_leaves_what_others_run_faster(sr, dt, batch, m, n, k, argmax, few):
    plan = nat.gemm_small_plan(sr, dt, m, n, k, argmax, batch=batch,
                               strides=(m * k, k * n, m * n))
    assert ("waves" in plan) == few, plan
