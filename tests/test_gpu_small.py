"""The few-output kernel (tg_gemm_small): every launch form, at the edges of its
tiles, k-steps and waves, against the oracle bit for bit, with guard bytes
around the outputs; and the Python entry points, which run it where
tg_gemm_small_plan names a form."""
import ctypes

import numpy as np
import pytest

from oracle import oracle
from tests import tg_cases as tc
from tests.test_gpu_nan import assert_nan_exact, nan_inputs

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"
GUARD, FILL = 64, 0xA5  # elements of padding before and after each output


def _small(sr, items, with_argmax, layout="row", gap=0, offset=0):
    """tg_gemm_small on a strided batch (gap: elements between items, offset:
    elements past a 16-byte boundary); None when it leaves the problem alone."""
    from tropical_gemm import _native as nat

    lib = nat.load()
    (m, k), n, batch = items[0][0].shape, items[0][1].shape[1], len(items)
    dt = items[0][0].dtype
    order = (lambda x: x) if layout == "row" else (lambda x: x.T)

    def packed(mats):
        size = mats[0].size + gap
        flat = np.zeros(offset + batch * size, dt)
        for t, x in enumerate(mats):
            flat[offset + t * size:offset + t * size + x.size] = np.ascontiguousarray(order(x)).ravel()
        return torch.from_numpy(flat).to(DEV), size

    ta, sa = packed([x for x, _ in items])
    tb, sb = packed([y for _, y in items])
    sc = m * n + gap

    def guarded(dtype):
        raw = torch.full(((2 * GUARD + offset + batch * sc) * np.dtype(dtype).itemsize,), FILL,
                         dtype=torch.uint8, device=DEV)
        return raw, raw.data_ptr() + (GUARD + offset) * np.dtype(dtype).itemsize

    craw, cptr = guarded(dt)
    iraw, iptr = guarded(np.int32) if with_argmax else (None, None)
    ran = ctypes.c_int(7)
    es = dt.itemsize
    nat.check(lib.tg_gemm_small(
        0, nat.SEMIRING[sr], nat.DTYPE[{v: s for s, v in tc.NP_DTYPES.items()}[dt.type]],
        nat.LAYOUT[layout], ta.data_ptr() + offset * es, tb.data_ptr() + offset * es, cptr, iptr,
        batch, m, n, k, sa, sb, sc, torch.cuda.current_stream().cuda_stream, ran))
    torch.cuda.synchronize()
    if not ran.value:
        return None

    def unpack(raw, dtype):
        if raw is None:
            return [None] * batch
        flat = raw.cpu().numpy().view(dtype)
        used = np.zeros(flat.size, bool)
        out = []
        for t in range(batch):
            s = GUARD + offset + t * sc
            used[s:s + m * n] = True
            x = flat[s:s + m * n]
            out.append(x.reshape(m, n) if layout == "row" else x.reshape(n, m).T)
        assert (flat[~used].view(np.uint8) == FILL).all(), "bytes outside the outputs written"
        return out

    return list(zip(unpack(craw, dt), unpack(iraw, np.int32)))


def _check(sr, items, with_argmax, **kw):
    res = _small(sr, items, with_argmax, **kw)
    assert res is not None
    for (a, b), (c, am) in zip(items, res):
        c_ref, am_ref = oracle.gemm(sr, a, b, with_argmax=with_argmax)
        assert_nan = c_ref.dtype.kind == "f" and np.isnan(c_ref).any()
        if assert_nan:
            assert_nan_exact(c, am, c_ref, am_ref)
        elif with_argmax:
            np.testing.assert_array_equal(tc.bits(c), tc.bits(c_ref))
            np.testing.assert_array_equal(am.astype(np.int64), am_ref.astype(np.int64))
        else:
            np.testing.assert_array_equal(c, c_ref)  # the sign of a +-0 tie is open


# (batch, m, n, k), form: tiles of 4 x 16 (one row, ragged columns, K below,
# at and past a step of 64 or 32 k), 8 x 16, 16 x 16 and 32 x 32 outputs, the
# one-column form (N < 4), and K split over up to 16 waves.  Every form runs with
# and without argmax in every dtype (test_every_form_has_its_shapes).
SHAPES = [
    ((1, 1, 5, 1), "4x16 waves 1"), ((1, 3, 16, 63), "4x16"), ((1, 5, 17, 65), "4x16"),
    ((1, 67, 45, 131), "4x16"), ((1, 4, 1000, 4096), "4x16"), ((1, 16, 777, 1500), "4x16"),
    ((3, 100, 260, 33), "8x16"), ((1, 130, 515, 97), "8x16"),
    ((1, 250, 900, 129), "16x16"), ((20, 63, 49, 700), "8x16"),
    ((30, 129, 131, 30), "32x32"), ((9, 300, 200, 127), "32x32"),
    ((1, 20001, 31, 15), "32x32"), ((1, 20001, 31, 29), "32x32"),
    ((1, 1, 1, 7), "16x4"), ((1, 2, 3, 64), "16x4"), ((1, 1000, 1, 515), "16x4"),
    ((4, 33, 2, 2050), "16x4"),
]


# The shapes that other kernels run faster: (dtype, with_argmax) by shape.
OTHERS = {
    (30, 129, 131, 30): {("f32", True), ("f64", True), ("i32", True), ("i64", True)},
    (9, 300, 200, 127): {("f64", True)},
    (1, 20001, 31, 15): {("f32", True), ("i32", True)},
    (1, 20001, 31, 29): {("f64", True), ("i32", True), ("i64", True)},
}


def test_every_form_has_its_shapes():
    ran = {(form.split()[0], dt, am) for shape, form in SHAPES for dt in ("f32", "f64", "i32", "i64")
           for am in (True, False) if (dt, am) not in OTHERS.get(shape, ())}
    assert len(ran) == 5 * 4 * 2


@pytest.mark.parametrize("dt", ["f32", "f64", "i32", "i64"])
@pytest.mark.parametrize("shape,form", SHAPES, ids=["x".join(map(str, s)) for s, _ in SHAPES])
def test_small_forms(dt, shape, form):
    from tropical_gemm import _native as nat

    batch, m, n, k = shape
    rng = np.random.default_rng(m * 131 + n * 7 + k)
    dtype = tc.NP_DTYPES[dt]
    for sr in tc.SEMIRINGS:
        # Small whole numbers: ties between lanes, waves and steps.
        lo, hi = (1, 9) if sr == "maxmul" else (-9, 9)
        items = [(rng.integers(lo, hi, size=(m, k)).astype(dtype),
                  rng.integers(lo, hi, size=(k, n)).astype(dtype)) for _ in range(batch)]
        for with_argmax in (True, False):
            plan = nat.gemm_small_plan(sr, dt, m, n, k, with_argmax, batch=batch,
                                       strides=(m * k + 1, k * n + 1, m * n + 1), addresses=(8,) * 4)
            if (dt, with_argmax) in OTHERS.get(shape, ()):
                assert plan == "none"
                continue
            assert plan.startswith(form), plan
            print(f"[case] small {sr} {dt} {shape} argmax={with_argmax} {plan}", flush=True)
            _check(sr, items, with_argmax, gap=1, offset=1)


@pytest.mark.parametrize("dt", ["f32", "f64"])
@pytest.mark.parametrize("sr", tc.SEMIRINGS)
def test_small_nan_rule(sr, dt):
    for m, n, k in ((67, 45, 131), (40, 300, 300), (9, 3, 257)):
        print(f"[case] small NaN {sr} {dt} {m}x{n}x{k}", flush=True)
        a, b = nan_inputs(sr, tc.NP_DTYPES[dt], m, max(n, 8), k, seed=k)
        _check(sr, [(a, np.ascontiguousarray(b[:, :n]))], True)
        _check(sr, [(a, np.ascontiguousarray(b[:, :n]))], False)


@pytest.mark.parametrize("dt", ["f32", "f64", "i32", "i64"])
@pytest.mark.parametrize("sr", tc.SEMIRINGS)
def test_small_extremes(sr, dt):
    """Products that never beat the tropical zero, infinities, signed zeros,
    wrapping integers; column-major calls."""
    rng = np.random.default_rng(8)
    dtype = tc.NP_DTYPES[dt]
    m, n, k = 21, 37, 70
    if dtype in (np.float32, np.float64):
        vals = np.array([0.0, -0.0, 1.0, -1.0] + ([np.inf] if sr == "minplus" else
                                                  [-np.inf] if sr == "maxplus" else [0.5]), dtype)
    else:
        info = np.iinfo(dtype)
        vals = np.array([0, 1, -1, info.max, info.min, info.max // 2 + 1], dtype)
    a, b = rng.choice(vals, (m, k)), rng.choice(vals, (k, n))
    if sr != "maxmul" and dtype in (np.float32, np.float64):
        a[3] = vals[-1]  # a row of tropical zeros
    if sr == "maxmul":
        a[3] = 0
    for layout in ("row", "col"):
        print(f"[case] small extremes {sr} {dt} {layout}", flush=True)
        _check(sr, [(a, b)], True, layout=layout)


def test_small_reached_from_python():
    from tropical_gemm import _native as nat, ops

    rng = np.random.default_rng(5)
    a = rng.standard_normal((3, 41, 53)).astype(np.float32)
    b = rng.standard_normal((3, 53, 29)).astype(np.float32)
    assert nat.gemm_small_plan("maxplus", "f32", 41, 29, 53, batch=3) != "none"
    # Large products keep their kernels.
    assert nat.gemm_small_plan("maxplus", "f32", 4096, 4096, 4096) == "none"
    assert nat.gemm_small_plan("maxplus", "f32", 1024, 1024, 1024) == "none"
    c, am = ops.gemm_batched("maxplus", torch.from_numpy(a).to(DEV), torch.from_numpy(b).to(DEV))
    for t in range(3):
        c_ref, am_ref = oracle.gemm("maxplus", a[t], b[t])
        np.testing.assert_array_equal(tc.bits(c[t].cpu().numpy()), tc.bits(c_ref))
        np.testing.assert_array_equal(am[t].cpu().numpy().astype(np.int64), am_ref.astype(np.int64))
