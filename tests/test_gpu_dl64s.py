"""64-bit products on 64 x 64 direct-to-LDS tiles (tg_gemm_dl64s): f64 below
the 64 x 128 tiles' range and i64, in one to four K slices, at the edges of
tiles, k-tiles, slices and resolve windows, against the oracle bit for bit."""
import numpy as np
import pytest

from oracle import oracle
from tests import tg_cases as tc
from tests.test_gpu_nan import assert_nan_exact, nan_inputs
from tests.test_gpu_parity import _strided_batched, assert_exact, gpu_gemm

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

PLAN = {True: "dl64s_4x4_cl16", False: "dl64s_4x4"}

# Up to 256 tiles K runs in three (argmax) or four slices, above in one or two.
# (m, n, k): a last k-tile of 1, 2, 15 and 16 k, 33 and 34 k-tiles (slices of
# unequal length), odd and even rows (element and 16-byte loads), ragged last
# columns; 306 tiles; the first K of each rule; value-only i64 at 9 k-tiles (the
# fourth slice empty).
SHAPES = [(513, 511, 513), (514, 516, 514), (449, 577, 527), (576, 514, 528), (512, 520, 544),
          (1025, 1090, 513), (1030, 1026, 530)]
SHORT = {("f64", True): [(1473, 1500, 257), (1025, 1090, 385)],
         ("f64", False): [(513, 519, 257), (449, 577, 320), (1025, 1090, 351)],
         ("i64", True): [(1025, 1090, 257), (1473, 1501, 129), (1473, 1501, 301), (3001, 3003, 97)],
         ("i64", False): [(513, 511, 130), (515, 512, 97), (1025, 1090, 193)]}


def _data(sr, dtype, m, n, k):
    """Whole numbers with ties, winners in the last and in the first k."""
    rng = np.random.default_rng(m + 3 * n + 7 * k)
    lo, hi = (1, 50) if sr == "maxmul" else (-50, 50)
    a = rng.integers(lo, hi, size=(m, k))
    b = rng.integers(lo, hi, size=(k, n))
    a[::3, k - 1] = 60 if sr != "minplus" else -60
    b[k - 1, ::5] = 60 if sr != "minplus" else -60
    a[1::7, k - 2] = a[1::7, k - 1]
    a[2::9, 0] = a[2::9, k - 1]
    return a.astype(dtype), b.astype(dtype)


def _run(sr, dt, m, n, k, with_argmax, a, b, c_ref, am_ref):
    """The product with a workspace of its full size (tg_gemm allocates one only
    where it pays)."""
    from tropical_gemm import _native as nat

    lib = nat.load()
    assert nat.gemm_plan(sr, dt, m, n, k, with_argmax) == PLAN[with_argmax]
    print(f"[case] dl64s {sr} {dt} {m}x{n}x{k} argmax={with_argmax}", flush=True)
    ta, tb = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
    c = torch.empty((m, n), dtype=ta.dtype, device="cuda")
    am = torch.empty((m, n), dtype=torch.int32, device="cuda") if with_argmax else None
    wsb = lib.tg_gemm_workspace_size(nat.DTYPE[dt], 1, m, n, k, int(with_argmax))
    ws = torch.empty(max(wsb, 256), dtype=torch.uint8, device="cuda")
    nat.check(lib.tg_gemm_ws(0, nat.SEMIRING[sr], nat.DTYPE[dt], 0, ta.data_ptr(), tb.data_ptr(),
                             c.data_ptr(), None if am is None else am.data_ptr(), m, n, k,
                             ws.data_ptr(), wsb, torch.cuda.current_stream().cuda_stream))
    assert_exact(c.cpu().numpy(), None if am is None else am.cpu().numpy(), c_ref,
                 am_ref if with_argmax else None)


@pytest.mark.parametrize("dt", ["f64", "i64"])
@pytest.mark.parametrize("m,n,k", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
def test_dl64s_edges(dt, m, n, k):
    for sr in tc.SEMIRINGS:
        a, b = _data(sr, tc.NP_DTYPES[dt], m, n, k)
        c_ref, am_ref = oracle.gemm(sr, a, b)
        for with_argmax in (True, False):
            _run(sr, dt, m, n, k, with_argmax, a, b, c_ref, am_ref)


@pytest.mark.parametrize("dt,with_argmax", list(SHORT), ids=[f"{d}-{w}" for d, w in SHORT])
def test_dl64s_short_k(dt, with_argmax):
    srs = ("maxplus", "minplus", "maxmul", "maxplus")
    for sr, (m, n, k) in zip(srs, SHORT[dt, with_argmax]):
        a, b = _data(sr, tc.NP_DTYPES[dt], m, n, k)
        _run(sr, dt, m, n, k, with_argmax, a, b, *oracle.gemm(sr, a, b))


@pytest.mark.parametrize("m,n,k", [(513, 515, 515), (1090, 1024, 528)])
@pytest.mark.parametrize("sr", tc.SEMIRINGS)
def test_dl64s_nan_rule(sr, m, n, k):
    a, b = nan_inputs(sr, np.float64, m, n, k, seed=5)
    rows = np.unique(np.concatenate([np.arange(0, m, 19), [0, 1, 2, 3, 4, m - 1]]))
    c_ref, am_ref = oracle.gemm(sr, a[rows], b)
    for layout in ("row", "col"):
        for with_argmax in (True, False):
            print(f"[case] dl64s NaN {sr} {m}x{n}x{k} {layout} argmax={with_argmax}", flush=True)
            c, am = gpu_gemm(sr, a, b, with_argmax, layout=layout)
            assert_nan_exact(c[rows], am[rows] if with_argmax else None, c_ref,
                             am_ref if with_argmax else None)


@pytest.mark.parametrize("dt", ["f64", "i64"])
def test_dl64s_wrapping_zeros_and_batches(dt):
    """Batch strides that break the 16-byte alignment; wrapping i64 sums,
    signed zeros and rows that never beat the tropical zero."""
    rng = np.random.default_rng(9)
    m, n, k = 320, 330, 520
    if dt == "i64":
        info = np.iinfo(np.int64)
        vals = np.array([0, 1, -1, info.max, info.min, info.max // 2 + 1], np.int64)
    else:
        vals = np.array([0.0, -0.0, 1.0, -1.0, 0.5, -np.inf])
    for sr in ("maxplus", "maxmul"):
        use = vals if sr == "maxplus" else vals[:-1]
        items = [(rng.choice(use, (m, k)), rng.choice(use, (k, n))) for _ in range(3)]
        items[1][0][7] = use[-1] if sr == "maxplus" else 0
        print(f"[case] dl64s batch {sr} {dt}", flush=True)
        for (x, y), (c, am) in zip(items, _strided_batched(sr, items, gap_a=1, gap_c=3)):
            assert_exact(c, am, *oracle.gemm(sr, x, y))


def test_i64_without_workspace_keeps_the_exact_mode():
    from tropical_gemm import _native as nat

    assert nat.gemm_plan("maxplus", "i64", 512, 40000, 300, True) == "dl64s_4x4_cl16"
    assert nat.gemm_plan("maxplus", "i64", 512, 40000, 300, True,
                         workspace_bytes=64 << 20) == "tiles_exact"
