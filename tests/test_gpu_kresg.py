"""The K-resident i32 argmax kernel for any short K, M and N (tg_gemm_kresg)
at the edges of its tiles and of its key range, against the oracle bit for
bit."""
import numpy as np
import pytest

from oracle import oracle
from tests.test_gpu_parity import _strided_batched, assert_exact, gpu_gemm

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# (m, n, k, batch): last row tiles of 1, 15 and 16 rows; last column quads of
# 1, 2, 3 and 4 columns, one and several column tiles; last k quads of 1, 2, 3
# and 4 k, K of one and of all five k tiles of the 8-wave form; more row tiles
# than one round of waves; the 16-wave form at its first, a middle and its
# largest K (whole rounds of wave tiles); batches.
SHAPES = [(4097, 17, 12, 1), (1039, 64, 32, 1), (2000, 130, 21, 1), (2050, 255, 29, 1),
          (1025, 65, 33, 1), (335, 254, 50, 1), (529, 131, 97, 1), (70001, 66, 35, 1),
          (600, 317, 160, 1), (2001, 1601, 161, 1), (1970, 2046, 203, 1), (4096, 1024, 256, 1),
          (200, 61, 43, 7), (33, 70, 130, 40), (1100, 50, 24, 3)]


@pytest.mark.parametrize("sr", ["maxplus", "minplus"])
@pytest.mark.parametrize("m,n,k,batch", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
def test_short_k_keys(sr, m, n, k, batch):
    from tropical_gemm import _native as nat

    strides = (m * k, k * n, m * n) if batch > 1 else (0, 0, 0)
    assert nat.gemm_plan(sr, "i32", m, n, k, True, batch=batch, strides=strides) == "kresg"
    sign = 1 if sr == "maxplus" else -1
    small = batch * m * n * k < 500_000_000
    for data in ("keys", "edge", "rows", "panel", "wide") if small else ("rows", "wide"):
        rng = np.random.default_rng(m + 3 * n + 7 * k + len(data))
        print(f"[case] short-K keys {sr} {m}x{n}x{k} batch {batch} {data}", flush=True)
        items = []
        for t in range(batch):
            a = rng.integers(-20, 21, size=(m, k))
            b = rng.integers(-20, 21, size=(k, n))
            a[::3, k - 1] = 25 * sign  # winners and ties in the last quad
            a[1::3, k - 2] = a[1::3, max(0, k - 5)]
            b[k - 1, ::5] = 25 * sign
            if data == "edge":  # the ends of the key range
                a[::5, 0], a[2::7, k - 1] = -32768, 32767
                b[0, ::3], b[k - 1, 1::4] = 32767, -32768
            if data == "rows":  # wave tiles that leave it in their last and first k tiles
                a[min(m - 1, 21 + t), k - 1] = 40000 * sign
                a[m // 2, 0] = -32769
                a[m - 1, k // 2] = -2**31
            if data == "panel" and t != 1:  # the last column tile's panel leaves it
                b[k - 1, n - 1] = 32768
            if data == "wide":  # products that wrap, the tropical zero, the type's ends
                a = rng.integers(-2**31, 2**31, size=(m, k))
                b = rng.integers(-2**31, 2**31, size=(k, n))
                a[0], b[:, 0] = -2**31, 0
                a[1], b[:, 1] = 2**31 - 1, 0
            items.append((a.astype(np.int32), b.astype(np.int32)))
        if batch == 1:
            got = [gpu_gemm(sr, *items[0], True)]
        else:
            got = _strided_batched(sr, items)
        for (c, am), (a, b) in zip(got, items):
            assert_exact(c, am, *oracle.gemm(sr, a, b))


# The aligned sizes of tg_gemm_kresw whose wave tiles are few: the tensor entry
# point hands them on, from the few-output kernel's last size up.
@pytest.mark.parametrize("m,n,k,batch", [(1024, 1024, 64, 1), (2064, 512, 128, 1),
                                         (512, 128, 96, 13)])
def test_few_wave_tiles(m, n, k, batch):
    from tropical_gemm import _native as nat
    from tropical_gemm import ops

    strides = (m * k, k * n, m * n)
    assert nat.gemm_plan("maxplus", "i32", m, n, k, True, batch=batch, strides=strides) == "kresw"
    assert nat.gemm_small_plan("maxplus", "i32", m, n, k, True, batch=batch,
                               strides=strides) == "kresg"
    rng = np.random.default_rng(m + batch)
    a = rng.integers(-1000, 1001, size=(batch, m, k)).astype(np.int32)
    b = rng.integers(-50, 1, size=(batch, k, n)).astype(np.int32)
    a[-1, m // 2, k - 1] = 40000
    print(f"[case] few wave tiles {m}x{n}x{k} batch {batch}", flush=True)
    c, am = ops.gemm_batched("maxplus", torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda())
    for t in range(batch):
        assert_exact(c[t].cpu().numpy(), am[t].cpu().numpy(), *oracle.gemm("maxplus", a[t], b[t]))
