"""The workspace entry points under HIP graph capture.

Every entry point that takes a caller workspace launches kernels only (no
allocation, no memset: buffers that must start at zero are cleared by a fill
kernel), so a caller can capture it in a HIP graph and replay it.  The test
captures the forward paths (direct-to-LDS tiles with B^T staging, 64x128
tiles, split K, element loads in K slices, the K-resident kernels, the generic
tiles, their exact short-K mode, value-only, and the 64-bit direct-to-LDS kernels
with their operand class prepass, with and without argmax), the entry points
without a caller workspace (tg_gemm_small, and tg_gemm where its workspace is
optional) and both backward scatters, replays the graph
several times with new inputs copied in and eager work between the replays,
and checks every replay against eager calls on the same inputs, bit for bit
(the backward too: each gradient element receives a single contribution, so
the sum order cannot differ)."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"

# (name, semiring, dtype, m, k, n, argmax): one problem per forward path.
CASES = [
    ("direct-to-LDS", "maxplus", torch.float32, 2048, 1024, 2048, True),
    ("wide tiles", "minplus", torch.float32, 4096, 1024, 4096, True),
    ("split-K", "maxplus", torch.float32, 128, 4096, 128, True),
    ("K-resident", "maxplus", torch.int32, 512, 128, 128, True),
    ("generic tiles", "minplus", torch.float64, 77, 45, 93, True),
    ("exact short K", "maxplus", torch.float32, 1000, 16, 1024, True),
    ("value-only", "maxmul", torch.float32, 256, 256, 192, False),
    ("f64 direct-to-LDS", "maxplus", torch.float64, 1024, 640, 4096, True),
    ("f64 value-only", "minplus", torch.float64, 1024, 256, 4096, False),
    ("element loads", "maxplus", torch.float32, 1090, 515, 1201, True),
    ("element loads, four slices", "maxplus", torch.float32, 513, 1027, 511, True),
    ("element loads, value-only", "minplus", torch.int32, 700, 300, 701, False),
    ("any short K", "maxplus", torch.int32, 2000, 61, 130, True),
    ("f64 64x64 tiles", "maxplus", torch.float64, 700, 641, 701, True),
    ("f64 64x64 tiles, value-only", "minplus", torch.float64, 700, 400, 701, False),
    ("i64 64x64 tiles", "maxplus", torch.int64, 513, 600, 514, True),
    ("i64 64x64 tiles, value-only", "minplus", torch.int64, 513, 130, 514, False),
]

# (semiring, dtype, m, k, n, argmax): few outputs, and i32 keys on few row tiles.
SMALL_CASES = [
    ("maxplus", torch.float32, 67, 131, 45, True),
    ("minplus", torch.float64, 300, 400, 300, False),
    ("maxplus", torch.int64, 5, 65, 17, True),
    ("maxplus", torch.int32, 2064, 128, 512, True),
]
# tg_gemm with a workspace that it allocates outside a capture and does without
# inside one: 32-bit, f64 and i64 argmax, f64 value-only.
OPTIONAL_CASES = [
    ("maxplus", torch.float32, 1000, 300, 1001, True),
    ("minplus", torch.float64, 1500, 512, 1500, True),
    ("maxplus", torch.float64, 700, 420, 701, False),
    ("minplus", torch.int64, 1000, 1000, 1000, True),
]
DT_CODE = {torch.float32: "f32", torch.float64: "f64", torch.int32: "i32", torch.int64: "i64"}


def _vp(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def _fill(t, gen):
    if t.dtype.is_floating_point:
        t.copy_(torch.randn(t.shape, generator=gen, device=DEV, dtype=t.dtype).abs())
    else:
        t.copy_(torch.randint(-1000, 1001, t.shape, generator=gen, device=DEV, dtype=t.dtype))


def test_forward_paths_replay_like_eager():
    from tropical_gemm import _native as nat

    lib = nat.load()
    gen = torch.Generator(device=DEV)
    gen.manual_seed(77)
    bufs = []
    for name, sr, dt, m, k, n, argmax in CASES:
        a = torch.empty((m, k), dtype=dt, device=DEV)
        b = torch.empty((k, n), dtype=dt, device=DEV)
        c = torch.empty((m, n), dtype=dt, device=DEV)
        am = torch.empty((m, n), dtype=torch.int32, device=DEV) if argmax else None
        d = nat.DTYPE[DT_CODE[dt]]
        wsb = lib.tg_gemm_workspace_size(d, 1, m, n, k, int(argmax))
        ws = torch.empty(max(wsb, 256), dtype=torch.uint8, device=DEV)
        bufs.append((name, sr, d, m, k, n, a, b, c, am, ws, wsb))

    def run_all(stream):
        s = ctypes.c_void_p(stream.cuda_stream)
        for name, sr, d, m, k, n, a, b, c, am, ws, wsb in bufs:
            nat.check(lib.tg_gemm_ws(0, nat.SEMIRING[sr], d, 0, _vp(a), _vp(b), _vp(c), _vp(am),
                                     m, n, k, _vp(ws), wsb, s))

    for _, _, _, _, _, _, a, b, *_ in bufs:
        _fill(a, gen)
        _fill(b, gen)
    run_all(torch.cuda.current_stream())  # eager warm-up (device queries cached)
    torch.cuda.synchronize()

    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run_all(torch.cuda.current_stream())
    for rep in range(3):
        print(f"[case] graph replay {rep}", flush=True)
        for _, _, _, _, _, _, a, b, *_ in bufs:
            _fill(a, gen)
            _fill(b, gen)
        graph.replay()
        torch.cuda.synchronize()
        got = [(c.clone(), None if am is None else am.clone()) for *_, c, am, _, _ in bufs]
        # Eager work between replays, then the eager reference on the same inputs.
        junk = torch.randn(1 << 20, device=DEV).cumsum(0)
        del junk
        run_all(torch.cuda.current_stream())
        torch.cuda.synchronize()
        for (name, *_, c, am, _, _), (gc, gam) in zip(bufs, got):
            assert torch.equal(gc.view(torch.uint8), c.view(torch.uint8)), f"{name}: values, replay {rep}"
            if am is not None:
                assert torch.equal(gam, am), f"{name}: argmax, replay {rep}"


def test_entry_points_without_workspace_replay_like_eager():
    """tg_gemm_small and tg_gemm: no allocation nodes, whatever kernel the eager
    call takes."""
    from tropical_gemm import _native as nat

    lib = nat.load()
    gen = torch.Generator(device=DEV)
    gen.manual_seed(79)
    bufs = []
    for sr, dt, m, k, n, argmax in SMALL_CASES + OPTIONAL_CASES:
        d = DT_CODE[dt]
        small = len(bufs) < len(SMALL_CASES)
        am = torch.empty((m, n), dtype=torch.int32, device=DEV) if argmax else None
        if small:
            assert nat.gemm_small_plan(sr, d, m, n, k, argmax) != "none"
        else:
            assert lib.tg_gemm_alloc_bytes(nat.SEMIRING[sr], nat.DTYPE[d], 0, 256, 256, 256,
                                           256 if argmax else None, 1, m, n, k, 0, 0, 0) > 0
            assert nat.gemm_plan(sr, d, m, n, k, argmax, workspace_bytes=0).startswith("tiles")
        bufs.append((small, nat.SEMIRING[sr], nat.DTYPE[d], m, k, n,
                     torch.empty((m, k), dtype=dt, device=DEV),
                     torch.empty((k, n), dtype=dt, device=DEV),
                     torch.empty((m, n), dtype=dt, device=DEV), am))

    def fill():
        for *_, a, b, _, _ in bufs:
            _fill(a, gen)
            _fill(b, gen)

    def run_all(stream):
        s = ctypes.c_void_p(stream.cuda_stream)
        for small, sr, d, m, k, n, a, b, c, am in bufs:
            if small:
                ran = ctypes.c_int(0)
                nat.check(lib.tg_gemm_small(0, sr, d, 0, _vp(a), _vp(b), _vp(c), _vp(am), 1, m, n,
                                            k, m * k, k * n, m * n, s, ran))
                assert ran.value == 1
            else:
                nat.check(lib.tg_gemm(0, sr, d, 0, _vp(a), _vp(b), _vp(c), _vp(am), m, n, k, s))

    fill()
    run_all(torch.cuda.current_stream())
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run_all(torch.cuda.current_stream())
    for rep in range(3):
        print(f"[case] graph replay without workspace {rep}", flush=True)
        fill()
        graph.replay()
        torch.cuda.synchronize()
        got = [(c.clone(), None if am is None else am.clone()) for *_, c, am in bufs]
        junk = torch.randn(1 << 20, device=DEV).cumsum(0)
        del junk
        run_all(torch.cuda.current_stream())
        torch.cuda.synchronize()
        for q, ((*_, c, am), (gc, gam)) in enumerate(zip(bufs, got)):
            assert torch.equal(gc.view(torch.uint8), c.view(torch.uint8)), f"case {q}, replay {rep}"
            if am is not None:
                assert torch.equal(gam, am), f"case {q}: argmax, replay {rep}"


@pytest.mark.parametrize("k", [512, 9000, 40000])
def test_backward_replays_like_eager(k):
    """grad_A and grad_B under capture: bins in LDS at K = 512 and 9000
    (grad_B in three passes over its keys at 9000), in the gradients
    themselves at K = 40000 (grad_A; grad_B takes ten passes)."""
    from tropical_gemm import _native as nat

    lib = nat.load()
    m, n = 192, 160
    gen = torch.Generator(device=DEV)
    gen.manual_seed(78)
    d = nat.DTYPE["f32"]
    g = torch.empty((m, n), device=DEV)
    # Distinct argmax per row and per column: every gradient element gets at
    # most one contribution, so results do not depend on the summation order.
    idx = torch.empty((m, n), dtype=torch.int32, device=DEV)
    ga = torch.empty((m, k), device=DEV)
    gb = torch.empty((k, n), device=DEV)

    def refill():
        g.copy_(torch.randn((m, n), generator=gen, device=DEV))
        perm = torch.randperm(k, generator=gen, device=DEV)[: m + n].to(torch.int32)
        rows = torch.arange(m, device=DEV, dtype=torch.int32)[:, None]
        cols = torch.arange(n, device=DEV, dtype=torch.int32)[None, :]
        idx.copy_(perm[(rows + cols) % (m + n)])

    def run(stream):
        s = ctypes.c_void_p(stream.cuda_stream)
        nat.check(lib.tg_backward_a(0, d, 0, _vp(g), _vp(idx), _vp(ga), m, n, k, s))
        nat.check(lib.tg_backward_b(0, d, 0, _vp(g), _vp(idx), _vp(gb), m, n, k, s))

    refill()
    run(torch.cuda.current_stream())
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run(torch.cuda.current_stream())
    for rep in range(3):
        print(f"[case] backward graph replay k={k} {rep}", flush=True)
        refill()
        graph.replay()
        torch.cuda.synchronize()
        ra, rb = ga.clone(), gb.clone()
        run(torch.cuda.current_stream())
        torch.cuda.synchronize()
        assert torch.equal(ra, ga) and torch.equal(rb, gb), f"replay {rep}"
        # And the scatter itself: grad_A[i, idx[i, j]] == g[i, j] (one term each).
        gh, ih = g.cpu().numpy(), idx.cpu().numpy()
        rows = np.arange(m)[:, None].repeat(n, 1)
        assert np.array_equal(ra.cpu().numpy()[rows, ih], gh)
