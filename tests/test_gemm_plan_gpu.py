"""The dense planner's choice: held against what it chose from, measured here, for large row counts (four-wave heights and
the ping-pong kernel), the weight stream's limits, and the switches and overrides."""
import pytest
import torch

from mlopamd import ops

pytestmark = pytest.mark.gpu
bf = torch.bfloat16
VARIANTS = {"ping-pong": (3, 256), "256": (5, 256), "224": (6, 224), "192": (6, 192), "160": (6, 160), "128": (6, 128)}


def best_times(runs, t, reps=5):
    """us of each run into ``t``, the best of ``reps`` in turn and of what is there."""
    for k in range(reps + 1):
        for name, run in runs.items():
            a, b = torch.cuda.Event(True), torch.cuda.Event(True)
            a.record()
            run()
            b.record()
            b.synchronize()
            if k:
                t[name] = min(t[name], a.elapsed_time(b) * 1e3)


# shapes on which a model of the time went wrong before: long K at few tiles, a remainder of a few tiles, one round
# nearly full; then ordinary ones
@pytest.mark.parametrize("M,N,K", [(560, 6144, 16384), (700, 6144, 16384), (768, 6144, 16384), (1300, 5120, 5120), (640, 10240, 8192),
                                   (2300, 8192, 28672), (2048, 3072, 3072), (890, 28672, 4096), (2600, 4096, 4096), (1152, 4096, 14336),
                                   # where tiles of 224 rows save rounds, and five rounds of them
                                   (400, 28672, 4096), (892, 28672, 4096), (1100, 28672, 4096), (3700, 28672, 4096)])
def test_large_rows(gpu, M, N, K):
    """The choice is at most 15 % slower than the best variant: over what the model is fitted to it is 12 % at worst, at these
    2 %, and what else runs on the host moves a best of five by up to 5 % (measured again, up to four times, where it moved
    more)."""
    ops._sk_reserve(torch.device(gpu))
    x = torch.randn(M, K, device=gpu, dtype=bf)
    n = int(6e8 / (2 * N * K)) + 2  # more than the caches hold: a layer's weights are read once per step
    w = [(0.02 * torch.randn(N, K, device=gpu)).to(bf) for _ in range(n)]
    out = torch.empty(M, N, device=gpu, dtype=bf)
    no_ws = torch.empty(0, device=gpu)
    plan = torch.ops.mlop.gemm_dense_plan

    def run(variant):
        def go():
            plan(*variant)
            try:
                for a in w:
                    torch.ops.mlop.gemm(out, x, a, no_ws, 0)
            finally:
                plan(-1, -1, -1, -1)
        return go

    runs = {"choice": run((-1, -1, -1, -1)), **{name: run((v, bm, 256, -1)) for name, (v, bm) in VARIANTS.items()}}
    t = dict.fromkeys(runs, 1e30)
    for _ in range(4):
        best_times(runs, t)
        if t["choice"] <= 1.15 * min(t[v] for v in VARIANTS):
            break
    assert t["choice"] <= 1.15 * min(t[v] for v in VARIANTS), {k: round(v / n, 1) for k, v in t.items()}


@pytest.mark.parametrize("M,N,K,stream", [
    # two row tiles: not in one K range where the four-wave kernel has a grid (columns in 256s, K >= 192), nor above 320 rows
    (256, 28672, 4096, True), (257, 28672, 4096, False), (384, 12288, 4096, False), (300, 12296, 4096, True), (300, 28672, 128, True),
    (320, 8192, 7168, True), (321, 8192, 7168, False), (384, 4096, 14336, True), (385, 4096, 14336, False),
    # slabs beside the weights
    (96, 8192, 3584, True), (97, 8192, 3584, False), (160, 8192, 3584, True), (192, 8192, 3584, False), (256, 5120, 5120, True),
    (64, 8192, 28672, False), (65, 8192, 28672, True)])
def test_weight_stream_limits(gpu, M, N, K, stream):
    ops._sk_reserve(torch.device(gpu))
    assert (torch.ops.mlop.gemm_plan(M, N, K)[0] == 7) == stream


@pytest.mark.parametrize("M,N,K", [(16, 6144, 4096), (16, 28672, 4096), (64, 28672, 4096), (100, 6144, 4096), (200, 28672, 4096), (200, 4096, 14336)])
def test_cache_policy_switches(gpu, M, N, K):
    """The weights of the weight-streaming tiles go by gemm_small_nt, whichever kernel has them."""
    ops._sk_reserve(torch.device(gpu))
    o = torch.ops.mlop
    prev = o.gemm_small_nt(-1)
    try:
        for nt in (0, 1, 6, 7):
            o.gemm_small_nt(nt)
            assert o.gemm_plan(M, N, K)[4] == (nt & 1)
    finally:
        o.gemm_small_nt(prev)


@pytest.mark.parametrize("M", [5, 16, 32, 64, 65])
@pytest.mark.parametrize("N", [6144, 28672, 49152])
def test_small_tile_switch(gpu, M, N):
    """gemm_small_tile's tiles are what runs at up to 64 rows, on wide weights too."""
    prev = torch.ops.mlop.gemm_small_tile()
    try:
        for tile, bn in ((0, 64), (32, 32), (64, 64)):
            torch.ops.mlop.gemm_small_tile(tile)
            v, bm, n = torch.ops.mlop.gemm_plan(M, N, 4096)[:3]
            if M <= 64:
                assert (v, n, bm) == (0, bn, 64 if tile == 0 else 16 if M <= 16 else 32 if M <= 32 else 64)
    finally:
        torch.ops.mlop.gemm_small_tile(prev)


@pytest.mark.parametrize("bm,rows", [(-1, 128), (0, 128), (64, 128), (128, 128), (160, 160), (192, 192), (224, 224), (256, 128)])
def test_four_wave_override(gpu, bm, rows):
    """Variant 6 takes any tile height, as ever: the three between as they are, the half height for all others."""
    ops._sk_reserve(torch.device(gpu))
    x = torch.randn(300, 256, device=gpu, dtype=bf)
    w = (0.05 * torch.randn(512, 256, device=gpu)).to(bf)
    try:
        torch.ops.mlop.gemm_dense_plan(6, bm, 256, -1)
        assert torch.ops.mlop.gemm_plan(300, 512, 256)[:3] == [6, rows, 256]
        y = ops.gemm(x, w)
    finally:
        torch.ops.mlop.gemm_dense_plan(-1, -1, -1, -1)
    z = x.float() @ w.float().t()
    assert ((y.float() - z).abs() <= 2.0 ** -8 * z.abs() + 2.0 ** -19 * (x.float().abs() @ w.float().abs().t()) + 1e-6).all()
