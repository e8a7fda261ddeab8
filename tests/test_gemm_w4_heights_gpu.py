"""The four-wave GEMM's 160- and 192-row tiles (gemm_w4.hip) against fp32: every epilogue, row counts around a tile and
a 16-row block, the shortest K of the peeled loop, whole rounds with the next tile prefetched, K-half tails."""
import pytest
import torch

from mlopamd import ops
from mlopamd.ops import reference as ref

pytestmark = pytest.mark.gpu
bf = torch.bfloat16


@pytest.fixture(params=[160, 192, 224])
def height(gpu, request):
    ops._sk_reserve(torch.device(gpu))
    torch.ops.mlop.gemm_dense_plan(6, request.param, 256, -1)
    try:
        yield request.param
    finally:
        torch.ops.mlop.gemm_dense_plan(-1, -1, -1, -1)


# M in tiles of the height plus an offset: one row, the 16-row blocks' edges, a full tile, several
@pytest.mark.parametrize("tiles,off,N,K", [(0, 1, 256, 192), (0, 17, 512, 256), (0, 159, 256, 320), (1, 0, 768, 192), (1, 1, 256, 448),
                                           (2, -16, 512, 192), (3, 5, 20736, 256), (7, -3, 12288, 192), (16, 0, 4096, 256), (4, 9, 6144, 4096)])
@pytest.mark.parametrize("epi", [0, 1, 8])
def test_tiles(gpu, height, tiles, off, N, K, epi):
    M = tiles * height + off
    torch.manual_seed(M + N + K)
    x = torch.randn(M, K, device=gpu, dtype=bf)
    w = (0.05 * torch.randn(N, K, device=gpu)).to(bf)
    kw = {"act_from": 128} if epi == 8 else {}
    outs = [ops.gemm(x, w, epi=epi, **kw) for _ in range(3)]
    y = x.float() @ w.float().t()
    sums = 2.0 ** -20 * (x.float().abs() @ w.float().abs().t())  # fp32 sums in another order
    if epi == 1:  # roundings of gate, up, silu(gate) and the product
        g, u = ops.deinterleave_cols(y).chunk(2, -1)
        sg, su = ops.deinterleave_cols(sums).chunk(2, -1)
        exp, bound = g * g.sigmoid() * u, 4 * 2.0 ** -8 * g.abs() * u.abs() + sg * u.abs() + su * g.abs()
    else:
        exp = torch.cat([y[:, :128], ref.gelu_tanh(y[:, 128:])], -1) if epi else y
        bound = 2.0 ** -8 * exp.abs() + 2 * sums
    assert ((outs[0].float() - exp).abs() <= bound + 1e-6).all()
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


@pytest.mark.parametrize("variant,bm", [(6, 128), (6, 160), (6, 192), (6, 224), (5, 256)])
@pytest.mark.parametrize("off", [1, 8, 9, 100])
@pytest.mark.parametrize("epi", [0, 1])
def test_rows_past_the_last(gpu, variant, bm, off, epi):
    """Rows past A's last load nothing: what the LDS holds there (here a product of NaN before) reaches no output, and
    the waits that count the dropped loads still cover the others, a workgroup's next tile's among them (513 tiles: two or three
    each, a third of them partial, behind whole ones and before them)."""
    N, K, M = 171 * 256, 448, 2 * bm + off
    torch.manual_seed(M)
    w = (0.05 * torch.randn(N, K, device=gpu)).to(bf)
    nan = torch.full((4 * bm, K), float("nan"), device=gpu, dtype=bf)
    x = torch.randn(M, K, device=gpu, dtype=bf)
    ops._sk_reserve(torch.device(gpu))
    torch.ops.mlop.gemm_dense_plan(variant, bm, 256, -1)
    try:
        whole = ops.gemm(torch.cat([x, x, x])[:3 * bm], w, epi=epi)[:M]  # the same rows with no partial tile
        for _ in range(4):
            ops.gemm(nan, w)
            assert torch.equal(ops.gemm(x, w, epi=epi), whole)
    finally:
        torch.ops.mlop.gemm_dense_plan(-1, -1, -1, -1)


# K a multiple of 2048 and not, halves of it, several bands of tiles; weights that the cache behind the L2s holds and not
@pytest.mark.parametrize("M,N,K", [(130, 512, 2048), (130, 512, 2112), (700, 4096, 2048), (1300, 6144, 4096), (257, 16384, 10240),
                                   (1000, 8192, 18432)])
def test_k_walk(gpu, height, M, N, K):
    """XCDs start at different eighths of K: the same sums in another order, and the same ones every time."""
    torch.manual_seed(M + K)
    x = torch.randn(M, K, device=gpu, dtype=bf)
    w = (0.05 * torch.randn(N, K, device=gpu)).to(bf)
    outs = [ops.gemm(x, w) for _ in range(3)]
    y = x.float() @ w.float().t()
    bound = 2.0 ** -8 * y.abs() + 2 * 2.0 ** -20 * (x.float().abs() @ w.float().abs().t())
    assert ((outs[0].float() - y).abs() <= bound + 1e-6).all()
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


@pytest.mark.parametrize("M", [300, 1500])
def test_rope(gpu, height, M):
    from mlopamd.models.layers import rope_table

    Hq, Hkv, D, K, BS = 32, 8, 128, 1024, 16
    torch.manual_seed(M)
    cs = rope_table(D, 8192, 5e5, device=gpu)
    x = torch.randn(M, K, device=gpu, dtype=bf)
    w = (0.03 * torch.randn((Hq + 2 * Hkv) * D, K, device=gpu)).to(bf)
    pos = torch.randint(0, 8000, (M,), device=gpu, dtype=torch.int32)
    slots = torch.randperm((M // BS + 8) * BS, device=gpu)[:M].to(torch.int32)
    slots[5] = slots[M - 1] = -1
    kc = torch.zeros(M // BS + 8, Hkv, BS, D, device=gpu, dtype=bf)
    vc = torch.zeros_like(kc)
    q = torch.empty(M, Hq, D, device=gpu, dtype=bf)
    assert torch.ops.mlop.gemm_rope_cache(q, kc, vc, x, w, pos, cs, slots)
    kr, vr = torch.zeros_like(kc).cpu(), torch.zeros_like(vc).cpu()
    qr = ref.rope_cache((x.float() @ w.float().t()).to(bf).cpu(), pos.cpu(), cs.cpu(), slots.cpu(), kr, vr, Hq)
    for got, want in ((q, qr), (kc, kr), (vc, vr)):  # the product's rounding may fall the other way: one ulp, rotated
        torch.testing.assert_close(got.float().cpu(), want.float(), atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("M", [161, 500, 1537])
def test_norm_chain(gpu, height, M):
    """Residual add with row sums of squares, then the products that scale their rows by them."""
    H, eps = 4096, 1e-5
    assert torch.ops.mlop.w4_chain_ok(M, H, 512) and torch.ops.mlop.w4_chain_ok(M, 512, H)
    torch.manual_seed(M)
    a = torch.randn(M, 512, device=gpu, dtype=bf)
    w = (0.05 * torch.randn(H, 512, device=gpu)).to(bf)
    r0 = torch.randn(M, H, device=gpu, dtype=bf)
    y = r0.float() + a.float() @ w.float().t()
    for _ in range(2):
        res, ss = r0.clone(), ops.ss_buffer(M, H, gpu)
        ops.gemm_res_ss(a, w, res, ss)
        assert ((res.float() - y).abs() <= 2.0 ** -8 * y.abs() + 2.0 ** -7 * (a.float() @ w.float().t()).abs() + 1e-3).all()
        tot = ops.ss_parts(ss, M, H)[1]
        torch.testing.assert_close(tot, res.float().pow(2).sum(-1), rtol=1e-4, atol=0)
        unit = res.float() * torch.rsqrt(res.float().pow(2).mean(-1, keepdim=True) + eps)
        for epi in (0, 1):
            w2 = (0.02 * torch.randn(512, H, device=gpu)).to(bf)
            got, z = ops.gemm_rs(res, w2, ss, eps, epi).float(), unit @ w2.float().t()
            if epi:
                g, u = ops.deinterleave_cols(z).chunk(2, -1)
                z = g * g.sigmoid() * u
                bound = 5 * 2.0 ** -8 * g.abs() * u.abs()
            else:
                bound = 2.0 ** -8 * z.abs()
            assert ((got - z).abs() <= bound + 2e-3).all()


# a tile with rows past M, then another on the same workgroup, at short K (the next tile's first K-tile is in flight)
@pytest.mark.parametrize("variant,bm", [(6, 128), (6, 160), (6, 192), (6, 224), (5, 256)])
@pytest.mark.parametrize("tiles,off", [(1, 1), (2, 17), (5, 3)])
@pytest.mark.parametrize("K", [192, 448])
def test_tile_after_a_partial_one(gpu, variant, bm, tiles, off, K):
    M, N = tiles * bm + off, 32768
    torch.manual_seed(M + K)
    x = torch.randn(M, K, device=gpu, dtype=bf)
    w = (0.05 * torch.randn(N, K, device=gpu)).to(bf)
    y = x.float() @ w.float().t()
    bound = 2.0 ** -8 * y.abs() + 2.0 ** -19 * (x.float().abs() @ w.float().abs().t()) + 1e-6
    ops._sk_reserve(torch.device(gpu))
    torch.ops.mlop.gemm_dense_plan(variant, bm, 256, -1)
    try:
        for _ in range(30):
            assert ((ops.gemm(x, w).float() - y).abs() <= bound).all()
    finally:
        torch.ops.mlop.gemm_dense_plan(-1, -1, -1, -1)
