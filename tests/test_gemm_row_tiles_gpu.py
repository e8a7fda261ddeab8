"""The LDS-ring GEMM's tiles of 96 and 192 rows against fp32: the edges of their row ranges and of 16-row blocks, K in
several ranges and in one, a ragged last column tile, the gate / up unit, the residual add + norm of the reduce."""
import pytest
import torch

from mlopamd import ops

pytestmark = pytest.mark.gpu
bf = torch.bfloat16


@pytest.mark.parametrize("M,bm", [(65, 96), (80, 96), (81, 96), (96, 96), (129, 192), (161, 192), (176, 192), (177, 192), (192, 192)])
@pytest.mark.parametrize("N,K,epi", [(2048, 4096, 0), (4096, 2048, 0), (1032, 1088, 0), (4096, 2048, 1), (1024, 192, 1), (264, 64, 0)])
def test_row_tiles(gpu, M, bm, N, K, epi):
    ops._sk_reserve(torch.device(gpu))
    p = torch.ops.mlop.gemm_plan(M, N, K)
    assert p[0] == 0 and p[1] == bm and p[2] == 64
    torch.manual_seed(M + N + K)
    x = torch.randn(M, K + 8, device=gpu, dtype=bf)[:, :K]
    w = (0.05 * torch.randn(N, K, device=gpu)).to(bf)
    outs = [ops.gemm(x, w, epi=epi) for _ in range(3)]
    y = x.float() @ w.float().t()
    sums = 2.0 ** -20 * (x.float().abs() @ w.float().abs().t())  # fp32 sums in another order
    if epi:  # roundings of gate, up, silu(gate) and the product
        g, u = ops.deinterleave_cols(y).chunk(2, -1)
        sg, su = ops.deinterleave_cols(sums).chunk(2, -1)
        exp, bound = g * g.sigmoid() * u, 4 * 2.0 ** -8 * g.abs() * u.abs() + sg * u.abs() + su * g.abs()
    else:
        exp, bound = y, 2.0 ** -8 * y.abs() + 2 * sums
    assert ((outs[0].float() - exp).abs() <= bound + 1e-6).all()
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


@pytest.mark.parametrize("M", [66, 96, 150, 192])
def test_add_norm(gpu, M):
    N = K = 4096
    torch.manual_seed(M)
    x, r0 = torch.randn(M, K, device=gpu, dtype=bf), torch.randn(M, N, device=gpu, dtype=bf)
    w, g = (0.02 * torch.randn(N, K, device=gpu)).to(bf), torch.rand(N, device=gpu).to(bf)
    res = r0.clone()
    out = ops.gemm_add_rmsnorm(x, w, res, g, 1e-5)
    y = x.float() @ w.float().t()
    exp = r0.float() + y
    assert ((res.float() - exp).abs() <= 2.0 ** -8 * (exp.abs() + y.abs()) + 1e-3).all()  # the product's and the sum's rounding
    z = res.float() * torch.rsqrt(res.float().pow(2).mean(-1, keepdim=True) + 1e-5) * g.float()
    torch.testing.assert_close(out.float(), z, rtol=2.0 ** -7, atol=1e-3)
