"""GEMM + residual add + norm over K ranges on the four-wave kernel against fp32: every tile height at the edges of its
rows, ranges of unequal and of least length, rows of x further apart than they are long, and the sizes that the rule takes."""
import pytest
import torch

from mlopamd import ops

pytestmark = pytest.mark.gpu
bf = torch.bfloat16


def check(x, w, g, r0):
    outs = []
    for _ in range(3):
        res = r0.clone()
        outs.append((ops.gemm_add_rmsnorm(x, w, res, g, 1e-5), res))
    (out, res), N = outs[0], w.shape[0]
    y = x.float() @ w.float().t()
    sums = 2.0 ** -20 * (x.float().abs() @ w.float().abs().t())  # fp32 sums in another order
    exp = r0.float() + y
    # the product's rounding and the sum's
    assert ((res.float() - exp).abs() <= 2.0 ** -8 * (exp.abs() + 2 * y.abs()) + 2 * sums + 1e-6).all()
    z = res.float() * torch.rsqrt(res.float().pow(2).mean(-1, keepdim=True) + 1e-5) * g.float()
    assert ((out.float() - z).abs() <= 2.0 ** -7 * z.abs() + 1e-6).all()  # two roundings
    assert all(torch.equal(a, out) and torch.equal(b, res) for a, b in outs) and out.shape == (x.shape[0], N)


def operands(gpu, M, N, K, pad=0):
    torch.manual_seed(M + N + K)
    return (torch.randn(M, K + pad, device=gpu, dtype=bf)[:, :K], (0.05 * torch.randn(N, K, device=gpu)).to(bf),
            (1 + 0.1 * torch.randn(N, device=gpu)).to(bf), torch.randn(M, N, device=gpu, dtype=bf))


@pytest.mark.parametrize("bm", [128, 160, 192, 224, 256])
@pytest.mark.parametrize("tiles,short,N,K,splits", [(1, 0, 256, 384, 2), (2, 1, 512, 704, 3), (3, 15, 768, 1600, 8), (2, 17, 256, 4160, 5)])
def test_tiles(gpu, bm, tiles, short, N, K, splits):
    args = operands(gpu, bm * tiles - short, N, K, 8 * short)
    ops._sk_reserve(torch.device(gpu))
    torch.ops.mlop.gemm_dense_plan(8, bm, 256, splits)
    try:
        assert torch.ops.mlop.gemm_workspace(args[0].shape[0], N, K, 2) == splits * args[0].shape[0] * N
        check(*args)
    finally:
        torch.ops.mlop.gemm_dense_plan(-1, 0, 0, 0)


@pytest.mark.parametrize("M,N,K", [(257, 5120, 13824), (320, 4096, 4096), (385, 1024, 1536), (500, 2048, 8192), (641, 4096, 4096),
                                   (892, 4096, 14336), (1023, 768, 9088), (2100, 1280, 7680)])
def test_rule(gpu, M, N, K):
    ops._sk_reserve(torch.device(gpu))
    assert torch.ops.mlop.gemm_workspace(M, N, K, 2) >= 2 * M * N
    check(*operands(gpu, M, N, K))


@pytest.mark.parametrize("M,N,K", [(256, 5120, 13824), (319, 4096, 4096), (900, 4096, 1472), (8000, 4096, 4096)])
def test_not_taken(gpu, M, N, K):
    """Below and above: what the sizes had before (the small-row plans' ranges, or one product and a pass)."""
    ops._sk_reserve(torch.device(gpu))
    torch.ops.mlop.gemm_dense_plan(8, 128, 256, 1)
    try:
        n = torch.ops.mlop.gemm_workspace(M, N, K, 2)
    finally:
        torch.ops.mlop.gemm_dense_plan(-1, 0, 0, 0)
    assert torch.ops.mlop.gemm_workspace(M, N, K, 2) == n


def test_captured(gpu):
    """Replays of a captured call, the program's own work and synchronisations between them."""
    x, w, g, r0 = operands(gpu, 500, 2048, 8192)
    want = r0.clone()
    out = ops.gemm_add_rmsnorm(x, w, want, g, 1e-5)
    res, graph = r0.clone(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = ops.gemm_add_rmsnorm(x, w, res, g, 1e-5)
    for _ in range(4):
        res.copy_(r0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, out) and torch.equal(res, want)
        other = r0.clone()
        assert torch.equal(ops.gemm_add_rmsnorm(x, w, other, g, 1e-5), out)


def test_rows_too_far_apart(gpu, monkeypatch):
    """Rows of x further apart than the four-wave kernel's offsets reach: the op says no and has written nothing, and the call, with
    or without a tensor for its result, is the product and the norm one behind the other."""
    M, N, K = 400, 4096, 4096
    x, w, g, r0 = operands(gpu, M, N, K)
    n = torch.ops.mlop.gemm_workspace(M, N, K, 2)
    assert n >= 2 * M * N
    far = torch.empty(M, 2_700_000, device=gpu, dtype=bf)[:, :K]
    out, res = torch.zeros(M, N, device=gpu, dtype=bf), r0.clone()
    assert not torch.ops.mlop.gemm_add_rmsnorm(out, res, far, w, g, torch.empty(n, device=gpu), 1e-5)
    assert torch.equal(res, r0) and not out.any()
    del far
    want_res = r0.clone()
    want = ops.add_rmsnorm(ops.gemm(x, w), want_res, g, 1e-5)
    monkeypatch.setattr(torch.ops.mlop, "gemm_add_rmsnorm", lambda *a: False)
    for given in (None, out):
        res = r0.clone()
        got = ops.gemm_add_rmsnorm(x, w, res, g, 1e-5, given)
        assert torch.equal(got, want) and torch.equal(res, want_res) and (given is None or got is given)
