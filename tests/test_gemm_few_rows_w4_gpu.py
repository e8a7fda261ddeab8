"""gate_up and output heads of 129 - 256 rows on the four-wave kernel (few_rows_w4) against fp32, at the edges of its tiles and of
its rule: one tile of the batch's height, two of 128 rows, K that is not whole 2048, the 256 x 128 tiles' sizes, the rows at which
products of the weight stream go over."""
import pytest
import torch

from mlopamd import ops

pytestmark = pytest.mark.gpu
bf = torch.bfloat16


def run(gpu, M, N, K, epi):
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


def height(M):
    """One tile of the batch's height."""
    bm = -(-M // 32) * 32
    return (5 if bm == 256 else 6, bm)


# the kernel that each is to run on: variant and rows, of the weight stream (7) or of four-wave tiles
GATE_UP = {(20480, 1024): lambda M: (6, 128), (36864, 2048): height, (40960, 1088): height,
           (28672, 4096): lambda M: (6, 128) if M > 224 else (7, -(-M // 32) * 32)}
HEAD = {(36864, 2048): height, (40960, 1088): height, (128256, 1024): lambda M: height(M) if M > 192 else (7, -(-M // 32) * 32)}


@pytest.mark.parametrize("M", [129, 160, 161, 193, 224, 225, 255, 256])
@pytest.mark.parametrize("N,K", GATE_UP)
def test_gate_up(gpu, M, N, K):
    ops._sk_reserve(torch.device(gpu))
    assert tuple(torch.ops.mlop.gemm_plan(M, N, K, 1)[:2]) == GATE_UP[N, K](M)
    run(gpu, M, N, K, 1)


@pytest.mark.parametrize("M", [129, 191, 192, 193, 224, 256])
@pytest.mark.parametrize("N,K", HEAD)
def test_head(gpu, M, N, K):
    ops._sk_reserve(torch.device(gpu))
    assert tuple(torch.ops.mlop.gemm_plan(M, N, K)[:2]) == HEAD[N, K](M)
    run(gpu, M, N, K, 0)


def test_rule(gpu):
    """Which kernel a plain product has; gemm_plan says it."""
    ops._sk_reserve(torch.device(gpu))
    plan = lambda *a: tuple(torch.ops.mlop.gemm_plan(*a)[:2])  # noqa: E731
    assert plan(256, 128256, 4096) == (5, 256) and plan(240, 36864, 2048)[0] in (5, 6) and plan(200, 40960, 4096) == (6, 224)
    assert plan(128, 128256, 4096)[0] == 7 and plan(256, 32768, 8192)[0] == 7 and plan(256, 128264, 4096)[0] == 7 and plan(160, 65536, 960)[0] == 7

