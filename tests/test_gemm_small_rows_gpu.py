"""Which kernel has a product of 1 - 32 rows: the weight-streaming kernel (gemm_ws.hip), the GEMV or the planner's tiles, and
what the switches that ask for one of them do."""
import pytest
import torch

from mlopamd import ops

pytestmark = pytest.mark.gpu
bf = torch.bfloat16


def operands(gpu, M, N, K):
    torch.manual_seed(M + N + K)
    return torch.randn(M, K, device=gpu, dtype=bf), (0.02 * torch.randn(N, K, device=gpu)).to(bf)


@pytest.fixture
def switches(gpu):
    """Every switch of the products as it was, whatever the test set."""
    o = torch.ops.mlop
    ops._sk_reserve(torch.device(gpu))
    prev = {f: f(-1) for f in (o.gemm_ws_max_m, o.gemm_small_tile, o.gemm_small_nt)}
    yield
    for f, v in prev.items():
        f(v)
    o.gemm_dense_plan(-1, -1, -1, -1)


@pytest.mark.parametrize("switch", [("gemm_small_tile", 32), ("gemm_small_nt", 6), ("gemm_dense_plan", 0, 64, 64, 2)], ids=lambda s: s[0])
@pytest.mark.parametrize("M", [5, 9, 16])
@pytest.mark.parametrize("N,K", [(6144, 4096), (4096, 4096)])
def test_switches_are_followed(gpu, switches, M, N, K, switch):
    """A product on a tile that a switch asks for is the same with the weight-streaming kernel on as without it: bit for bit,
    plain, gate / up and with the residual add + norm."""
    x, w = operands(gpu, M, N, K)
    r0, g = torch.randn(M, N, device=gpu, dtype=bf), torch.ones(N, device=gpu, dtype=bf)

    def outs():
        r = r0.clone()
        return [ops.gemm(x, w), ops.gemm(x, w, epi=ops.EPI_SILU_MUL), ops.gemm_add_rmsnorm(x, w, r, g, 1e-5), r]

    getattr(torch.ops.mlop, switch[0])(*switch[1:])
    on = outs()
    torch.ops.mlop.gemm_ws_max_m(0)
    assert all(torch.equal(a, b) for a, b in zip(on, outs()))
