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


@pytest.mark.parametrize("switch", [("gemm_small_tile", 32), ("gemm_dense_plan", 0, 64, 64, 2)], ids=lambda s: s[0])
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


@pytest.mark.parametrize("M", [2, 4, 8, 16])
@pytest.mark.parametrize("N,K", [(6144, 4096), (4096, 1152), (8192, 2176)])
def test_cache_policy_changes_no_bit(gpu, switches, M, N, K):
    """gemm_small_nt is where the weights go, not which kernel multiplies: one and two steps in flight, 16 and 32 rows."""
    o, outs = torch.ops.mlop, []
    x, w = operands(gpu, M, N, K)
    for nt in (7, 6):
        o.gemm_small_nt(nt)
        assert o.gemm_plan(M, N, K) == [-2, 0, 0, 1, nt & 1]
        outs.append([ops.gemm(x, w), ops.gemm(x, w, epi=ops.EPI_SILU_MUL)])
    assert all(torch.equal(a, b) for a, b in zip(*outs))


@pytest.mark.parametrize("M,N,K", [(1, 4096, 4096), (1, 128256, 4096), (2, 6144, 4096), (2, 2048, 4096), (4, 1024, 4096), (4, 4096, 14336),
                                   (5, 6144, 4096), (16, 24576, 4096), (16, 6144, 4160), (16, 256, 1024), (17, 6144, 4096)])
def test_plan_says_what_runs(gpu, switches, M, N, K):
    """gemm_plan's -2 is where a plain product is the weight-streaming kernel's, bit for bit, with no slabs reserved; without
    that kernel it names another form, whose product is in another order."""
    o = torch.ops.mlop
    x, w = operands(gpu, M, N, K)
    y, z = ops.gemm(x, w), torch.empty(M, N, device=gpu, dtype=bf)
    variant = o.gemm_plan(M, N, K)[0]
    if variant == -2:
        assert o.gemm_ws(z, x, w, 0, False, 0.0) and torch.equal(y, z)
        assert o.gemm_workspace(M, N, K, 0) == 0
        o.gemm_ws_max_m(0)
        assert o.gemm_plan(M, N, K)[0] == (-1 if M <= 4 else 0 if N < 24449 else 7)
    else:
        o.gemm_ws_max_m(0)
        assert o.gemm_plan(M, N, K)[0] == variant and torch.equal(ops.gemm(x, w), y)
    assert (variant == -2) == ((M, N, K) in [(1, 128256, 4096), (2, 6144, 4096), (4, 4096, 14336), (5, 6144, 4096), (16, 24576, 4096),
                                             (16, 6144, 4096)])


@pytest.mark.parametrize("M", [2, 3, 4])
def test_rows_off_16_bytes_stay_on_the_gemv(gpu, switches, M):
    """Rows that begin 8 bytes off a multiple of 16 are not for LDS-DMA: QKV + RoPE and the chain's products of up to 4 rows are
    the GEMV's there, bit for bit, and the chain's of more rows are refused."""
    from mlopamd.models.layers import rope_table

    o, K, hq, hkv = torch.ops.mlop, 4096, 32, 8
    N = (hq + 2 * hkv) * 128
    x, w = operands(gpu, 8, 8, K + 8)[0][:, 4:4 + K], operands(gpu, 1, N, K)[1]
    assert x.data_ptr() % 16 == 8 and x.stride(0) % 8 == 0
    cs = rope_table(128, 64, 10000.0, device=gpu)
    pos, slots = torch.arange(M, device=gpu, dtype=torch.int32), torch.arange(M, device=gpu, dtype=torch.int32)

    def outs(a):
        kc, vc = (torch.zeros(2, hkv, 16, 128, device=gpu, dtype=bf) for _ in range(2))
        r, ss = torch.ones(M, K, device=gpu, dtype=bf), ops.ss_buffer(M, K, gpu)
        q = ops.qkv_rope_cache(a, w, pos, cs, slots, kc, vc, hq)
        q2 = ops.qkv_rope_cache_rs(a, w, pos, cs, slots, kc.clone(), vc.clone(), hq, ss, 1e-5)
        ops.gemm_res_ss(a, w[:K], r, ss)
        return q, kc, vc, q2, r, ops.gemm_rs(a, w, ss, 1e-5, ops.EPI_SILU_MUL)

    here = outs(x[:M])
    with pytest.raises(RuntimeError):
        ops.gemm_rs(x, w, ops.ss_buffer(8, K, gpu), 1e-5, ops.EPI_SILU_MUL)
    o.gemm_ws_max_m(0)
    assert all(torch.equal(a, b) for a, b in zip(here, outs(x[:M].clone())))


@pytest.mark.parametrize("M", [3, 4, 8])
def test_rows_far_apart(gpu, M):
    """Rows of A that span more than 32 bits of bytes are not for the weight-streaming kernel, whose offsets have that many."""
    K, N = 512, 4096
    lda = -(-(1 << 31) // (M - 1)) + 64  # elements: the last row begins beyond 2^32 bytes
    lda -= lda % 8
    assert torch.ops.mlop.gemm_on_ws(M, N, K, 0) and (M - 1) * lda * 2 >= 1 << 32
    x = torch.empty((M - 1) * lda + K, device=gpu, dtype=bf).as_strided((M, K), (lda, 1))
    dense, w = operands(gpu, M, N, K)
    x.copy_(dense)
    y = dense.double() @ w.double().t()
    # the result's rounding to bf16, and fp32 sums of K products
    bound = 2.0 ** -8 * y.abs() + K * 2.0 ** -23 * (dense.double().abs() @ w.double().abs().t())
    out = torch.empty(M, N, device=gpu, dtype=bf)
    torch.ops.mlop.gemm(out, x, w, torch.empty(1, device=gpu), 0)
    assert bool(((out.double() - y).abs() <= bound).all())
