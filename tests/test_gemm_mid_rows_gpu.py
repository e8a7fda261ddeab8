"""The weight stream of gemm_mid.hip at up to 64 rows: 32- and 64-row tiles of 128 and 256 columns at the ends of their rows,
columns and rings, the gate / up form that takes its rows' RMSNorm factors itself, and QKV + RoPE at 17 - 32 rows on the
weight-streaming kernel."""
import pytest
import torch

from mlopamd import ops

pytestmark = pytest.mark.gpu
bf = torch.bfloat16
EPS = 1e-5


def operands(gpu, M, N, K):
    torch.manual_seed(M * N + K)
    wide = torch.full((M, K + 64), float("nan"), device=gpu, dtype=bf)  # what follows a row must not reach the sums
    a = wide[:, :K]
    a.copy_(torch.randn(M, K, device=gpu))
    w = torch.full((N + 32, K), float("nan"), device=gpu, dtype=bf)[:N]
    w.copy_(0.05 * torch.randn(N, K, device=gpu))
    return a, w


def bound(y, a, w, K):
    """bf16 result of fp32 sums: half an ulp, and K / 32 accumulations each off by at most 2^-23 of the sum of magnitudes."""
    return 2.0 ** -8 * y.abs() + (K / 32 + 4) * 2.0 ** -23 * (a.abs() @ w.abs().t()) + 1e-6


# 193 column tiles of 128 (and two thirds of one), 320 of them (two workgroups per CU), 193 of 256; one K-step, fewer than a
# ring holds, more
@pytest.mark.parametrize("M", [17, 31, 32, 33, 64])
@pytest.mark.parametrize("N,K", [(24664, 64), (24664, 192), (24664, 1088), (40960, 448), (49240, 64), (49240, 576)])
def test_plain(gpu, M, N, K):
    plan = torch.ops.mlop.gemm_plan(M, N, K)
    assert plan[0] == 7 and plan[1] == (M + 31) // 32 * 32 and plan[2] == (256 if N > 48896 else 128)
    a, w = operands(gpu, M, N, K)
    out = torch.full((M + 1, N), 7.0, device=gpu, dtype=bf)
    torch.ops.mlop.gemm(out[:M], a, w, torch.empty(1, device=gpu), 0)
    ad, wd = a.double(), w.double()
    y = ad @ wd.t()
    assert bool(((out[:M].double() - y).abs() <= bound(y, ad, wd, K)).all())
    assert bool((out[M:] == 7.0).all())


@pytest.mark.parametrize("M", [17, 32])
@pytest.mark.parametrize("N,K", [(32776, 192), (40824, 1088)])
def test_few_second_tiles(gpu, M, N, K):
    """64-row tiles of few rows, where 32-row ones would give some CUs a second one."""
    assert torch.ops.mlop.gemm_plan(M, N, K)[:3] == [7, 64, 128]
    a, w = operands(gpu, M, N, K)
    out = torch.full((M + 1, N), 7.0, device=gpu, dtype=bf)
    torch.ops.mlop.gemm(out[:M], a, w, torch.empty(1, device=gpu), 0)
    ad, wd = a.double(), w.double()
    y = ad @ wd.t()
    assert bool(((out[:M].double() - y).abs() <= bound(y, ad, wd, K)).all())
    assert bool((out[M:] == 7.0).all())


@pytest.mark.parametrize("M", [9, 16, 32, 33, 64])
@pytest.mark.parametrize("N,K", [(24608, 128), (24608, 1152), (40960, 384), (49184, 640)])
def test_gate_up_of_the_residual(gpu, M, N, K):
    a, w = operands(gpu, M, N, K)
    a[M // 2] *= 100.0
    out = torch.full((M + 1, N // 2), 7.0, device=gpu, dtype=bf)
    ss = torch.full((M * (K // 128 + 1),), float("nan"), device=gpu)  # not read
    prev = torch.ops.mlop.gemm_ws_max_m(-1)
    torch.ops.mlop.gemm_ws_max_m(64)
    try:
        assert torch.ops.mlop.gemm_rs(out[:M], a, w, ss, EPS, 1, False)
    finally:
        torch.ops.mlop.gemm_ws_max_m(prev)
    ad, wd = a.double(), w.double()
    y = ad @ wd.t() * torch.rsqrt(ad.square().mean(-1, keepdim=True) + EPS)
    gu = y.view(M, N // 32, 2, 16)
    g, u = gu[:, :, 0].reshape(M, -1), gu[:, :, 1].reshape(M, -1)
    exp = g * g.sigmoid() * u
    # gate, up and the activation are rounded to bf16 before the product is
    assert bool(((out[:M].double() - exp).abs() <= 2.0 ** -6 * exp.abs() + 2.0 ** -7 * u.abs() * g.abs() + 1e-5).all())
    assert bool((out[M:] == 7.0).all())


@pytest.mark.parametrize("M", [17, 23, 32])
@pytest.mark.parametrize("hq,hkv,K", [(32, 8, 1152), (22, 1, 2048)])
def test_qkv_rope(gpu, M, hq, hkv, K):
    from mlopamd.models.layers import rope_table

    D, BS, NB, N = 128, 16, 8, (hq + 2 * hkv) * 128
    a, w = operands(gpu, M, N, K)
    assert torch.ops.mlop.gemm_rope_supported(M, N, K)
    cs = rope_table(D, 512, 10000.0, device=gpu)
    pos = torch.randint(0, 512, (M,), device=gpu, dtype=torch.int32)
    slots = torch.randperm(NB * BS, device=gpu)[:M].to(torch.int32)
    slots[3] = -1  # a row that is not kept
    kc, vc = (torch.full((NB, hkv, BS, D), 3.0, device=gpu, dtype=bf) for _ in range(2))
    q = ops.qkv_rope_cache(a, w, pos, cs, slots, kc, vc, hq)
    qkv = (a.double() @ w.double().t()).float().cpu()
    kr, vr = (torch.full((NB, hkv, BS, D), 3.0) for _ in range(2))
    qr = ops.reference.rope_cache(qkv, pos.cpu(), cs.cpu(), slots.cpu(), kr, vr, hq)
    # the projections' bf16 rounding through a rotation of two of them, and the result's own
    tol = dict(rtol=2.0 ** -8, atol=2.0 ** -8 * float(qkv.abs().max()))
    for x, y in ((q, qr), (kc, kr), (vc, vr)):
        torch.testing.assert_close(x.float().cpu(), y.float(), **tol)
