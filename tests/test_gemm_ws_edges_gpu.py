"""The weight-streaming MFMA GEMM (gemm_ws.hip) where its steps, images and row blocks end: 1 - 16 rows, K of one step
up to a last round that not every wave has, 16 and 32 weight rows per workgroup, A's rows in a wider matrix."""
import pytest
import torch

from mlopamd import ops

pytestmark = pytest.mark.gpu
bf = torch.bfloat16
EPS = 1e-5


@pytest.fixture
def plan(gpu, request):
    torch.ops.mlop.gemm_ws_plan(*request.param)
    yield
    torch.ops.mlop.gemm_ws_plan(0, 0)


def bound(y, a, w, K):
    """bf16 result of fp32 sums: half an ulp of the result and of the sums' bf16 rounding before an add, and K / 32
    accumulations (the matrix cores add 32 products at a time) plus the waves' eight, each off by at most 2^-23 of the sum of
    magnitudes."""
    return 2.0 ** -7 * y.abs() + (K / 32 + 16) * 2.0 ** -23 * (a.abs() @ w.abs().t()) + 1e-6


@pytest.mark.parametrize("plan", [(1, 1), (1, 2), (2, 1), (2, 2)], indirect=True, ids=["16x1", "16x2", "32x1", "32x2"])
@pytest.mark.parametrize("M", [1, 2, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("N,K", [(32, 128), (96, 1024), (160, 1152), (64, 2176), (1056, 4096)])
def test_ends(gpu, plan, M, N, K):
    torch.manual_seed(M * N + K)
    wide = torch.full((M, K + 64), float("nan"), device=gpu, dtype=bf)  # what follows a row must not reach the sums
    a = wide[:, :K]
    a.copy_(torch.randn(M, K, device=gpu))
    guard = torch.full((N + 32, K), float("nan"), device=gpu, dtype=bf)
    w = guard[:N]
    w.copy_(0.05 * torch.randn(N, K, device=gpu))
    ad, wd = a.double(), w.double()
    y = ad @ wd.t()
    out = torch.full((M + 1, N), 7.0, device=gpu, dtype=bf)
    assert torch.ops.mlop.gemm_ws(out[:M], a, w, 0, False, 0.0)
    assert bool(((out[:M].double() - y).abs() <= bound(y, ad, wd, K)).all())
    assert bool((out[M:] == 7.0).all())
    # residual form
    r0 = torch.randn(M, N, device=gpu, dtype=bf)
    r = r0.clone()
    assert torch.ops.mlop.gemm_ws(r, a, w, 5, False, 0.0)
    z = r0.double() + y
    assert bool(((r.double() - z).abs() <= bound(z, ad, wd, K) + 2.0 ** -8 * y.abs()).all())
    # gate / up of rows scaled by their RMSNorm factor
    s = torch.empty(M, N // 2, device=gpu, dtype=bf)
    assert torch.ops.mlop.gemm_ws(s, a, w, 1, True, EPS)
    f = torch.rsqrt(ad.square().mean(-1, keepdim=True) + EPS)
    gu = (y * f).view(M, N // 32, 2, 16)
    g, u = gu[:, :, 0].reshape(M, -1), gu[:, :, 1].reshape(M, -1)
    exp = g * g.sigmoid() * u
    # gate, up and the activation are rounded to bf16 before the product is
    assert bool(((s.double() - exp).abs() <= 2.0 ** -6 * exp.abs() + 2.0 ** -7 * u.abs() * g.abs() + 1e-5).all())


def test_infinities_stay_in_their_row(gpu):
    """An infinite activation makes its own row's sums infinite or NaN and no other's, also where the row lies in a step
    that fewer waves have."""
    M, N, K = 5, 64, 1152
    a = torch.randn(M, K, device=gpu, dtype=bf)
    w = (0.05 * torch.randn(N, K, device=gpu)).to(bf)
    a[2, K - 1] = float("inf")
    out = torch.empty(M, N, device=gpu, dtype=bf)
    assert torch.ops.mlop.gemm_ws(out, a, w, 0, False, 0.0)
    keep = [0, 1, 3, 4]
    assert bool(torch.isfinite(out[keep]).all())
    assert torch.equal(out[2].float(), torch.where(w[:, K - 1] > 0, float("inf"), -float("inf")).float())


@pytest.mark.parametrize("M,N,K", [(1, 65536, 4096), (3, 3072, 2048), (16, 6144, 4096), (9, 320, 1152)])
def test_public_products_take_it(gpu, M, N, K):
    """ops.gemm at the sizes of the rule (and, last, one that is not a whole block of 32 rows)."""
    torch.manual_seed(N)
    a = torch.randn(M, K, device=gpu, dtype=bf)
    w = (0.02 * torch.randn(N, K, device=gpu)).to(bf)
    y = a.double() @ w.double().t()
    assert bool(((ops.gemm(a, w).double() - y).abs() <= bound(y, a.double(), w.double(), K)).all())
