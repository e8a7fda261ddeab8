"""The QKV projection's split-K slabs summed by the RoPE + cache kernel: every count of slabs around a batch of four."""
import pytest
import torch

from mlopamd import ops
from mlopamd.models.layers import rope_table
from mlopamd.ops import reference as ref

pytestmark = pytest.mark.gpu
bf = torch.bfloat16


@pytest.mark.parametrize("splits", [2, 3, 4, 5, 7, 8])
@pytest.mark.parametrize("M", [17, 65])
def test_slabs(gpu, splits, M):
    Hq, Hkv, D, K, BS = 32, 8, 128, 4096, 16
    torch.manual_seed(M + splits)
    cs = rope_table(D, 8192, 5e5, device=gpu)
    x = torch.randn(M, K, device=gpu, dtype=bf)
    w = (0.03 * torch.randn((Hq + 2 * Hkv) * D, K, device=gpu)).to(bf)
    pos = torch.randint(0, 8000, (M,), device=gpu, dtype=torch.int32)
    slots = torch.randperm((M // BS + 2) * BS, device=gpu)[:M].to(torch.int32)
    slots[3] = -1
    kc = torch.zeros(M // BS + 2, Hkv, BS, D, device=gpu, dtype=bf)
    vc = torch.zeros_like(kc)
    q = torch.empty(M, Hq, D, device=gpu, dtype=bf)
    ops._sk_reserve(torch.device(gpu))
    torch.ops.mlop.gemm_dense_plan(0, 64, 64, splits)
    try:
        assert torch.ops.mlop.gemm_rope_cache(q, kc, vc, x, w, pos, cs, slots)
    finally:
        torch.ops.mlop.gemm_dense_plan(-1, -1, -1, -1)
    kr, vr = torch.zeros_like(kc).cpu(), torch.zeros_like(vc).cpu()
    qr = ref.rope_cache((x.float() @ w.float().t()).to(bf).cpu(), pos.cpu(), cs.cpu(), slots.cpu(), kr, vr, Hq)
    for got, want in ((q, qr), (kc, kr), (vc, vr)):  # the product's rounding may fall the other way: one ulp, rotated
        torch.testing.assert_close(got.float().cpu(), want.float(), atol=2e-2, rtol=2e-2)
