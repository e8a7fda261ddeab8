"""RMSNorm on either side of the row counts from which a wave takes a row (norm.hip wave_rows)."""
import pytest
import torch

from mlopamd import ops
from mlopamd.ops import reference as ref

pytestmark = pytest.mark.gpu
bf = torch.bfloat16


@pytest.mark.parametrize("M,H", [(255, 512), (256, 512), (257, 1024), (3199, 2048), (3201, 2048), (699, 4096), (702, 4096), (1025, 8192)])
def test_either_side(gpu, M, H):
    torch.manual_seed(M)
    x, r = (torch.randn(M, H, device=gpu, dtype=bf) for _ in range(2))
    w = (1 + 0.1 * torch.randn(H, device=gpu)).to(bf)
    y_ref, r_ref = ref.add_rmsnorm(x, r, w, 1e-5)
    # the factor's last bit may turn the rounding of x * factor, and that the rounding of its product with w: an ulp each
    tol = dict(atol=0.0, rtol=2.0 ** -6)
    y = ops.add_rmsnorm(x, r, w, 1e-5)
    assert torch.equal(r, r_ref)
    torch.testing.assert_close(y.float(), y_ref.float(), **tol)
    torch.testing.assert_close(ops.rmsnorm(x, w, 1e-5).float(), ref.rmsnorm(x, w, 1e-5).float(), **tol)


# where every CU has one workgroup of four rows: its ends, and the rows of 2048 without an add that begin before them
@pytest.mark.parametrize("M,H", [(399, 2048), (401, 2048), (768, 2048), (769, 2048), (1024, 2048), (1025, 2048), (704, 8192), (705, 8192), (1022, 8192),
                                 (1024, 8192)])
def test_one_workgroup_each(gpu, M, H):
    test_either_side(gpu, M, H)
