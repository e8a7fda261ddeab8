"""The rule by which products of 2 - 32 rows go to the weight-streaming kernel (gemm_ws.hip ws_fast), against what both forms
measured: shapes where that kernel is at least 3 % slower stay off it, those where it is 3 % faster are on it."""
import pytest
import torch

from mlopamd import ops

pytestmark = pytest.mark.skipif(not ops.available(), reason="the extension is not built")

PLAIN = {  # (M, N, K): weight-streaming kernel's time over the planner's
    (5, 256, 4096): 0.66, (16, 512, 4096): 0.80, (16, 768, 6144): 0.96, (9, 1024, 8192): 0.93, (16, 256, 8192): 1.044, (12, 768, 9216): 1.09,
    (16, 1024, 9216): 1.155, (16, 1280, 6144): 0.90, (14, 2048, 8192): 0.91, (9, 1280, 9216): 0.94, (14, 1536, 9216): 1.05, (16, 2560, 8192): 0.89,
    (16, 3072, 9216): 0.96, (8, 3072, 14336): 0.93, (16, 3072, 14336): 1.06, (9, 3072, 28672): 1.05, (16, 3072, 28672): 1.165, (16, 3584, 14336): 0.96,
    (9, 3584, 28672): 0.97, (14, 3584, 28672): 1.032, (8, 4096, 28672): 0.94, (16, 4096, 14336): 0.954, (16, 5120, 14336): 0.61, (16, 6144, 4096): 0.75,
    (16, 8192, 512): 0.90, (16, 10240, 256): 0.88, (5, 16384, 512): 1.12, (16, 65536, 256): 1.285, (9, 128256, 768): 1.06, (16, 40960, 1024): 0.85,
    (8, 128256, 1024): 0.88, (12, 24576, 3072): 0.96, (16, 28672, 4096): 1.078, (9, 30016, 5120): 1.06, (16, 50304, 3072): 1.048, (8, 28672, 4096): 0.98,
    (6, 4480, 17024): 1.115, (7, 4192, 8192): 0.94, (12, 4416, 9088): 1.05, (16, 4224, 4096): 0.9, (2, 4256, 4736): 1.09, (2, 8480, 11136): 1.10,
    (2, 12704, 8192): 1.10, (2, 5120, 4096): 0.94, (2, 9216, 2048): 0.85, (2, 14336, 4096): 0.91, (2, 4096, 14336): 0.89, (2, 8192, 4096): 0.89,
}


@pytest.mark.parametrize("shape", PLAIN, ids=str)
def test_plain(shape):
    ratio = PLAIN[shape]
    for epi in (0, 1):
        assert torch.ops.mlop.gemm_on_ws(*shape, epi) == (ratio < 1), ratio
