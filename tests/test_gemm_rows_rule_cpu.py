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


ADD_NORM = {  # and with the residual add and the norm behind the product
    (16, 512, 2048): 0.965, (9, 512, 4096): 1.084, (16, 1024, 2048): 0.97, (12, 1024, 4096): 1.08, (16, 1024, 8192): 1.37, (5, 1536, 4096): 0.915,
    (16, 2048, 2048): 0.86, (12, 2048, 8192): 1.10, (9, 2560, 4096): 0.907, (14, 2560, 8192): 1.056, (9, 3072, 8192): 0.934, (14, 3072, 9216): 1.072,
    (5, 3072, 11008): 0.834, (16, 3072, 14336): 1.157, (12, 4096, 11008): 0.90, (16, 4096, 4096): 0.89, (14, 4096, 28672): 1.055, (5, 4096, 28672): 0.956,
    (16, 5120, 14336): 0.62, (16, 8192, 8192): 0.8, (8, 1024, 3584): 1.06, (6, 4352, 5120): 1.05, (13, 4352, 14336): 1.19, (5, 1792, 9856): 1.15,
    (6, 1280, 512): 0.77, (5, 1920, 512): 0.81, (8, 640, 1024): 0.93,
}


@pytest.mark.parametrize("shape", ADD_NORM, ids=str)
def test_add_norm(shape):
    assert torch.ops.mlop.gemm_on_ws(*shape, 5) == (ADD_NORM[shape] < 1)


ROPE = {  # QKV + RoPE + cache
    (5, 768, 1024): 0.55, (8, 384, 2048): 0.6, (16, 1024, 1024): 0.476, (32, 768, 4096): 0.90, (32, 768, 6144): 1.14, (20, 1280, 8192): 1.21, (28, 1280, 5120): 1.15,
    (12, 1280, 8192): 0.997, (16, 1280, 8192): 1.055, (16, 1536, 8192): 0.95, (20, 1536, 8192): 1.06, (20, 2048, 5120): 0.943, (28, 2048, 6144): 1.04,
    (20, 2560, 7168): 0.982, (32, 2560, 8192): 1.17, (24, 3072, 8192): 0.943, (32, 3840, 6144): 0.958, (24, 4096, 8192): 0.803, (17, 5120, 5120): 1.035,
    (32, 5120, 8192): 1.10, (32, 5120, 4096): 0.978, (32, 6144, 4096): 0.838, (32, 7168, 8192): 0.836, (32, 8192, 6144): 0.93, (20, 10240, 6144): 0.951,
    (32, 9216, 7168): 1.08, (24, 10240, 8192): 0.945, (16, 4864, 7168): 1.0, (16, 6144, 4096): 0.74,
    (25, 3072, 7808): 1.115, (32, 4096, 8064): 1.114, (18, 2304, 7552): 1.08, (26, 3072, 7168): 1.064, (28, 4096, 7936): 1.052, (26, 2560, 5760): 1.068,
    (20, 3072, 5888): 0.865, (19, 3712, 4608): 0.812, (19, 3328, 8192): 0.815,
}


@pytest.mark.parametrize("shape", ROPE, ids=str)
def test_rope(shape):
    assert torch.ops.mlop.gemm_on_ws(*shape, 3) == (ROPE[shape] <= 1)


@pytest.mark.parametrize("N,bm", [(24640, 32), (32768, 32), (32832, 64), (36864, 64), (40832, 64), (40960, 32), (48832, 32), (50304, 32)])
def test_rows_of_the_weight_stream(N, bm):
    """Its 32-row tiles, slower than those of 64 where few CUs have a second one."""
    for M in (17, 32):
        assert torch.ops.mlop.gemm_plan(M, N, 4096)[:2] == [7, bm]
    assert torch.ops.mlop.gemm_plan(33, N, 4096)[:2] == [7, 64]


def test_few_rows_use_no_scratch():
    """Up to 256 rows a product may run beside another stream's that uses the four-wave and grouped kernels' scratch for partial tiles
    (captured decode steps of Dibedra: experts beside the dense products), so none of its tiles is cut into K-halves."""
    four_wave = 0
    for M in (129, 150, 160, 161, 192, 193, 224, 225, 256):
        for N in range(16384, 163841, 256):
            for K in (1024, 1088, 2048, 4096, 8192):
                if N * K >= 1 << 30:
                    continue
                for epi in (0, 1):
                    variant, bm = torch.ops.mlop.gemm_plan(M, N, K, epi)[:2]
                    if variant not in (5, 6):
                        continue
                    four_wave += 1
                    tail = -(-M // bm) * (N // 256) % 256
                    assert tail == 0 or 2 * tail > 256 or K // 64 % 2, (M, N, K, epi)
    assert four_wave > 0


FEW = {  # (M, N, K, SiLU-mul): four-wave kernel's time over the weight stream's or the 256 x 128 tiles'
    (240, 28672, 4096, 1): 0.85, (256, 28672, 4096, 1): 0.87, (225, 28672, 4096, 1): 0.87, (190, 28672, 4096, 1): 1.10, (160, 28672, 4096, 1): 1.15,
    (240, 57344, 8192, 1): 0.97, (256, 57344, 8192, 1): 0.98, (190, 57344, 8192, 1): 1.07, (150, 57344, 8192, 1): 1.09,
    (197, 57344, 4096, 0): 1.09, (210, 57344, 4096, 1): 1.10, (224, 57344, 4096, 0): 1.07, (150, 57344, 4096, 1): 1.3, (190, 49152, 4096, 1): 1.09,
    (200, 49152, 3072, 0): 0.95, (210, 49152, 3072, 0): 0.95, (225, 128256, 4096, 0): 0.85, (256, 128256, 4096, 0): 0.89, (160, 128256, 4096, 0): 1.02,
    (150, 36864, 4096, 1): 0.81, (200, 36864, 4096, 1): 0.71, (256, 36864, 4096, 1): 0.71, (150, 20480, 4096, 1): 0.86, (256, 20480, 4096, 1): 0.90,
    (242, 72704, 5312, 1): 0.89, (239, 97024, 2048, 0): 0.81, (245, 18688, 1024, 1): 0.78, (191, 33280, 1024, 0): 0.67,
}


@pytest.mark.parametrize("shape", FEW, ids=str)
def test_few_rows(shape):
    """gate_up and heads of 129 - 256 rows: on the four-wave kernel where it is faster by more than 3 %, not where it is slower so."""
    assert (torch.ops.mlop.gemm_plan(*shape)[0] in (5, 6)) == (FEW[shape] < 1), FEW[shape]


@pytest.mark.parametrize("N,K,epi,over", [(28672, 4096, 1, 225), (57344, 8192, 1, 225), (128256, 4096, 0, 225), (128256, 8192, 0, 225), (36864, 4096, 1, 129)])
def test_few_rows_change_over(N, K, epi, over):
    """Where the rule leaves the weight stream; heads at 193 - 224 rows are among what it leaves there."""
    assert [M for M in range(120, 257) if torch.ops.mlop.gemm_plan(M, N, K, epi)[0] in (5, 6)] == list(range(over, 257))
