"""k_w4r_gemm of up to 64 rows with one strip per wave: strips that do not fill the last workgroup, one split and two, four, seven, steps in whole fours and not, shapes that keep two strips.
One rounding to T of sums of K products that are good to K 2^-24: against float64 of the dequantised weights."""
import pytest
import torch

from proxy_inference_engine_amd import hip_ops as ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N,K", [(32, 256), (96, 1024), (160, 2048), (4128, 4096), (5120, 3072), (1024, 7168), (6144, 4096), (16416, 512)])
@pytest.mark.parametrize("M", [6, 32, 33, 64])
def test_against_the_dequantised_weights(M, N, K, dtype):
    g = torch.Generator(device="cuda").manual_seed(N + K)
    codes, scales, biases = ops.quantize((torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).to(dtype))
    x = torch.randn(M, K, generator=g, device="cuda").to(dtype)
    q = torch.stack([(codes.view(torch.int32) >> (4 * i)) & 15 for i in range(8)], dim=-1).reshape(N, K // 64, 64).float()
    w = (q * scales.float().unsqueeze(-1) + biases.float().unsqueeze(-1)).to(dtype).double().view(N, K)   # (the product is exact, the sum rounded to fp32 and then to T: mx.dequantize)
    want = x.double() @ w.t()
    got = ops.quantized_matmul_rows(x, ops.repack_w4s(codes, scales, biases))
    bound = want.abs() * 2.0 ** (-8 if dtype == torch.bfloat16 else -11) + K * 2.0 ** -24 * (x.double().abs() @ w.abs().t())
    assert bool(((got.double() - want).abs() <= bound).all())


@pytest.mark.parametrize("N,K", [(96, 1024), (320, 5120), (224, 2880), (1024, 7168), (4096, 14336), (6176, 4096)])
@pytest.mark.parametrize("M", [65, 100, 128, 160, 192, 256])
def test_many_rows_against_the_dequantised_weights(M, N, K):
    """Row blocks of three to eight, rings of four, three and two steps: one split (23 steps are a prime number) and up to sixteen, whole rounds of the ring and not."""
    test_against_the_dequantised_weights(M, N, K, torch.bfloat16)
