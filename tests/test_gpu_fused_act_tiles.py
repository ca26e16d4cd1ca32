"""The gated MLP's product in tiles of one and of two strips per wave: rows on both sides of every tile height, a last tile of a few columns, against 64 bits."""
import pytest
import torch

from proxy_inference_engine_amd import hip_ops as ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,eps", [(torch.bfloat16, 2.0 ** -8), (torch.float16, 2.0 ** -11)])
@pytest.mark.parametrize("half,K", [(68, 128), (1412, 192), (3420, 1280), (8192, 512)])   # (8192: two strips from 509 rows on)
@pytest.mark.parametrize("M", [33, 64, 65, 129, 257, 509])
def test_gated_rows_against_64_bits(M, half, K, dtype, eps):
    g = torch.Generator(device="cuda").manual_seed(half + M)
    x = torch.randn(M, K, generator=g, device="cuda").to(dtype)
    w = (torch.randn(2 * half, K, generator=g, device="cuda") * K ** -0.5).to(dtype)
    bias = torch.randn(2 * half, generator=g, device="cuda").to(dtype)
    got = ops.linear_rows(x, ops.pack_linear(w), bias, swiglu=True).double()
    p = x.double() @ w.double().t()
    v = p + bias.double()
    gate, up = v[:, 0::2], v[:, 1::2]
    want = gate * torch.sigmoid(gate) * up
    # eps (half a unit in the last place of 1) where the product, the biased pair, silu and the result are rounded; sums of K products in fp32 add K 2^-24 of the products' size; |silu'| < 1.1.  A value below 16 bits' normal range (fp16) keeps 2^-24.
    off = eps * (p.abs() + v.abs()) + K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    bound = 1.1 * up.abs() * off[:, 0::2] + gate.abs() * off[:, 1::2] + 2 * eps * want.abs() + 1.1 * off[:, 0::2] * off[:, 1::2] + 2.0 ** -24 + 1e-5 * want.abs()
    assert got.shape == want.shape and bool(((got - want).abs() <= 1.05 * bound).all())
