"""Packed fp32 products with a factor (mi355_linear_packed_scaled, an output head's logits): the unscaled product's values times the factor, to the bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("m,n,k", [(1, 1000, 256), (3, 40, 4096), (17, 32768, 2048), (64, 32000, 2048), (64, 1007, 512), (5, 515, 288)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_scaled_product(m, n, k, dtype):
    """Whole and split sums, ragged columns, and K that the ring does not take (288)."""
    from sglang_custom_amd import ops

    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g).to(dtype).to(DEV)
    w = torch.randn(n, k, generator=g).to(dtype).to(DEV)
    wp = ops.pack_weight(w)
    for scale in (0.3, -2.0):
        got = ops.linear_packed(x, wp, n, out_dtype=torch.float32, scale=scale)
        assert torch.equal(got, ops.linear_packed(x, wp, n, out_dtype=torch.float32) * scale)
    want = (x.double() @ w.double().T) * scale
    # the product's rounding to dtype (half an ulp of at most 2^-8 or 2^-11 relative) and k fp32 sums
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    assert ((got.double() - want).abs() <= 1.01 * eps * want.abs() + abs(scale) * k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)).all()
