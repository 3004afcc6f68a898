"""Few 16-bit rows quantised inside the fp8 product behind them (mi355_fp8_quant_packed_partials) against the two launches: the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("m,n,k", [(1, 4096, 4096), (2, 72, 512), (5, 2048, 2048), (7, 1280, 1536), (8, 4096, 4096), (6, 516, 3584), (8, 6144, 1024)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rows_quantised_in_the_product(m, n, k, dtype):
    """Rows of one wave and of two, one split and many, strided rows, a row of zeros, of a large value and of an infinity."""
    from sglang_custom_amd import ops

    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k + 8, generator=g).to(dtype).to(DEV)[:, :k]
    x[m // 2] = 0.0 if m > 2 else 1.0
    x[0, k - 1] = 3e4
    if m > 5:
        x[4, 3] = float("inf")
    wq, _ = ops.per_token_quant_fp8(torch.randn(n, k, generator=g).to(dtype).to(DEV))
    wp = ops.pack_weight_fp8(wq)
    part, scales = ops.fp8_quant_packed_partials(x, wp, n)
    xq, xs = ops.per_token_quant_fp8(x.contiguous())
    want = ops.fp8_packed_partials(xq, wp, n)
    assert torch.equal(scales.view(-1), xs.view(-1)) and part.shape == want.shape
    assert torch.equal(part.view(torch.int32), want.view(torch.int32)) or torch.equal(part.nan_to_num(123.0), want.nan_to_num(123.0))


def test_what_is_not_served():
    from sglang_custom_amd import ops

    for m, n, k in ((9, 4096, 4096), (8, 4096, 4608), (8, 4096, 3840), (8, 4098, 4096)):
        x = torch.zeros(m, k, dtype=torch.bfloat16, device=DEV)
        assert ops.fp8_quant_packed_partials(x, torch.zeros(((n + 63) // 64) * 64 * k, dtype=torch.uint8, device=DEV), n) is None
