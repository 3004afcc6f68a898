"""The GELUs in the epilogue of the tiled projection (mi355_linear_tiled, epilogues 2 and 3) against float64 of the product that the same kernel
gives without them."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("act", ["gelu_erf", "gelu_tanh_mul"])
@pytest.mark.parametrize("m,n,k", [(1, 16, 128), (257, 272, 192), (300, 4096, 2048), (4500, 4112, 256), (8200, 8192, 2048)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_unit_of_the_rounded_product(act, m, n, k, dtype):
    """Rows and columns that end inside a tile, and tiles beyond whole rounds of the chip with and without a split K.  The unit acts on the
    product's rounded values, the same ones: one rounding (2^-8, fp16 2^-11, of the result; its smallest numbers are 2^-24 apart) and
    the unit's fp32 error (1e-6 of z where the result is not its tail, times the up column)."""
    from sglang_custom_amd import ops

    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g).to(dtype).to(DEV)
    w = torch.randn(n, k, generator=g).mul_(3 * k ** -0.5).to(dtype).to(DEV)
    split = act == "gelu_erf"       # (gate / up tiles are cut elsewhere than the plain product's)
    z, up = ops.linear_tiled(x, w, None, split_tail=split).double(), 1.0
    if act == "gelu_erf":
        want = 0.5 * z * torch.special.erfc(-z * 0.5 ** 0.5)
    else:
        z, up = z[:, : n // 2], z[:, n // 2:]
        want = z * torch.sigmoid(2 * math.sqrt(2 / math.pi) * (z + 0.044715 * z ** 3)) * up
        up = up.abs()
    got = ops.linear_tiled(x, w, None, split_tail=split, act=act)
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    assert ((got.double() - want).abs() <= 1.01 * unit * want.abs() + 1e-6 * z.abs().clamp(max=1) * up * (z.abs() < 6) + 2.0 ** -24).all()
    if not split:      # gate or up rounded to its neighbour; the unit's steepest slope is 1.13
        cut = ops.linear_tiled(x, w, None, split_tail=True, act=act).double()
        assert ((cut - want).abs() <= 2 * unit * (1.13 * z.abs() * up + 2 * want.abs() + 0.01)).all() and (cut != got.double()).float().mean() < 0.02


def test_refused_with_a_bias_or_another_unit():
    from sglang_custom_amd import ops

    x, w = (torch.zeros(s, dtype=torch.bfloat16, device=DEV) for s in ((256, 128), (32, 128)))
    for act in ("gelu_erf", "gelu_tanh_mul"):
        with pytest.raises(RuntimeError):
            ops.linear_tiled(x, w, torch.zeros(32, dtype=torch.bfloat16, device=DEV), act=act)
        with pytest.raises(AssertionError):
            ops.linear_tiled(x, w, None, silu_mul=True, act=act)
