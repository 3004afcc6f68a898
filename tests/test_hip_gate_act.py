"""The gated units in the epilogue of the packed gate / up product (mi355_linear_packed_act_mul) against the product and the unit's own launch."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("act", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("m,n,k", [(1, 16, 256), (3, 1040, 512), (16, 11264, 2048), (17, 2064, 768), (64, 11264, 2048), (40, 4096, 8192)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_unit_in_the_epilogue(act, m, n, k, dtype):
    """Whole and split products, rows and columns that end inside a tile.  Packing orders the weight's rows, not a sum's terms, but the two products
    may split K differently: equal but for a rounding of gate or up to its neighbour (2^-8 of either, 1.1 is the units' steepest slope)."""
    from sglang_custom_amd import ops

    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g).to(dtype).to(DEV)
    w = torch.randn(n, k, generator=g).mul_(k ** -0.5).to(dtype).to(DEV)
    got = ops.linear_packed_silu_mul(x, ops.pack_weight_gate_up(w), n, act=act)
    gu = ops.linear_packed(x, ops.pack_weight(w), n)
    gate, up = gu[:, : n // 2], gu[:, n // 2:]
    want = ops.silu_and_mul(gu) if act == "silu" else ops.gelu_tanh_and_mul(gate, up)
    eps = 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10
    assert ((got.float() - want.float()).abs() <= eps * (1.1 * gate.float().abs() * up.float().abs() + want.float().abs() + 0.01)).all()
    assert (got != want).float().mean() < 0.02
