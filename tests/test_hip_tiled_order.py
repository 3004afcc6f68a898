"""The tiled GEMM's workgroup -> tile order: every tile once, whatever the bands, columns and equal runs per XCD come out as."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


# tile counts: one; fewer than XCDs; a short last band beside narrow last blocks; runs that do not divide; one row band of one
# row; many rows of one column
@pytest.mark.parametrize("mt,nt", [(1, 1), (1, 7), (9, 5), (18, 6), (17, 1), (3, 13), (8, 4), (10, 9)])
@pytest.mark.parametrize("silu", [False, True])
def test_every_tile_is_written_once(mt, nt, silu):
    """y must equal x w^T (K = 128) in every tile; a row short of a whole tile, sixteen columns short of one.  The operands are
    small integers, so the sums are exact and the results their roundings to bf16."""
    from sglang_custom_amd import ops

    g = torch.Generator().manual_seed(mt * 100 + nt)
    cols = nt * (128 if silu else 256) - 16
    M, N, K = mt * 256 - 1, cols * (2 if silu else 1), 128
    x = torch.randint(-2, 3, (M, K), generator=g).to(torch.bfloat16).to(DEV)
    w = torch.randint(-2, 3, (N, K), generator=g).to(torch.bfloat16).to(DEV)
    want = (x.float() @ w.float().T).to(torch.bfloat16)
    if silu:
        want = ops.silu_and_mul(want.contiguous())
    for _ in range(2):
        got = ops.linear_tiled(x, w, None, silu_mul=silu)
        torch.cuda.synchronize()
        assert torch.equal(got, want)
