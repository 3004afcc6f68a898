"""Post-norms that sum a decode product's splits (mi355_norm_residual_add_partials) against the norm of the summed product: the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("rms", [False, True])
@pytest.mark.parametrize("m,n,k", [(1, 2048, 5632), (64, 2048, 11264), (3, 264, 512), (17, 4096, 1024), (5, 8192, 2048), (64, 6144, 768)])
@pytest.mark.parametrize("dtype,last", [(torch.bfloat16, False), (torch.bfloat16, True), (torch.float16, False)])
def test_splits_summed_by_the_norm(rms, m, n, k, dtype, last):
    """One split and many, rows of one to four register groups, with and without a norm behind (last)."""
    from sglang_custom_amd import ops

    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, n, generator=g).to(DEV)
    a = torch.randn(m, k, generator=g).to(dtype).to(DEV)
    wp = ops.pack_weight(torch.randn(n, k, generator=g).mul_(k ** -0.5).to(dtype).to(DEV))
    w_out, w_next = torch.randn(2, n, generator=g).to(dtype).to(DEV)
    w_next = None if last else w_next
    part, y = ops.linear_packed_partials(a, wp, n), ops.linear_packed(a, wp, n)
    x1, x2 = x.clone(), x.clone()
    got = ops.norm_residual_add_partials(x1, part, w_out, w_next, 1e-6, rms)
    want = ops.rmsnorm_residual_add_next(x2, y, w_out, w_next, 1e-6, copy=True) if rms else ops.layernorm_residual_add(x2, y, w_out, w_next, 1e-6)
    assert torch.equal(x1, x2) and not torch.equal(x1, x)
    assert (got is None and want is None) or torch.equal(got, want)
