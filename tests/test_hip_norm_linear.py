"""mi355_norm_linear_packed against the two launches that it takes the place of (themselves checked against the oracle)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def ops():
    from sglang_custom_amd import ops as o

    return o


# (rows, K, columns, splits of the partials): one and two groups of a row a lane, up to four and up to eight splits, columns that leave waves
# of the last workgroup idle, K in several splits of the product, one chunk
@pytest.mark.parametrize("m,k,n,splits", [(1, 256, 16, 1), (1, 2048, 3072, 8), (2, 2048, 16384, 4), (1, 4096, 6144, 5), (1, 4096, 28672, 8), (2, 768, 1040, 3),
                                          (2, 1024, 2048, 7)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_one_launch_for_two(ops, m, k, n, splits, dtype):
    g = torch.Generator().manual_seed(m * k + n)
    part = torch.randn(splits, m, k, generator=g).mul_(0.5).to(DEV)
    res, nw = torch.randn(m, k, generator=g).to(dtype).to(DEV), torch.randn(k, generator=g).mul_(0.1).add_(1).to(dtype).to(DEV)
    w = torch.randn(n, k, generator=g).mul_(k ** -0.5).to(dtype).to(DEV)
    for silu in (False, True):
        want_splits = ops.norm_linear_packed_splits(m, n, k, silu)
        if silu and want_splits == 0:
            assert ops.norm_linear_packed_splits(m, n, k) > 1        # the activation needs whole sums
            continue
        wp = ops.pack_weight_gate_up(w) if silu else ops.pack_weight(w)
        old = res.clone()
        x = ops.fused_add_rmsnorm_partials(part, old, nw, 1e-5)      # old: the new residual
        want = ops.linear_packed_silu_mul(x, wp, n) if silu else ops.linear_packed_partials(x, wp, n)
        before = res.clone()
        got, new = ops.norm_linear_packed(part, res, nw, 1e-5, wp, n, silu)
        assert torch.equal(new, old) and torch.equal(res, before) and got.shape == want.shape
        # the squares' sum rounds elsewhere (1e-7), so an element of x may round to its neighbour: one in 2^24 / 2^9 does, by 2^-8 of itself; all of
        # them would be 2^-8 of the result
        assert ((got.float() - want.float()).norm() <= 2.0 ** -10 * want.float().norm())
        if not silu:
            exact = x.double() @ w.double().T
            assert (got.double().sum(0) - exact).norm() <= 2.0 ** -10 * exact.norm()


def test_what_it_refuses(ops):
    assert ops.norm_linear_packed_splits(3, 3072, 2048) == 0 and ops.norm_linear_packed_splits(1, 3072, 2048 + 128) == 0
    assert ops.norm_linear_packed_splits(1, 70000, 2048) == 0 and ops.norm_linear_packed_splits(2, 6144, 8192) == 0
    part, res = torch.zeros(9, 1, 256, device=DEV), torch.zeros(1, 256, dtype=torch.bfloat16, device=DEV)
    w = ops.pack_weight(torch.zeros(64, 256, dtype=torch.bfloat16, device=DEV))
    with pytest.raises(AssertionError):
        ops.norm_linear_packed(part, res, res[0], 1e-5, w, 64)
    lib, out = ops._lib_(), torch.zeros(1, 1, 64, device=DEV)
    rc = lib.mi355_norm_linear_packed(None, out.data_ptr(), res.data_ptr(), part.data_ptr(), 1, res.data_ptr(), res.data_ptr(), 1e-5, w.data_ptr(), 1, 64, 256,
                                      ops._dt(res), ops._stream(res))
    assert rc != 0          # the residual in place
