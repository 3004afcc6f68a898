"""The normed add's vector output pass and its picked rows, four at a time: group widths that are and are not multiples of eight,
row counts about the batch of four, results and weights off the 16-byte grid (the scalar pass)."""
import pytest
import torch
import verozen_cases as cases

from sglang_custom_amd import ops
from oracle import verozen_ref as ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D,groups,n,off", [
    (8, 1, 1, 0),          # one vector
    (2048, 4, 8, 0),       # one pass of the workgroup exactly
    (2056, 1, 5, 0),       # one thread of a second pass; a batch of one row behind a full one
    (2064, 2, 4, 0),       # 1032 a group
    (48, 4, 3, 0),         # twelve a group: the scalar pass
    (2048, 4, 7, 1),       # a weight off the grid: the scalar pass over the same row
])
def test_group_norm_of_picked_rows(dtype, D, groups, n, off):
    g = torch.Generator().manual_seed(D + n)
    T, R, eps = 5, 23, 1e-5
    x = torch.randn(T, D, generator=g)
    big = torch.randn(R, D, generator=g).bfloat16().float()
    w = (1 + 0.1 * torch.randn(D + off, generator=g)).bfloat16().double()[off:]
    rows = torch.randint(0, R, (T, n), generator=g, dtype=torch.int32)
    coef = torch.rand(T, n, generator=g)
    want = ref.group_rms_norm(1.5 * x.double() + (coef.double()[:, :, None] * big.double()[rows.long()]).sum(1), w, groups, eps)
    wd = torch.zeros(D + off, dtype=dtype, device="cuda")[off:].copy_(w)
    xd = x.cuda()
    h = ops.scaled_add_group_rmsnorm(xd, big.to("cuda", dtype), 1.5, wd, groups, eps, rows=rows.cuda(), coef=coef.cuda())
    # fp32 throughout: n + 1 products and sums of at most 8 magnitudes, then the norm -- the bound of the existing cases;
    # bf16 values are held by all three types (fp16: to 2^-25), so the inputs are the same numbers
    cases._close(xd, want, 2e-6 * (1 if n <= 3 else 2), "the fp32 stream")
    cases._close(h, want, cases._tol(dtype), "its copy")
