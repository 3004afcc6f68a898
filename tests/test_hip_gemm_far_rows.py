"""Tiled products whose rows lie 2^23 elements and more apart, further than a buffer's 31-bit offsets reach: the bits of the same rows close
together, one row (whose stride torch does not take for one) and many; and K of that length against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
STRIDES = [(1 << 23) - 8, 1 << 23, (1 << 24) + 24]       # the last that a buffer serves, the first that it does not, one beyond


@pytest.fixture(scope="module")
def ops():
    from sglang_custom_amd import ops as o
    return o


def far(x, stride):
    m, k = x.shape
    buf = torch.empty((m - 1) * stride + k, dtype=x.dtype, device=DEV)
    rows = buf.as_strided((m, k), (stride, 1))
    rows.copy_(x)
    assert rows.stride(0) == stride
    return rows


# one row; a ragged half tile and two tiles of rows, with K tiles that are an odd number, two, and shared by splits; more tiles than CUs
@pytest.mark.parametrize("m,n,k", [(1, 528, 192), (130, 272, 128), (300, 2048, 2048), (300, 33024, 256)])
@pytest.mark.parametrize("stride", STRIDES)
def test_linear_tiled(ops, m, n, k, stride):
    g = torch.Generator(device=DEV).manual_seed(m + n)
    x, w, b = (torch.randn(*s, device=DEV, generator=g).bfloat16() for s in ((m, k), (n, k), (n,)))
    rows = far(x, stride)
    for kw in ({"bias": b}, {"silu_mul": True}, {"act": "gelu_erf"}, {"act": "gelu_tanh_mul"}):
        for split in (False, True):
            assert torch.equal(ops.linear_tiled(rows, w, split_tail=split, **kw), ops.linear_tiled(x, w, split_tail=split, **kw)), (kw, split)


@pytest.mark.parametrize("m", [1, 300])
@pytest.mark.parametrize("stride", STRIDES)
def test_qkv_proj_rope_tiled(ops, m, stride):
    hq, hkv, k = 6, 2, 320
    g = torch.Generator(device=DEV).manual_seed(m)
    x, w = torch.randn(m, k, device=DEV, generator=g).bfloat16(), torch.randn((hq + 2 * hkv) * 128, k, device=DEV, generator=g).bfloat16()
    cs = torch.randn(400, 128, device=DEV, generator=g)
    pos, loc = torch.arange(m, device=DEV), torch.randperm(m + 5, device=DEV, generator=g)[:m]
    got = []
    for rows in (x, far(x, stride)):
        kb, vb = (torch.zeros(m + 5, hkv, 128, dtype=torch.bfloat16, device=DEV) for _ in range(2))
        got.append((ops.qkv_proj_rope_tiled(rows, w, hq, hkv, 128, pos, cs, True, kb, vb, loc), kb, vb))
    for a, b in zip(*got):
        assert torch.equal(a, b)


@pytest.mark.parametrize("form", ["bf16", "fp8"])
def test_long_rows(ops, form):
    """K past 2^23: x and W of that many columns.  Small whole numbers: every fp32 sum is exact (below 2^24), so the result is its rounding."""
    m, n, k = 17, 32, (1 << 23) + 128
    g = torch.Generator(device=DEV).manual_seed(5)
    x, w = (torch.randint(-1, 2, (r, k), device=DEV, generator=g, dtype=torch.int8) for r in (m, n))
    ref = torch.stack([(x.short() * r).sum(1, dtype=torch.int64) for r in w], 1)
    if form == "fp8":
        one = torch.ones(max(m, n), device=DEV)
        x8, w8 = x.float().to(torch.float8_e4m3fn), w.float().to(torch.float8_e4m3fn)
        assert ops.linear_few_supported(m, n, k, torch.bfloat16, fp8=True)
        got = [ops.fp8_scaled_mm_tiled(x8, w8, one[:m], one[:n], torch.bfloat16),
               ops.linear_few(x8, w8, x_scale=one[:m].clone(), w_scale=one[:n].clone(), out_dtype=torch.bfloat16)]
    else:
        xb, wb = x.bfloat16(), w.bfloat16()
        assert ops.linear_tiled_supported(m, n, k, torch.bfloat16) and ops.linear_few_supported(m, n, k, torch.bfloat16)
        got = [ops.linear_tiled(xb, wb), ops.linear_tiled(xb, wb, split_tail=True), ops.linear_few(xb, wb)]
    for y in got:
        assert torch.equal(y, ref.bfloat16())
