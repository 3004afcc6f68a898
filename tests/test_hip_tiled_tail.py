"""Tiled projections whose tiles beyond whole rounds share K: small integers, whose sums are exact in any order, so every result must be
the one without splits, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
# rows, columns, K: no whole round (one tile; one live row in the second; sixteen splits), tails of 16 and 128 tiles behind a whole
# round, K tiles that do not divide by the splits, tails of 50 and 41 (33 and 8 of pairs) with ragged last rows and columns
SHAPES = [(65, 240, 2048), (257, 2048, 8192), (4100, 4080, 1088), (2048, 12288, 2624), (300, 4096, 14336), (4103, 4368, 1152), (8200, 2064, 2048)]


@pytest.fixture(scope="module")
def ops():
    from sglang_custom_amd import ops as o
    return o


def ints(g, *shape):
    return torch.randint(-2, 3, shape, generator=g).float().to(DEV)


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("silu", [False, True], ids=["plain", "silu_mul"])
@pytest.mark.parametrize("form", ["bf16", "f16", "fp8"])
def test_split_tiles_equal_whole_ones(ops, m, n, k, silu, form):
    g = torch.Generator().manual_seed(m + k)
    if silu:
        n = n // 32 * 32
    fp8 = form == "fp8"
    if fp8:
        k *= 2      # the same bytes
    assert ops.tiled_tail_splits(m, n, k, fp8, silu) > 1
    x, w, b = ints(g, m, k), ints(g, n, k), ints(g, n)
    if fp8:
        xs, ws = 2.0 ** torch.randint(-3, 2, (m,), generator=g).float().to(DEV), 2.0 ** torch.randint(-3, 2, (n,), generator=g).float().to(DEV)
        bias = None if silu else b.bfloat16()
        call = lambda split: ops.fp8_scaled_mm_tiled(x.to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn), xs, ws, torch.bfloat16, bias, silu_mul=silu,
                                                     split_tail=split)
        ref = ((x @ w.T) * xs[:, None] * ws + (0 if silu else b)).bfloat16()
    else:
        dt = torch.bfloat16 if form == "bf16" else torch.float16
        wide = torch.empty(m, k + 8, dtype=dt, device=DEV)
        wide[:, :k] = x
        bias = None if silu else b.to(dt)
        call = lambda split: ops.linear_tiled(wide[:, :k], w.to(dt), bias, silu_mul=silu, split_tail=split)
        ref = (x @ w.T + (0 if silu else b)).to(dt)
    if silu:
        ref = ops.silu_and_mul(ref.contiguous())
    whole = call(False)
    assert torch.equal(whole, ref)
    for _ in range(2):
        assert torch.equal(call(True), whole)




@pytest.mark.parametrize("m,k,hq,hkv", [(300, 2048, 8, 2), (2820, 1088, 30, 9)])
def test_split_tiles_rotate_and_write_the_cache(ops, m, k, hq, hkv):
    g = torch.Generator().manual_seed(m)
    n = (hq + 2 * hkv) * 128
    assert ops.tiled_tail_splits(m, n, k) > 1
    x, w = ints(g, m, k).bfloat16(), ints(g, n, k).bfloat16()
    pos = torch.randint(0, 500, (m,), generator=g).to(DEV)
    angle = torch.rand(500, 64, generator=g) * 6
    cs = torch.cat([angle.cos(), angle.sin()], 1).to(DEV)
    loc = torch.randperm(m + 9, generator=g)[:m].to(DEV)
    got = []
    for split in (False, True):
        kb, vb = (torch.zeros(m + 9, hkv, 128, dtype=torch.bfloat16, device=DEV) for _ in range(2))
        got.append((ops.qkv_proj_rope_tiled(x, w, hq, hkv, 128, pos, cs, True, kb, vb, loc, split_tail=split), kb, vb))
    for a, b in zip(*got):
        assert torch.equal(a, b)


# more tiles than CUs, so that workgroups take a second one: whole (408 tiles: their rest shares nothing), with K tiles that are two, odd and
# many; and behind whole ones, a rest of 32 tiles that shares K.  Ragged last rows
@pytest.mark.parametrize("m,k,hq,hkv", [(4100, 128, 30, 9), (4100, 320, 30, 9), (4090, 1024, 38, 5), (2820, 1088, 30, 9)])
@pytest.mark.parametrize("form", ["bf16", "f16", "fp8", "fp8 f16"])
@pytest.mark.parametrize("cs_f32", [True, False])
def test_qkv_rope_over_several_tiles_a_workgroup(ops, m, k, hq, hkv, form, cs_f32):
    """The projection as torch has it (exact: whole numbers), then the rotation and cache write of their own kernel."""
    g = torch.Generator().manual_seed(m + k)
    dt, fp8 = torch.float16 if "f16" in form.replace("bf16", "") else torch.bfloat16, "fp8" in form
    if fp8:
        k *= 2
    n = (hq + 2 * hkv) * 128
    assert -(-m // 256) * n // 256 > 256 and (ops.tiled_tail_splits(m, n, k, fp8) > 1) == (m == 2820)
    x, w = ints(g, m, k), ints(g, n, k)
    pos = torch.randint(0, 500, (m,), generator=g).to(DEV)
    angle = torch.rand(500, 64, generator=g) * 6
    cs = torch.cat([angle.cos(), angle.sin()], 1).to(DEV, torch.float32 if cs_f32 else dt)
    loc = torch.randperm(m + 9, generator=g)[:m].to(DEV, torch.int32 if m % 4 else torch.int64)
    xs, ws = (2.0 ** torch.randint(-3, 2, (r,), generator=g).float().to(DEV) if fp8 else torch.ones(r, device=DEV) for r in (m, n))
    ref = ((x @ w.T) * xs[:, None] * ws).to(dt)
    kb, vb, kr, vr = (torch.zeros(m + 9, hkv, 128, dtype=dt, device=DEV) for _ in range(4))
    q, kk, v = ref.split([hq * 128, hkv * 128, hkv * 128], dim=-1)
    ops.rope_inplace(pos, q, kk, 128, cs, True, v=v, k_buffer=kr, v_buffer=vr, loc=loc)
    for split in (False, True):
        if fp8:
            f8 = torch.float8_e4m3fn
            got = ops.qkv_proj_rope_tiled(x.to(f8), w.to(f8), hq, hkv, 128, pos, cs, True, kb, vb, loc, xs, ws, dt, split_tail=split)
        else:
            got = ops.qkv_proj_rope_tiled(x.to(dt), w.to(dt), hq, hkv, 128, pos, cs, True, kb, vb, loc, split_tail=split)
        assert torch.equal(got, ref) and torch.equal(kb, kr) and torch.equal(vb, vr)


def test_a_workspace_that_is_too_small_is_refused(ops):
    lib = ops._lib_()
    m, n, k = 300, 4096, 14336
    need = lib.mi355_tiled_tail_workspace_bytes(m, n, k, 0, 0)
    assert need == ops.tiled_tail_splits(m, n, k) * 32 * 65536 * 4
    x, w = torch.zeros(m, k, dtype=torch.bfloat16, device=DEV), torch.zeros(n, k, dtype=torch.bfloat16, device=DEV)
    y, ws = torch.empty(m, n, dtype=torch.bfloat16, device=DEV), torch.empty(need - 16, dtype=torch.uint8, device=DEV)
    rc = lib.mi355_linear_tiled_ws(y.data_ptr(), x.data_ptr(), w.data_ptr(), None, m, n, k, k, 1, 0, ws.data_ptr(), ws.numel(),
                                   torch.cuda.current_stream().cuda_stream)
    assert rc != 0
