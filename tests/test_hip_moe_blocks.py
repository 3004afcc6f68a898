"""GPU: the mixture's block sizes and plans at their edges -- 256-row blocks that do no work for padding rows, the sorted plan past
its register-kept pairs, narrow fp32 products -- against plain float64 / integer restatements."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def ops():
    from sglang_custom_amd import ops as o

    return o


@pytest.mark.parametrize("T,E,top,block", [(1, 5, 1, 64), (3, 2, 2, 256), (64, 32, 4, 256), (300, 200, 2, 128), (5000, 32, 4, 256),
                                           (16384, 3, 1, 64), (16385, 7, 1, 256), (9000, 1500, 3, 64)])
def test_align_sorts_every_pair_once(ops, T, E, top, block):
    g = torch.Generator().manual_seed(T + E)
    ids = torch.rand(T, E, generator=g).topk(top, -1).indices.int() if E * T < 10 ** 7 else torch.randint(0, E, (T, top), generator=g).int()
    if E > 4:
        ids[ids == 1] = 0                      # one expert without rows
    lib = ops._lib_()
    padded = (T * top + min(E, T * top) * (block - 1) + block - 1) // block * block
    src, rows = torch.empty(padded, dtype=torch.int32, device=DEV), torch.empty((T, top), dtype=torch.int32, device=DEV)
    te, nt = torch.full((padded // block,), -7, dtype=torch.int32, device=DEV), torch.empty(1, dtype=torch.int32, device=DEV)
    d = ids.to(DEV).contiguous()
    ops.check(lib.mi355_moe_align(src.data_ptr(), rows.data_ptr(), te.data_ptr(), nt.data_ptr(), d.data_ptr(), T, top, E, block, padded,
                                  ops._stream(d)), "moe_align")
    src, rows, te, nt = src.cpu(), rows.cpu().long(), te.cpu(), int(nt.item())
    counts = torch.bincount(ids.flatten().long(), minlength=E)
    assert nt == int(((counts + block - 1) // block).sum())
    assert rows.flatten().unique().numel() == T * top and int(rows.max()) < nt * block
    assert torch.equal(src[rows], torch.arange(T, dtype=torch.int32)[:, None].expand(T, top))
    assert torch.equal(te[rows // block], ids)
    live = (src[: nt * block] >= 0).view(nt, block)
    assert int(live.sum()) == T * top and not (~live[:, :-1] & live[:, 1:]).any()        # a block's rows lie in front of its padding
    assert (src[nt * block:] == -1).all()


@pytest.mark.parametrize("sizes", [(0, 1, 8), (15, 16, 17), (127, 128, 129), (255, 256, 257), (500, 3, 300), (512, 241, 120)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_blocks_of_256_rows_skip_padding(ops, sizes, dtype):
    """An expert's last block at every edge of the 8-, 16- and 128-row pieces; both GEMMs.  One rounding of the float64 product
    (2^-8 / 2^-11 relative) plus the fp32 sums' 1e-5 of the row's scale."""
    g = torch.Generator().manual_seed(sum(sizes))
    E, K, N = 3, 192, 320
    T = sum(sizes)
    ids = torch.cat([torch.full((n,), e, dtype=torch.int32) for e, n in enumerate(sizes)])[torch.randperm(T, generator=g)][:, None].contiguous()
    x = torch.randn(T, K, generator=g).to(dtype)
    up, down = (torch.randn(E, N, K, generator=g) * K ** -0.5).to(dtype), (torch.randn(E, K, N, generator=g) * N ** -0.5).to(dtype)
    plan = ops.moe_align(ids.to(DEV), E, tiled_ok=True)
    assert plan.block == 256
    a = ops.moe_grouped_linear(x.to(DEV), up.to(DEV), plan, gather=True, gelu=False, relu2=True)
    rows = plan.rows.long().cpu()[:, 0]
    e = ids[:, 0].long()
    want = torch.einsum("tk,tnk->tn", x.double(), up.double()[e]).clamp_min(0) ** 2
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    assert ((a.cpu()[rows].double() - want).abs() <= ulp * want.abs() + 1e-5 * 16).all()
    b = ops.moe_grouped_linear(a, down.to(DEV), plan, gather=False, gelu=False).cpu()[rows]
    want = torch.einsum("tn,tkn->tk", a.cpu()[rows].double(), down.double()[e])
    assert ((b.double() - want).abs() <= ulp * want.abs() + 1e-5 * 16).all()


@pytest.mark.parametrize("T,N,K,off", [(65, 1, 8, 0), (100, 16, 2048, 0), (257, 33, 200, 0), (300, 512, 264, 8), (1000, 5, 4, 0), (70, 513, 64, 0), (90, 40, 37, 0),
                                       (2100, 100, 64, 0), (4100, 24, 64, 0), (4100, 64, 64, 0), (8200, 320, 64, 0), (8200, 321, 64, 0)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_narrow_products_in_fp32(ops, T, N, K, off, dtype):
    """fp32 results of mi355_linear on both sides of the narrow kernel's conditions.  Each of K terms and partial sums rounds once in
    fp32: 2 sqrt(K) 2^-24 times the root of the summed squares bounds what is seen; 4 x that is allowed, and for bf16 operands the one
    rounding of the sum to bf16 (half an ulp: 2^-9 relative, 2^-8 where the sum's own error moves it over a rounding boundary)."""
    g = torch.Generator().manual_seed(T * N + K)
    x, w = torch.randn(T, K + off, generator=g).to(dtype), torch.randn(N, K, generator=g).to(dtype)
    got = ops.linear(x.to(DEV)[:, off:], w.to(DEV), out_dtype=torch.float32).cpu().double()
    xd, wd = x[:, off:].double(), w.double()
    want = xd @ wd.T
    ulp = 0.0 if dtype == torch.float32 else 2.0 ** -8
    assert ((got - want).abs() <= ulp * want.abs() + 8 * K ** 0.5 * 2.0 ** -24 * ((xd ** 2) @ (wd ** 2).T).sqrt() + 1e-12).all()
    if dtype != torch.float32:
        assert torch.equal(got, got.bfloat16().double())


@pytest.mark.parametrize("d", [8, 192, 20, 7])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_gated_unit_of_listed_rows(ops, d, dtype):
    """The listed rows get the bits that the launch over every row gives them, whatever the others hold; the rest stays unwritten."""
    g = torch.Generator().manual_seed(d)
    x = torch.randn(70, 2 * d, generator=g).to(dtype).to(DEV)
    rows = torch.randperm(70, generator=g)[:24].reshape(8, 3).int()
    others = torch.ones(70, dtype=torch.bool)
    others[rows.flatten().long()] = False
    want, listed = ops.silu_and_mul(x), rows.to(DEV)
    x[others] = float("nan")
    out = torch.full((70, d), 3.0, dtype=dtype, device=DEV)
    ops.check(ops._lib_().mi355_silu_and_mul_rows(out.data_ptr(), x.data_ptr(), listed.data_ptr(), 24, d, ops._dt(x), ops._stream(x)), "rows")
    got = ops.silu_and_mul_rows(x, listed)
    torch.cuda.synchronize()
    assert torch.equal(out[~others], want[~others]) and (out[others] == 3.0).all() and torch.equal(got[~others], want[~others])


@pytest.mark.parametrize("holes", [(0, 5), (0, 200, 255), (100, 101, 254), tuple(range(0, 256, 2)), tuple(range(1, 256))])
def test_padding_anywhere_in_a_tile(ops, holes):
    """A caller's own row map may leave rows out in front of others (a plan of this library never does): the others are all there.
    Small integers, so sums are exact."""
    g = torch.Generator().manual_seed(len(holes))
    K, N = 128, 272
    x = torch.randint(-2, 3, (50, K), generator=g).to(torch.bfloat16).to(DEV)
    w = torch.randint(-2, 3, (2, N, K), generator=g).to(torch.bfloat16).to(DEV)
    rows = torch.randint(0, 50, (512,), generator=g).int()
    rows[list(holes)] = -1
    rows[256:400] = -1
    te, used, rd = torch.tensor([1, 0], dtype=torch.int32, device=DEV), torch.tensor([2], dtype=torch.int32, device=DEV), rows.to(DEV)
    y = torch.full((512, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.check(ops._lib_().mi355_moe_grouped_linear_tiled(y.data_ptr(), x.data_ptr(), K, w.data_ptr(), rd.data_ptr(), te.data_ptr(), used.data_ptr(),
                                                         0, 512, N, K, ops._dt(x), ops._stream(x)), "tiled")
    torch.cuda.synchronize()
    for tile, e in ((0, 1), (1, 0)):
        r = rows[256 * tile: 256 * tile + 256]
        keep = r >= 0
        want = (x.float()[r[keep].long().to(DEV)] @ w[e].float().T).to(torch.bfloat16)
        assert torch.equal(y[256 * tile: 256 * tile + 256][keep.to(DEV)], want)


@pytest.mark.parametrize("K", [128, 192, 448])
def test_every_expert_walks_all_of_k(ops, K):
    """Experts start K at different tiles of 64 and go round its end: two, three and seven of them for nine experts (more than there
    are tiles to start from).  Small integers, so sums are exact; a tile skipped or taken twice shows."""
    g = torch.Generator().manual_seed(K)
    E, N, x = 9, 272, torch.randint(-2, 3, (40, K), generator=g).to(torch.bfloat16).to(DEV)
    w = torch.randint(-2, 3, (E, N, K), generator=g).to(torch.bfloat16).to(DEV)
    rows = torch.randint(0, 40, (E * 256,), generator=g).int().to(DEV)
    te, used = torch.arange(E, dtype=torch.int32, device=DEV), torch.tensor([E], dtype=torch.int32, device=DEV)
    y = torch.full((E * 256, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.check(ops._lib_().mi355_moe_grouped_linear_tiled(y.data_ptr(), x.data_ptr(), K, w.data_ptr(), rows.data_ptr(), te.data_ptr(),
                                                         used.data_ptr(), 0, E * 256, N, K, ops._dt(x), ops._stream(x)), "tiled")
    torch.cuda.synchronize()
    for e in range(E):
        part = slice(256 * e, 256 * e + 256)
        assert torch.equal(y[part], (x.float()[rows[part].long()] @ w[e].float().T).to(torch.bfloat16)), e


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gelu_of_the_tiles(ops, dtype):
    """The activation in the epilogue through products that copy their input: -20 .. 20 against float64, within half an ulp of the result's
    type, 2^-20 for the polynomial and z^2 2^-24 for the exponent's two roundings (exp(-z^2 / 2) at -12: 4e-6), and 2^-121 where the
    exponential is no normal number; infinity stays, minus infinity and NaN give NaN as z * (1 + erf) does."""
    x = torch.zeros(256, 128, dtype=dtype)
    x[:, :63] = torch.linspace(-20, 20, 256 * 63).view(256, 63).to(dtype)
    big = 3e38 if dtype == torch.bfloat16 else 6e4
    x[:3, 63] = torch.tensor([big, -big, float("nan")])
    w = torch.zeros(1, 64, 128, dtype=dtype)
    w[0, :, :64] = torch.eye(64)
    w[0, 63, 63] = 4.0 if dtype == torch.bfloat16 else 6e4
    w[0, 63, 64:] = 0.0
    x[0, 64:] = 0.0
    rows, te, used = torch.arange(256, dtype=torch.int32, device=DEV), torch.zeros(1, dtype=torch.int32, device=DEV), torch.ones(1, dtype=torch.int32, device=DEV)
    y, xd, wd = torch.empty(256, 64, dtype=dtype, device=DEV), x.to(DEV), w.to(DEV)
    ops.check(ops._lib_().mi355_moe_grouped_linear_tiled(y.data_ptr(), xd.data_ptr(), 128, wd.data_ptr(), rows.data_ptr(), te.data_ptr(), used.data_ptr(),
                                                         1, 256, 64, 128, ops._dt(xd), ops._stream(xd)), "tiled")
    torch.cuda.synchronize()
    z = x[3:, :63].double()
    want = 0.5 * z * torch.erfc(-z / 2 ** 0.5)
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    least = 2.0 ** -121 if dtype == torch.bfloat16 else 2.0 ** -25      # (half the spacing of fp16's smallest numbers)
    assert ((y[3:, :63].cpu().double() - want).abs() <= (ulp + 2.0 ** -20 + z ** 2 * 2.0 ** -24) * want.abs() + least).all()
    if dtype == torch.bfloat16:
        assert y[0, 63] == float("inf") and y[1, 63].isnan()
    else:
        assert y[0, 63] == float("inf")     # (3.6e9 rounds to infinity; its negative to zero)
    assert y[2].isnan().any()
