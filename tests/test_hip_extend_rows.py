"""Prefill attention on the 32-row matrix-core tiles at the edges of its key tiles (64 keys, whose cache slots are read a tile ahead),
of its query tiles (128 rows of 32 a wave) and of a paged prefix, against float64 on the CPU."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def ops():
    from sglang_custom_amd import ops as o
    return o


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("kv8", [False, True], ids=["cache16", "cache_fp8"])
@pytest.mark.parametrize("hq,hkv,d", [(6, 2, 128), (6, 2, 64), (4, 4, 64)])
@pytest.mark.parametrize("causal", [True, False])
def test_tile_edges_over_a_paged_prefix(ops, dtype, kv8, hq, hkv, d, causal):
    g = torch.Generator().manual_seed(hq * 100 + d)
    prefix = [0, 1, 63, 64, 65, 127, 128, 129, 200, 0]
    ext = [1, 129, 64, 1, 127, 33, 128, 31, 65, 300]
    T, P = sum(ext), sum(prefix)
    q, k, v = (torch.randn(T, h, d, generator=g).to(dtype) for h in (hq, hkv, hkv))
    qkv = torch.cat([x.reshape(T, -1) for x in (q, k, v)], 1).to(DEV)      # rows a stride apart, as a fused projection leaves them
    qg, kg, vg = (x.view(T, h, d) for x, h in zip(qkv.split([hq * d, hkv * d, hkv * d], 1), (hq, hkv, hkv)))
    kb, vb = (torch.randn(P + 5, hkv, d, generator=g).to(dtype) for _ in range(2))
    if kv8:
        kb, vb = kb.to(torch.float8_e4m3fn), vb.to(torch.float8_e4m3fn)
    slots = torch.randperm(P + 5, generator=g)[:P]
    ind = [torch.tensor([0] + x).cumsum(0).to(torch.int32).to(DEV) for x in (ext, prefix)]
    o = torch.full((T, hq, d), float("nan"), device=DEV, dtype=dtype)
    ops.extend_attention_fwd(qg, kg, vg, o, kb.to(DEV), vb.to(DEV), ind[0], ind[1], slots.to(torch.int32).to(DEV), None, causal, None, max(ext), d ** -0.5)
    o = o.cpu().double()
    # half a unit in the last place of the output, and of a weight where 16-bit weights meet the values: one rounding at head
    # dimension 128 (at 64 none; u^2 of their size stays allowed); 1e-5 for fp32 sums and exponentials
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    at = had = 0
    for n, pre in zip(ext, prefix):
        rows = slots[had:had + pre]
        K = torch.cat([kb[rows].double() if not kv8 else kb.float()[rows].double(), k[at:at + n].double()])
        V = torch.cat([vb[rows].double() if not kv8 else vb.float()[rows].double(), v[at:at + n].double()])
        K, V = (x.repeat_interleave(hq // hkv, 1) for x in (K, V))
        s = torch.einsum("qhd,khd->hqk", q[at:at + n].double(), K) * d ** -0.5
        if causal:
            s.masked_fill_(torch.arange(pre + n) > pre + torch.arange(n)[:, None], -float("inf"))
        p = s.softmax(-1)
        ref, size = (torch.einsum("hqk,khd->qhd", p, x) for x in (V, V.abs()))
        tol = u * ref.abs() + ((u if d == 128 else u * u) + 1e-5) * size
        assert bool(((o[at:at + n] - ref).abs() <= tol).all()), (n, pre)
        at, had = at + n, had + pre


@pytest.mark.gpu
@pytest.mark.parametrize("skip_prefix", [False, True])
@pytest.mark.parametrize("pre,ext", [([0, 70], [65, 3]), ([130, 63], [129, 64])])
def test_custom_mask_at_head_dimension_64(ops, pre, ext, skip_prefix):
    """A mask of its own per query -- holes, a row that sees its own key alone, keys behind the query -- over a prefix and new tokens around
    tile edges, against float32 softmax; bound: the output's rounding to bf16 (2^-8 of values up to 3) and a tenth of that for fp32 sums."""
    torch.manual_seed(sum(pre) + sum(ext))
    hq, hkv, d = 8, 2, 64
    seq = [a + b for a, b in zip(pre, ext)]
    slots = torch.randperm(sum(seq) + 5)[: sum(seq)].int()
    kc, vc = torch.randn(sum(seq) + 5, hkv, d).bfloat16(), torch.randn(sum(seq) + 5, hkv, d).bfloat16()
    T = sum(ext)
    q, k, v = torch.randn(T, hq, d).bfloat16(), torch.randn(T, hkv, d).bfloat16(), torch.randn(T, hkv, d).bfloat16()
    masks, indptr, want, at, was = [], [0], [], 0, 0
    for a, b in zip(pre, ext):
        m = torch.rand(b, a + b) < 0.5
        m[torch.arange(b), a + torch.arange(b)] = True
        m[0] = False
        m[0, a] = True
        masks.append(m.flatten())
        indptr.append(indptr[-1] + m.numel())
        seen = m.clone()
        if skip_prefix:
            seen[:, :a] = True
        kk = torch.cat([kc[slots[was: was + a].long()], k[at: at + b]]).float().repeat_interleave(hq // hkv, 1)
        vv = torch.cat([vc[slots[was: was + a].long()], v[at: at + b]]).float().repeat_interleave(hq // hkv, 1)
        s = torch.matmul(q[at: at + b].float().transpose(0, 1), kk.permute(1, 2, 0)) * d ** -0.5
        p = torch.softmax(s.masked_fill(~seen, float("-inf")), -1)
        want.append(torch.matmul(p, vv.transpose(0, 1)).transpose(0, 1))
        at, was = at + b, was + a
    dev = lambda t: t.to("cuda")
    o = torch.empty(T, hq, d, dtype=torch.bfloat16, device="cuda")
    qo = torch.tensor([0] + ext, dtype=torch.int32).cumsum(0).int()
    kvp = torch.tensor([0] + pre, dtype=torch.int32).cumsum(0).int()
    ops.extend_attention_fwd(dev(q), dev(k), dev(v), o, dev(kc), dev(vc), dev(qo), dev(kvp), dev(slots), dev(torch.cat(masks)), True,
                             dev(torch.tensor(indptr)), max(ext), d ** -0.5, skip_prefix_custom_mask=skip_prefix)
    want = torch.cat(want)
    assert (o.cpu().float() - want).abs().max() <= 3 * 2 ** -8 * 1.1


def _extend(ops, q, k, v, kb, vb, slots, prefix, ext, causal=True, mask=None, scale=1.0):
    """One call; mask: bytes per request [ext, prefix + ext], in a list."""
    dev = lambda x: None if x is None else x.to(DEV)
    qo, kv = ([0] + list(torch.tensor(x).cumsum(0)) for x in (ext, prefix))
    mi = None if mask is None else torch.tensor([0] + [m.numel() for m in mask]).cumsum(0)
    o = torch.full(q.shape, float("nan"), device=DEV, dtype=q.dtype)
    ops.extend_attention_fwd(dev(q), dev(k), dev(v), o, dev(kb), dev(vb), dev(torch.tensor(qo, dtype=torch.int32)), dev(torch.tensor(kv, dtype=torch.int32)),
                             dev(slots.to(torch.int32)), dev(torch.cat([m.flatten() for m in mask]).to(torch.uint8)) if mask else None, causal, dev(mi),
                             max(ext), scale, skip_prefix_custom_mask=False)
    return o


@pytest.mark.parametrize("form", ["causal", "all", "mask", "cache_fp8"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
def test_values_that_are_no_numbers(ops, dtype, form):
    """Head dimension 64: infinities and NaN in value rows reach the queries that see their keys, in their own feature, and no other
    number changes by more than fp32 sums in another order do."""
    g = torch.Generator().manual_seed(5)
    D, hq, hkv, prefix, ext = 64, 4, 2, [70, 0, 3], [130, 140, 40]
    T, P = sum(ext), sum(prefix)
    q, k, v = (torch.randn(T, h, D, generator=g).to(dtype) for h in (hq, hkv, hkv))
    kb, vb = (torch.randn(P + 1, hkv, D, generator=g).to(dtype) for _ in range(2))
    if form == "cache_fp8":
        kb, vb = kb.to(torch.float8_e4m3fn), vb.to(torch.float8_e4m3fn)
    slots = torch.randperm(P, generator=g) + 1
    seen, mask = [], None
    for n, pre in zip(ext, prefix):
        m = torch.arange(pre + n) <= pre + torch.arange(n)[:, None] if form != "all" else torch.ones(n, pre + n, dtype=torch.bool)
        if form == "mask":
            m = m & ((torch.rand(n, pre + n, generator=g) < 0.6) | (torch.arange(pre + n) == pre + torch.arange(n)[:, None]))
        seen.append(m)
    if form == "mask":
        mask = seen
    call = lambda v_, vb_: _extend(ops, q, k, v_, kb, vb_, slots, prefix, ext, form != "all", mask, D ** -0.5)
    plain = call(v, vb).cpu()
    v2, vb2, expect = v.clone(), vb.clone(), plain.double()
    # (request, key, feature, value); feature 9 of request 0 gets both infinities
    for b, key, f, x in ((0, 0, 3, "inf"), (0, 69, 9, "nan" if form == "cache_fp8" else "-inf"), (0, 75, 9, "inf"), (0, 199, 63, "nan"), (0, 131, 40, "-inf"),
                         (1, 0, 0, "inf"), (1, 64, 31, "nan"), (1, 130, 32, "inf"), (2, 2, 5, "nan"), (2, 42, 7, "-inf")):
        pre, at, had = prefix[b], sum(ext[:b]), sum(prefix[:b])
        if form == "cache_fp8" and key < pre:
            x = "nan"      # (e4m3fn has no infinities)
        if key < pre:
            if form == "cache_fp8":
                vb2.view(torch.uint8)[slots[had + key], :, f] = 0x7F
            else:
                vb2[slots[had + key], :, f] = float(x)
        else:
            v2[at + key - pre, :, f] = float(x)
        rows = expect[at:at + ext[b]]
        rows[seen[b][:, key], :, f] += float(x)
    for _ in range(2):
        got = call(v2, vb2).cpu().double()
        assert torch.equal(got.isnan(), expect.isnan())
        assert torch.equal(got.isinf(), expect.isinf()) and (got[got.isinf()] == expect[got.isinf()]).all()
        ok = expect.isfinite()
        assert (got[ok] - expect[ok]).abs().max() <= 2.0 ** (-7 if dtype == torch.bfloat16 else -10)     # a bit of values up to 4
    assert torch.equal(call(v, vb).cpu(), plain)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
def test_weights_of_fp32(ops, dtype):
    """Head dimension 64 multiplies values by fp32 weights.  The terms of every sum are alike in size (values grow as weights fall) and cancel, so
    that the result is the sum's error: 0.5 to 0.8 times 2^-20 of the terms' root sum of squares in fp32, 5 with weights of 16 bits in
    bf16 and 7.5 with two fp16 terms (each in torch on the CPU, the same values)."""
    g = torch.Generator().manual_seed(3)
    D, prefix, ext = 64, [200, 70, 0], [1, 9, 160]
    P, T = sum(prefix), sum(ext)
    kb, vb, k, v = (torch.zeros(n, 1, D, dtype=dtype) for n in (P, P, T, T))
    refs, sizes = [], []
    for b, (pre, n) in enumerate(zip(prefix, ext)):
        at, had, N = sum(ext[:b]), sum(prefix[:b]), pre + n
        t = -(6 * torch.rand(N, generator=g)).to(dtype).double()
        t[N // 3] = 0
        w = t.exp()
        x = (torch.randn(N, D, generator=g, dtype=torch.float64) / w[:, None]).to(dtype).double()
        for i in torch.argsort(w)[:5].flip(0):
            x[i] = 0
            x[i] = (-(w[:, None] * x).sum(0) / w[i]).to(dtype).double()
        kb[had:had + pre, 0, 0], k[at:at + n, 0, 0] = t[:pre].to(dtype), t[pre:].to(dtype)
        vb[had:had + pre, 0], v[at:at + n, 0] = x[:pre].to(dtype), x[pre:].to(dtype)
        refs.append((w[:, None] * x).sum(0) / w.sum())
        sizes.append((w[:, None] * x).square().sum(0).sqrt() / w.sum())
    q = torch.zeros(T, 2, D, dtype=dtype)
    q[..., 0] = 1
    got = _extend(ops, q, k, v, kb, vb, torch.arange(P), prefix, ext, causal=False).cpu().double()
    for b, (ref, size) in enumerate(zip(refs, sizes)):
        rows = got[sum(ext[:b]):sum(ext[:b + 1])]
        assert ((rows - ref).abs() / size).max() < 2 * 2 ** -20, b


@pytest.mark.parametrize("first,second", [(3, 7), (7, 3), (3, 70), (70, 3), (140, 5)], ids=lambda x: str(x))
def test_weights_below_the_normal_range(ops, first, second):
    """Head dimension 64: a value of 2^120 at a weight of 2^-129.8, beside a zero at weight 1, in the same tile and in others, in front and behind: 2^-9.8,
    up to the bits that bf16 terms have there (multiples of 2^-133)."""
    D, N = 64, 150
    kb, vb = torch.zeros(N, 1, D), torch.zeros(N, 1, D)
    kb[:, :, 0] = -2000.0
    kb[first, :, 0], vb[first] = -90.0, 2.0 ** 120
    kb[second, :, 0] = 0.0
    q = torch.zeros(2, 4, D)
    q[..., 0] = 1
    new = torch.zeros(2, 1, D)
    new[..., 0] = -2000.0
    q, new, kb, vb = (t.to(torch.bfloat16) for t in (q, new, kb, vb))
    want = 2.0 ** 120 * torch.exp(torch.tensor(-90.0, dtype=torch.float64)).item()
    for mask in (None, [torch.ones(2, N + 2, dtype=torch.bool)]):
        got = _extend(ops, q, new, torch.zeros_like(new), kb, vb, torch.arange(N), [N], [2], mask=mask)
        assert (got.double() / want - 1).abs().max() < 2 ** -4
