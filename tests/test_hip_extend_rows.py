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
    # dimension 128, the rest after two of them at 64; 1e-5 for fp32 sums and exponentials
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
    tile edges, against float32 softmax; bound: weights and V exact to 2^-16, the output's rounding to bf16 (2^-8 of values up to 3)."""
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
