"""Decode attention on the matrix cores at the edges of a tile and of the number range: rows that no key of the range stands for, infinite
value rows, weights far below the largest, sequences of no tokens."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
KINDS = [(64, torch.bfloat16, False), (64, torch.float16, False), (128, torch.bfloat16, False), (128, torch.float16, False), (128, torch.bfloat16, True)]
IDS = ["d64-bf16", "d64-f16", "d128-bf16", "d128-f16", "d128-fp8"]


@pytest.fixture(scope="module")
def ops():
    from sglang_custom_amd import ops

    return ops


def _batch(lens, seed=0):
    """Page table, request rows and the newest token's slot of sequences with slots of their own (slot 0: nobody's)."""
    g = torch.Generator().manual_seed(seed)
    perm = (torch.randperm(sum(lens), generator=g) + 1).int()
    r2t = torch.zeros(len(lens), max(lens) + 4, dtype=torch.int32)
    for b, part in enumerate(perm.split(list(lens))):
        r2t[b, : len(part)] = part
    loc = torch.tensor([int(r2t[b, n - 1]) for b, n in enumerate(lens)])
    return r2t.to(DEV), torch.arange(len(lens), device=DEV), loc.to(DEV), sum(lens) + 1


@pytest.mark.parametrize("hq,hkv", [(8, 2), (8, 1), (2, 2)])
@pytest.mark.parametrize("D,dtype,fp8", KINDS, ids=IDS)
def test_newest_slot_held_no_numbers(ops, D, dtype, fp8, hq, hkv):
    """The fused launch writes the newest token's rows itself; what their slot held before leaves no trace in the result."""
    lens = [1, 2, 15, 16, 17, 31, 33, 48, 63, 64, 65, 80, 81, 97, 129, 200]
    r2t, rpi, loc, slots = _batch(lens)
    bs, lens_t = len(lens), torch.tensor(lens, device=DEV)
    g = torch.Generator().manual_seed(D + hq)
    part = torch.randn(2, bs, (hq + 2 * hkv) * D, generator=g).to(DEV)
    cache = torch.cat([torch.randn(256, D // 2, generator=g).cos(), torch.randn(256, D // 2, generator=g).sin()], 1).to(DEV)
    kb0, vb0 = (torch.randn(slots, hkv, D, generator=g).to(DEV, dtype) for _ in range(2))
    if fp8:
        kb0, vb0 = kb0.to(torch.float8_e4m3fn), vb0.to(torch.float8_e4m3fn)
    for splits in (1, 3):
        for tickets in (None, torch.zeros(bs * hq, dtype=torch.int32, device=DEV)):
            got = []
            for stale in ((0.0, float("nan")) if fp8 else (0.0, float("nan"), float("inf"))):
                kb, vb = kb0.clone(), vb0.clone()
                for t in (kb, vb):
                    rows = torch.full((bs, hkv, D), stale, device=DEV)
                    t[loc] = rows.to(t.dtype)
                o = torch.empty(bs, hq, D, device=DEV, dtype=dtype)
                logits, lse = torch.empty(bs, hq, splits, D, device=DEV), torch.empty(bs, hq, splits, device=DEV)
                ops.decode_attention_fused_qkv(part, lens_t - 1, loc, cache, kb, vb, o, r2t, rpi, lens_t, logits, lse, splits, D ** -0.5, tickets=tickets)
                assert not o.isnan().any(), (splits, tickets is not None, stale)
                got.append(o)
            assert all(torch.equal(got[0], o) for o in got[1:])


def _paged(ops, q, kb, vb, lens, r2t, rpi, splits, tickets=None, scale=1.0):
    bs, hq, D = q.shape
    o = torch.empty_like(q)
    logits, lse = torch.empty(bs, hq, splits, D, device=DEV), torch.empty(bs, hq, splits, device=DEV)
    ops.decode_attention_paged(q, kb, vb, o, r2t, rpi, lens, logits, lse, splits, scale, tickets=tickets)
    return o


@pytest.mark.parametrize("hq,hkv", [(8, 2), (8, 1), (2, 2)])
@pytest.mark.parametrize("D,dtype,fp8", KINDS[:4], ids=IDS[:4])
def test_infinite_value_rows(ops, D, dtype, fp8, hq, hkv):
    """An infinite value makes its feature infinite, whatever its key's weight (the largest included), and touches no other."""
    lens = [1, 5, 16, 17, 64, 65, 90, 130]
    r2t, rpi, _, slots = _batch(lens, 1)
    g = torch.Generator().manual_seed(D + hq)
    q = (torch.randn(len(lens), hq, D, generator=g) * 0.3).to(DEV, dtype)
    kb, vb = (torch.randn(slots, hkv, D, generator=g).to(DEV, dtype) for _ in range(2))
    lens_t = torch.tensor(lens, device=DEV)
    for splits in (1, 3):
        plain = _paged(ops, q, kb, vb, lens_t, r2t, rpi, splits, scale=D ** -0.5)
        for key in (0, 4, 15, 16, 64, 89):      # (the sequences longer than that have it)
            v2, has = vb.clone(), [b for b, n in enumerate(lens) if n > key]
            rows = r2t[has, key].long()
            v2[rows, :, 3], v2[rows, :, D - 1] = float("inf"), float("-inf")
            got = _paged(ops, q, kb, v2, lens_t, r2t, rpi, splits, scale=D ** -0.5)
            assert (got[has][..., 3] == float("inf")).all() and (got[has][..., D - 1] == float("-inf")).all(), (splits, key)
            got[has, :, 3], got[has, :, D - 1] = plain[has, :, 3], plain[has, :, D - 1]
            assert torch.equal(got, plain)


@pytest.mark.parametrize("hq,hkv", [(8, 2), (8, 1), (2, 2)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
def test_weights_of_fp32(ops, dtype, hq, hkv):
    """Head dimension 64 multiplies values by fp32 weights.  The terms of every sum are alike in size (values grow as weights fall) and cancel, so
    that the result is the sum's error: 0.5 to 0.8 times 2^-20 of the terms' root sum of squares in fp32, 5 with weights of 16 bits in
    bf16 and 7.5 with two fp16 terms (each in torch on the CPU, the same values)."""
    D, lens = 64, [200, 77, 129]
    r2t, rpi, _, slots = _batch(lens, 2)
    g = torch.Generator().manual_seed(3)
    kb, vb = torch.zeros(slots, hkv, D, dtype=dtype), torch.zeros(slots, hkv, D, dtype=dtype)
    ref, size = torch.zeros(len(lens), hkv, D, dtype=torch.float64), torch.zeros(len(lens), hkv, D, dtype=torch.float64)
    for b, n in enumerate(lens):
        s = r2t[b, :n].long().cpu()
        for h in range(hkv):
            t = -(6 * torch.rand(n, generator=g)).to(dtype).double()
            t[n // 3] = 0
            w = t.exp()
            v = (torch.randn(n, D, generator=g, dtype=torch.float64) / w[:, None]).to(dtype).double()
            for k in torch.argsort(w)[:5].flip(0):
                v[k] = 0
                v[k] = (-(w[:, None] * v).sum(0) / w[k]).to(dtype).double()
            kb[s, h, 0], vb[s, h] = t.to(dtype), v.to(dtype)
            ref[b, h] = (w[:, None] * v).sum(0) / w.sum()
            size[b, h] = (w[:, None] * v).square().sum(0).sqrt() / w.sum()
    q = torch.zeros(len(lens), hq, D, dtype=dtype)
    q[..., 0] = 1
    ref, size = (t.repeat_interleave(hq // hkv, 1) for t in (ref, size))
    for splits in (1, 3):
        got = _paged(ops, q.to(DEV), kb.to(DEV), vb.to(DEV), torch.tensor(lens, device=DEV), r2t, rpi, splits)
        assert ((got.cpu().double() - ref).abs() / size).max() < 2 * 2 ** -20


@pytest.mark.parametrize("first,second", [(3, 7), (7, 3), (3, 70), (70, 3), (5, 30)], ids=lambda x: str(x))
@pytest.mark.parametrize("D", [64, 128])
def test_weights_below_the_normal_range(ops, D, first, second):
    """A value of 2^120 at a weight of 2^-129.8, beside a zero at weight 1, in the same tile and in others, in front and behind: 2^-9.8, up to
    the bits that 16-bit weights have left there at head dimension 128 (multiples of 2^-133)."""
    r2t, rpi, _, slots = _batch([80], 3)
    kb, vb = torch.zeros(slots, 1, D), torch.zeros(slots, 1, D)
    s = r2t[0, :80].long().cpu()
    kb[s, :, 0] = -2000.0
    kb[s[first], :, 0], vb[s[first]] = -90.0, 2.0 ** 120
    kb[s[second], :, 0] = 0.0
    q = torch.zeros(1, 4, D)
    q[..., 0] = 1
    for splits in (1, 2):
        got = _paged(ops, *(t.to(DEV, torch.bfloat16) for t in (q, kb, vb)), torch.tensor([80], device=DEV), r2t, rpi, splits)
        want = 2.0 ** 120 * torch.exp(torch.tensor(-90.0, dtype=torch.float64)).item()
        assert (got.double() / want - 1).abs().max() < (2 ** -7 if D == 64 else 2 ** -4), got.flatten()[:2]


@pytest.mark.parametrize("D,dtype,fp8", KINDS, ids=IDS)
@pytest.mark.parametrize("lens", [[0, 33, 0, 1, 0], [0, 0], [70, 0]], ids=lambda x: "-".join(map(str, x)))
def test_no_tokens(ops, D, dtype, fp8, lens):
    """Sequences of no tokens first, in the middle and last: zeros.  By index list (an index pointer cut from a longer one, whose first value
    lies past the pool), by page table and in the fused launch, where they leave the cache as it is."""
    hq, hkv, bs = 8, 2, len(lens)
    r2t, rpi, _, slots = _batch([max(n, 1) for n in lens], 4)
    lens_t, live = torch.tensor(lens, device=DEV), [b for b, n in enumerate(lens) if n]
    g = torch.Generator().manual_seed(D)
    q = torch.randn(bs, hq, D, generator=g).to(DEV, dtype)
    kb, vb = (torch.randn(slots, hkv, D, generator=g).to(DEV, torch.float8_e4m3fn if fp8 else dtype) for _ in range(2))
    first = slots + 1000
    indptr = torch.tensor([0, first] + [first + sum(lens[: i + 1]) for i in range(bs)], dtype=torch.int32, device=DEV)[1:]
    indices = torch.zeros(first + sum(lens) + 8, dtype=torch.int32)
    indices[first: first + sum(lens)] = torch.cat([r2t[b, :n].cpu() for b, n in enumerate(lens)])
    part = torch.randn(2, bs, (hq + 2 * hkv) * D, generator=g).to(DEV)
    cache = torch.cat([torch.randn(96, D // 2, generator=g).cos(), torch.randn(96, D // 2, generator=g).sin()], 1).to(DEV)
    loc = torch.tensor([int(r2t[b, max(n - 1, 0)]) for b, n in enumerate(lens)], device=DEV)
    for splits in (1, 3):
        logits, lse = torch.empty(bs, hq, splits, D, device=DEV), torch.empty(bs, hq, splits, device=DEV)
        outs = [torch.full((bs, hq, D), 7.0, device=DEV, dtype=dtype) for _ in range(5)]
        ops.decode_attention_fwd(q, kb, vb, outs[0], indptr, indices.to(DEV), logits, lse, splits, splits, D ** -0.5)
        tickets = torch.zeros(bs * hq, dtype=torch.int32, device=DEV)
        for o, tk in zip(outs[1:3], (None, tickets)):
            ops.decode_attention_paged(q, kb, vb, o, r2t, rpi, lens_t, logits, lse, splits, D ** -0.5, tickets=tk)
        assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
        for o, tk in zip(outs[3:], (None, tickets)):
            kb2, vb2 = kb.clone(), vb.clone()
            ops.decode_attention_fused_qkv(part, (lens_t - 1).clamp(min=0), loc, cache, kb2, vb2, o, r2t, rpi, lens_t, logits, lse, splits, D ** -0.5, tickets=tk)
            for b in set(range(bs)) - set(live):
                assert torch.equal(kb2[loc[b]].view(torch.uint8), kb[loc[b]].view(torch.uint8)) and torch.equal(vb2[loc[b]].view(torch.uint8), vb[loc[b]].view(torch.uint8))
        assert torch.equal(outs[3], outs[4]) and (tickets == 0).all()
        for o in outs:
            assert all((o[b] == 0).all() if b not in live else ((o[b].abs() < 6).all() and (o[b] != 0).any()) for b in range(bs))
