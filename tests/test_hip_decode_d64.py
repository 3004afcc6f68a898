"""Decode attention at head dimension 64 on the matrix cores: the launch that starts from the qkv projection's partials against the
separate ones bit for bit, and against float64, around its tiles of 16 keys, its steps of 64 and its splits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def ops():
    from sglang_custom_amd import ops

    return ops


@pytest.mark.parametrize("dtype,cache_dtype", [(torch.bfloat16, torch.float32), (torch.float16, torch.float16)], ids=["bf16", "f16"])
@pytest.mark.parametrize("hq,hkv,bs,maxlen,splits", [(32, 8, 9, 300, 1), (8, 8, 5, 70, 1), (16, 2, 6, 530, 3), (8, 4, 4, 129, 2), (8, 1, 3, 2100, 7)])
def test_fused_launch_and_float64(ops, dtype, cache_dtype, hq, hkv, bs, maxlen, splits):
    g = torch.Generator().manual_seed(hq * 100 + maxlen)
    D, hidden = 64, 1024
    n = (hq + 2 * hkv) * D
    wp = ops.pack_weight((torch.randn(n, hidden, generator=g) * 0.04).to(DEV, dtype))
    x = torch.randn(bs, hidden, generator=g).to(DEV, dtype)
    lens = torch.randint(1, maxlen, (bs,), generator=g)
    lens[0], lens[-1] = maxlen, 1
    for i in range(1, min(bs - 1, 6)):
        lens[i] = min(17 * i + 1, maxlen)       # the newest key in row i of tile i
    slots = int(lens.sum()) + 8
    perm = (torch.randperm(slots - 1, generator=g) + 1).int()
    r2t = torch.zeros(bs + 3, maxlen + 8, dtype=torch.int32)
    rpi = torch.randperm(bs + 3, generator=g)[:bs]
    for b, part in enumerate(perm[: int(lens.sum())].split(lens.tolist())):
        r2t[rpi[b], : len(part)] = part
    loc = torch.stack([r2t[rpi[b], int(lens[b]) - 1] for b in range(bs)]).long().to(DEV)
    r2t, rpi, lens = r2t.to(DEV), rpi.to(DEV), lens.to(DEV)
    cache = torch.cat([torch.randn(maxlen + 8, D // 2, generator=g).cos(), torch.randn(maxlen + 8, D // 2, generator=g).sin()], 1).to(DEV, cache_dtype)
    kb0, vb0 = (torch.randn(slots, hkv, D, generator=g).to(DEV, dtype) for _ in range(2))
    logits = torch.empty(bs, hq, 8, D, dtype=torch.float32, device=DEV)
    lse = torch.empty(bs, hq, 8, dtype=torch.float32, device=DEV)
    kb, vb = kb0.clone(), vb0.clone()
    q, k, v = ops.linear_packed(x, wp, n).split([hq * D, hkv * D, hkv * D], dim=-1)
    ops.rope_inplace(lens - 1, q, k, D, cache, True, v=v, k_buffer=kb, v_buffer=vb, loc=loc)
    q = q.reshape(bs, hq * D).contiguous().view(bs, hq, D)
    want = torch.empty(bs, hq, D, device=DEV, dtype=dtype)
    ops.decode_attention_paged(q, kb, vb, want, r2t, rpi, lens, logits, lse, splits, D ** -0.5)
    part = ops.linear_packed_partials(x, wp, n)
    for tickets in (None, torch.zeros(bs * hq, dtype=torch.int32, device=DEV)):     # merged by a second launch, and in the launch (twice)
        for _ in range(2 if tickets is not None else 1):
            kb2, vb2 = kb0.clone(), vb0.clone()
            o = torch.empty_like(want)
            ops.decode_attention_fused_qkv(part, lens - 1, loc, cache, kb2, vb2, o, r2t, rpi, lens, logits, lse, splits, D ** -0.5, tickets=tickets)
            assert torch.equal(kb, kb2) and torch.equal(vb, vb2)
            assert torch.equal(o, want)
    # rounding of the result (2^-9 of up to 3 in bf16) and as much again: scores, exponentials and sums in fp32 are far below it
    for b in range(bs):
        s = r2t[rpi[b], : int(lens[b])].long()
        kk, vv = (t[s].double().repeat_interleave(hq // hkv, 1).cpu() for t in (kb, vb))
        p = torch.softmax(torch.matmul(q[b].double().cpu()[:, None], kk.permute(1, 2, 0))[:, 0] * D ** -0.5, -1)
        ref = torch.matmul(p[:, None], vv.transpose(0, 1))[:, 0]
        assert (want[b].cpu().double() - ref).abs().max() <= ref.abs().max() * 2 ** (-8 if dtype == torch.bfloat16 else -10)


def test_empty_sequences(ops):
    """A sequence of no tokens beside others: zeros, with one split and more, by page table."""
    hq, hkv, D = 8, 2, 64
    q = torch.randn(3, hq, D, device=DEV).bfloat16()
    kb, vb = torch.randn(70, hkv, D, device=DEV).bfloat16(), torch.randn(70, hkv, D, device=DEV).bfloat16()
    lens = torch.tensor([0, 33, 0], device=DEV)
    r2t = torch.arange(1, 70, dtype=torch.int32, device=DEV).repeat(3, 1)[:, :40].contiguous()
    logits, lse = torch.empty(3, hq, 4, D, device=DEV), torch.empty(3, hq, 4, device=DEV)
    outs = []
    for splits in (1, 3):
        o = torch.full((3, hq, D), 7.0, device=DEV).bfloat16()
        ops.decode_attention_paged(q, kb, vb, o, r2t, torch.arange(3, device=DEV), lens, logits, lse, splits, D ** -0.5)
        assert (o[0] == 0).all() and (o[2] == 0).all() and o[1].abs().max() > 0
        outs.append(o)
    assert (outs[0].float() - outs[1].float()).abs().max() < 2e-2
