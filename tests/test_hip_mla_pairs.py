"""MLA decode over a 16-bit latent cache with two head groups per workgroup (one ring of rows for 32 heads)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


# head counts: two full groups, an odd group left over (a team without heads), a group of one head, seven groups;
# pair workgroups at the edge of the rule (128) and splits up to its last (4), with splits that a short row leaves empty
@pytest.mark.parametrize("bs,H,splits,neox,dt", [(64, 32, 2, False, torch.bfloat16), (43, 32, 3, True, torch.float16), (64, 48, 2, False, torch.bfloat16),
                                                 (128, 17, 1, True, torch.bfloat16), (32, 100, 2, False, torch.float16), (33, 64, 4, False, torch.bfloat16)])
def test_two_head_groups_share_the_rows(bs, H, splits, neox, dt):
    """Every sequence against float64 attention over the same rows.  Bound: the probabilities are rounded to the tensor type
    for P.V (u of every term), the result once more (u of the result); fp32 scores over 576 terms add less than a quarter of
    that.  The merge inside the launch bit for bit the merge launch, and with RoPE and the cache write inside bit for bit
    rope -> scatter -> decode."""
    from sglang_custom_amd import ops

    rank, rope = 512, 64
    D = rank + rope
    g = torch.Generator().manual_seed(bs + H)
    lens = torch.randint(1, 301, (bs,), generator=g).tolist()
    lens[:12] = [1, 2, 15, 16, 17, 31, 32, 33, 64, 65, 96, 97]
    total = sum(lens)
    cache0 = torch.randn(total + 1, 1, D, generator=g).to(dt).to(DEV)
    r2t = torch.zeros((bs, max(lens)), dtype=torch.int32)
    perm = torch.randperm(total, generator=g) + 1
    pos = 0
    for b, n in enumerate(lens):
        r2t[b, :n] = perm[pos: pos + n].int()
        pos += n
    slots = r2t
    r2t = r2t.to(DEV)
    rpi = torch.arange(bs, dtype=torch.int64, device=DEV)
    lt = torch.tensor(lens, dtype=torch.int64, device=DEV)
    q = torch.randn(bs, H, D, generator=g).to(dt).to(DEV)
    scale = D ** -0.5
    lg = torch.empty(bs * H * splits * rank, dtype=torch.float32, device=DEV)
    ls = torch.empty(bs * H * splits, dtype=torch.float32, device=DEV)
    tickets = torch.zeros(bs * H, dtype=torch.int32, device=DEV)

    def plain(q_in, cache, **kw):
        o = torch.full((bs, H, rank), float("nan"), dtype=dt, device=DEV)
        ops.decode_attention_mla(q_in, cache, o, r2t, rpi, lt, lg, ls, splits, rank, scale, **kw)
        torch.cuda.synchronize()
        return o

    got = plain(q, cache0, tickets=tickets)
    assert torch.equal(got.view(torch.int16), plain(q, cache0).view(torch.int16)) and not tickets.any()
    u = torch.finfo(dt).eps / 2
    for b, n in enumerate(lens):
        rows = cache0[slots[b, :n].long().to(DEV), 0].double()
        p = torch.softmax(q[b].double() @ rows.T * scale, dim=-1)
        want = p @ rows[:, :rank]
        bound = 1.25 * u * (p @ rows[:, :rank].abs() + want.abs()) + 1e-6
        assert bool(((got[b].double() - want).abs() <= bound).all()), (b, n, ((got[b].double() - want).abs() / bound).max().item())

    loc = torch.stack([r2t[b, n - 1] for b, n in enumerate(lens)]).to(torch.int64)
    positions = (lt - 1).clone()
    k_nope = torch.randn(bs, rank, generator=g).to(dt).to(DEV)
    k_pe_raw = torch.randn(bs, rope, generator=g).to(dt).to(DEV)
    cs = torch.cat([torch.randn(512, rope // 2, generator=g).cos(), torch.randn(512, rope // 2, generator=g).sin()], dim=1).to(DEV).contiguous()
    q_ref = q.clone()
    q_pe, k_pe = q_ref[..., rank:].contiguous().view(bs, -1), k_pe_raw.clone()
    ops.rope_inplace(positions, q_pe, k_pe, rope, cs, neox)
    q_ref[..., rank:] = q_pe.view(bs, H, rope)
    cache_ref, cache = cache0.clone(), cache0.clone()
    row = torch.cat([k_nope, k_pe], dim=-1).view(bs, 1, D)
    ops.set_kv_buffer(cache_ref, cache_ref, loc, row, row)
    want = plain(q_ref, cache_ref, tickets=tickets)
    fused = torch.full_like(want, float("nan"))
    ops.decode_attention_mla_fused_rope(q, k_nope, k_pe_raw, positions, loc, cs, neox, cache, fused, r2t, rpi, lt, lg, ls,
                                        splits, rank, scale, 0.0, tickets=tickets)
    torch.cuda.synchronize()
    assert torch.equal(cache.view(torch.int16), cache_ref.view(torch.int16))
    assert torch.equal(fused.view(torch.int16), want.view(torch.int16)) and not tickets.any()
