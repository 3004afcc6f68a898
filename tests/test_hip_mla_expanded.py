"""MLA prefill over kv_b_proj's output as it is: the rotation launch and the attention with the keys' rope part once per token."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("lens,H,nope,rope,vd,rank", [((37,), 16, 128, 64, 128, 512), ((1,), 128, 128, 64, 128, 512), ((300, 1, 129), 3, 128, 64, 128, 128),
                                                      ((5,), 2, 8, 16, 8, 8), ((9, 2), 5, 24, 256, 16, 48)])
@pytest.mark.parametrize("dt,cs_dt,neox", [(torch.bfloat16, torch.bfloat16, False), (torch.float16, torch.float32, False), (torch.bfloat16, torch.float32, True)])
@pytest.mark.parametrize("kv8", [False, True], ids=["cache16", "cache_fp8"])
def test_rotation_launch_and_expanded_attention(lens, H, nope, rope, vd, rank, dt, cs_dt, neox, kv8):
    """q, k_pe and the cache rows bit for bit mla_prefill_assemble's.  Attention (where the heads are of 128 + 64 and 128)
    against float64: the weights rounded to the tensor type (u of every term), the result once more; fp32 scores and exp add
    less than half of that."""
    from sglang_custom_amd import ops

    g = torch.Generator().manual_seed(rope + H)
    T = sum(lens)
    q, kv, lat, ckv = (torch.randn(s, generator=g).to(dt).to(DEV) for s in
                       ((T, H, nope + rope), (T, H, nope + vd), (T, 24 + rank + rope), (T, rank + 8)))
    k_pe, ckv = lat[:, 24 + rank:], ckv[:, :rank]
    cs = torch.cat([torch.randn(5000, rope // 2, generator=g).cos(), torch.randn(5000, rope // 2, generator=g).sin()], 1).to(cs_dt).to(DEV).contiguous()
    positions = torch.randint(0, 5000, (T,), generator=g).to(DEV)
    loc = (torch.randperm(2 * T + 2, generator=g)[:T] + 1).to(DEV)
    want_cache = torch.zeros((2 * T + 3, 1, rank + rope), dtype=torch.float8_e4m3fn if kv8 else dt, device=DEV)
    cache, want_q, got_q = want_cache.clone(), q.clone(), q.clone()
    want_k, _ = ops.mla_prefill_assemble(want_q, kv, k_pe, ckv, positions, cs, neox, want_cache, loc, nope, rope, vd)
    pe = ops.mla_prefill_rotate(got_q, k_pe, ckv, positions, cs, neox, cache, loc)
    torch.cuda.synchronize()
    bits = torch.uint8 if kv8 else torch.int16
    assert torch.equal(got_q.view(torch.int16), want_q.view(torch.int16)) and torch.equal(cache.view(bits), want_cache.view(bits))
    assert torch.equal(pe.view(torch.int16), want_k[:, 0, nope:].contiguous().view(torch.int16))
    if not ops.latent_prefill_attention_supported(nope, rope, vd, 0, False, dt):
        return
    n = torch.tensor(lens, dtype=torch.int32)
    start = torch.cumsum(n, 0).to(torch.int32) - n
    out = ops.latent_prefill_attention(got_q, kv, pe, start.to(DEV), n.to(DEV), positions, None, 0, max(lens), (nope + rope) ** -0.5)
    u = torch.finfo(dt).eps / 2
    for s, m in zip(start.tolist(), lens):
        mask = torch.ones(m, m, dtype=torch.bool, device=DEV).tril()
        for h in range(H):
            k = torch.cat([kv[s: s + m, h, :nope], pe[s: s + m]], 1).double()
            v = kv[s: s + m, h, nope:].double()
            p = torch.softmax((got_q[s: s + m, h].double() @ k.T * (nope + rope) ** -0.5).masked_fill(~mask, float("-inf")), -1)
            want = p @ v
            err, bound = (out[s: s + m, h].double() - want).abs(), 1.5 * u * (p @ v.abs() + want.abs()) + 1e-6
            assert bool((err <= bound).all()), (s, h, (err / bound).max().item())
