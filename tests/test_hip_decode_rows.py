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
