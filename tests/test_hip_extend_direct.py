"""Prefill attention whose tiles the load unit writes into LDS itself (16-bit rows at head dimension 128): the bits of the launch that takes
them through registers, which serves caches too large for 32-bit offsets, wherever a prefix ends in a tile; and float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


# prefixes that end at, before and behind a tile's edge, or are none; last blocks of one row, of a wave's 32 and of one more
@pytest.mark.parametrize("lens", [[(0, 1)], [(0, 129), (0, 64)], [(1, 33), (63, 32), (64, 65)], [(65, 200), (300, 1), (0, 161)], [(700, 130)]])
@pytest.mark.parametrize("head_major", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_direct_tiles_are_the_register_tiles(lens, head_major, dtype):
    from sglang_custom_amd import _lib, ops

    lib = _lib.load()
    hq, hkv, D = 8, 2, 128
    g = torch.Generator(device=DEV).manual_seed(sum(a + 7 * b for a, b in lens))
    T, P = sum(b for _, b in lens), sum(a for a, _ in lens)

    def rnd(*shape):
        return torch.randn(*shape, device=DEV, generator=g).to(dtype)

    qkv = rnd(T, (hq + 2 * hkv) * D)      # rows of a wider buffer
    q, k, v = qkv[:, :hq * D], qkv[:, hq * D:(hq + hkv) * D], qkv[:, (hq + hkv) * D:]
    slots = P + 9
    pools = [torch.full((hkv, slots, D) if head_major else (slots, hkv, D), float("nan"), device=DEV, dtype=dtype) for _ in range(2)]
    kb, vb = (p.transpose(0, 1) if head_major else p for p in pools)
    kvi = (torch.randperm(slots, device=DEV, generator=g)[:P] if P else torch.zeros(1, device=DEV)).int()
    for b in (kb, vb):
        if P:
            b[kvi.long()] = rnd(P, hkv, D)
    qo = torch.tensor([0] + torch.tensor([b for _, b in lens]).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    kvp = torch.tensor([0] + torch.tensor([a for a, _ in lens]).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    longest = max(b for _, b in lens)
    dt = ops._kvdt(q.view(T, hq, D), kb, vb)

    def run(num_slots, splits):
        o = torch.full((T, hq, D), float("nan"), device=DEV, dtype=dtype)
        need = lib.mi355_extend_attention_workspace_bytes(T, hq, D, splits) if splits > 1 else 0
        ws = torch.empty(max(need, 16), dtype=torch.uint8, device=DEV)
        assert lib.mi355_extend_attention_ws(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), pools[0].data_ptr(), pools[1].data_ptr(), qo.data_ptr(), kvp.data_ptr(),
            kvi.data_ptr(), None, None, 1, 1, len(lens), longest, hq, hkv, D, D, qkv.stride(0), qkv.stride(0), qkv.stride(0), num_slots, D ** -0.5, 0.0,
            0, dt, T, splits, ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream) == 0
        return o

    for splits in (1, 2):
        got = run(slots, splits)
        if not head_major:     # (there num_slots says where a head begins)
            assert torch.equal(got, run(1 << 25, splits))
        for b, (pre, ext) in enumerate(lens):
            s, c = int(qo[b]), kvi[int(kvp[b]):int(kvp[b]) + pre].long()
            kk, vv = (torch.cat([buf[c], x[s:s + ext].view(ext, hkv, D)]).double().repeat_interleave(hq // hkv, 1) for buf, x in ((kb, k), (vb, v)))
            sc = torch.einsum("qhd,khd->hqk", q[s:s + ext].view(ext, hq, D).double(), kk) * D ** -0.5
            sc = sc.masked_fill(~torch.ones(ext, pre + ext, dtype=torch.bool, device=DEV).tril(pre), -float("inf"))
            ref = torch.einsum("hqk,khd->qhd", torch.softmax(sc, -1), vv)
            # 16-bit weights and one rounding of the result, of values of norm one
            eps = 2 ** -8 if dtype == torch.bfloat16 else 2 ** -11
            assert (got[s:s + ext].double() - ref).norm() <= 1.5 * eps * ref.norm()


def test_cached_offsets_past_two_gib():
    """Slots whose rows lie more than 2^31 bytes behind the first: the offsets are unsigned."""
    from sglang_custom_amd import ops

    hq, hkv, D, slots, P, T = 8, 8, 128, 1_900_000, 100, 40
    if torch.cuda.get_device_properties(0).total_memory < 32 << 30:
        pytest.skip("8 GiB of cache")
    g = torch.Generator(device=DEV).manual_seed(3)
    kb, vb = (torch.zeros(slots, hkv, D, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    rows = [torch.randn(P, hkv, D, device=DEV, generator=g).bfloat16() for _ in range(2)]
    q, k, v = (torch.randn(T, h, D, device=DEV, generator=g).bfloat16() for h in (hq, hkv, hkv))
    qo, kvp = (torch.tensor([0, n], dtype=torch.int32, device=DEV) for n in (T, P))
    out = []
    for first in (5, slots - P - 5):
        at = torch.arange(first, first + P, device=DEV)
        kb[at], vb[at] = rows
        o = torch.empty(T, hq, D, device=DEV, dtype=torch.bfloat16)
        ops.extend_attention_fwd(q, k, v, o, kb, vb, qo, kvp, at.int(), None, True, None, T, D ** -0.5)
        out.append(o)
    assert torch.equal(out[0], out[1]) and bool((out[0] != 0).any())


@pytest.mark.parametrize("num_slots", [1, 0, 2_200_000])
def test_slots_past_four_gib(num_slots):
    """A cache of more than 4 GiB, its rows near, far and mixed within a tile, whatever count of slots the caller gives ([slots, heads, D] does
    not need it): the bits of a small cache with the same rows."""
    from sglang_custom_amd import _lib, ops

    lib = _lib.load()
    hq, hkv, D, slots, P, T = 8, 8, 128, 2_200_000, 300, 40
    if torch.cuda.get_device_properties(0).total_memory < 32 << 30:
        pytest.skip("9 GiB of cache")
    g = torch.Generator(device=DEV).manual_seed(4)
    rows = [torch.randn(P, hkv, D, device=DEV, generator=g).bfloat16() for _ in range(2)]
    q, k, v = (torch.randn(T, h, D, device=DEV, generator=g).bfloat16() for h in (hq, hkv, hkv))
    qo, kvp = (torch.tensor([0, n], dtype=torch.int32, device=DEV) for n in (T, P))

    def run(kb, vb, at, count, splits):
        o = torch.full((T, hq, D), float("nan"), device=DEV, dtype=torch.bfloat16)
        need = lib.mi355_extend_attention_workspace_bytes(T, hq, D, splits) if splits > 1 else 0
        ws, kvi = torch.empty(max(need, 16), dtype=torch.uint8, device=DEV), at.int()
        assert lib.mi355_extend_attention_ws(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), kb.data_ptr(), vb.data_ptr(), qo.data_ptr(), kvp.data_ptr(), kvi.data_ptr(), None,
            None, 1, 1, 1, T, hq, hkv, D, D, hq * D, hkv * D, hkv * D, count, D ** -0.5, 0.0, 0, ops._kvdt(q, kb, vb), T, splits, ws.data_ptr(), need,
            torch.cuda.current_stream().cuda_stream) == 0
        return o

    near = torch.arange(5, 5 + P, device=DEV)
    far = torch.arange(slots - 5 - P, slots - 5, device=DEV)
    edge = 0xFFFF0000 // (2 * hkv * D) - 100 + torch.arange(P, device=DEV)          # the first tiles within reach, the last ones not
    mixed = torch.where(torch.arange(P, device=DEV) % 7 == 3, far, near)
    kb, vb = (torch.full((slots, hkv, D), float("nan"), device=DEV, dtype=torch.bfloat16) for _ in range(2))
    want = [run(rows[0], rows[1], torch.arange(P, device=DEV), P, splits) for splits in (1, 2)]
    for at in (near, far, edge, mixed):
        kb[at], vb[at] = rows
        for splits in (1, 2):
            assert torch.equal(run(kb, vb, at, num_slots, splits), want[splits - 1])
