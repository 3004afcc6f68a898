"""GPU: attention of whole prompts over expanded latents (ops.latent_prefill_attention) against float64, at the edges of its
64-key tiles and 128-query blocks, both rotations, strided inputs."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rotate(x, pos, f, rot, interleaved, mag):
    if not rot:
        return x
    a = pos.double()[:, None, None] * f.double()
    c, s = mag * torch.cos(a), mag * torch.sin(a)
    out = x.clone()
    i = slice(0, rot, 2) if interleaved else slice(0, rot // 2)
    j = slice(1, rot, 2) if interleaved else slice(rot // 2, rot)
    out[..., i], out[..., j] = x[..., i] * c - x[..., j] * s, x[..., j] * c + x[..., i] * s
    return out


@pytest.mark.parametrize("lens", [(1, 65), (63, 64, 2), (127, 128, 129), (300, 1, 193)])
@pytest.mark.parametrize("dtype,rot,interleaved,H", [(torch.bfloat16, 64, True, 3), (torch.bfloat16, 64, False, 16), (torch.float16, 32, True, 2),
                                                     (torch.bfloat16, 0, False, 1)])
def test_latent_prefill_attention(lens, dtype, rot, interleaved, H):
    """Tolerance: T-rounded weights (half an ulp of 1 per key, averaged) and the rounded result: 2^-8 (bf16) / 2^-11 (fp16) of the
    values' scale each, and the scores' own rounding of q (2^-9 relative over 192 terms of unit size: 0.03 of a score in bf16)."""
    from sglang_custom_amd import ops

    assert ops.latent_prefill_attention_supported(128, 64, 128, rot, interleaved, dtype)
    g = torch.Generator().manual_seed(sum(lens) + H + rot)
    T = sum(lens)
    big = torch.randn(T, H * 192 + 40, generator=g).to(dtype)
    q = big[:, 8: 8 + H * 192].view(T, H, 192)
    kv = torch.randn(T, H, 256, generator=g).to(dtype)
    rows = torch.randn(T, 72, generator=g).to(dtype)
    f = torch.rand(32, generator=g) * 0.5
    pos = torch.cat([torch.arange(n) for n in lens])
    start = torch.tensor([sum(lens[:i]) for i in range(len(lens))], dtype=torch.int32)
    mag = 1.2
    bd, rd = big.to(DEV), rows.to(DEV)
    got = ops.latent_prefill_attention(bd[:, 8: 8 + H * 192].view(T, H, 192), kv.to(DEV), rd[:, 8:], start.to(DEV),
                                       torch.tensor(lens, dtype=torch.int32, device=DEV), pos.to(DEV), f.to(DEV), rot, max(lens), 0.1,
                                       interleaved=interleaved, rot_mag=mag).cpu().double()
    qd, kd, vd = q.double().clone(), kv.double()[..., :128], kv.double()[..., 128:]
    qd[..., 128:] = _rotate(qd[..., 128:], pos, f[: rot // 2], rot, interleaved, mag).to(dtype).double()
    k = torch.cat([kd, rows.double()[:, None, 8:].expand(T, H, 64)], -1)
    tol = 0.02 if dtype == torch.bfloat16 else 0.004
    for s, n in zip(start.tolist(), lens):
        sc = torch.einsum("qhd,khd->hqk", qd[s: s + n], k[s: s + n]) * 0.1
        sc = sc.masked_fill(torch.ones(n, n, dtype=torch.bool).triu(1), float("-inf"))
        want = torch.einsum("hqk,khd->qhd", torch.softmax(sc, -1), vd[s: s + n])
        assert (got[s: s + n] - want).abs().max() < tol, n
        assert (got[s: s + n] - want).norm() < 0.25 * tol * want.norm() + 1e-9


def test_refusals():
    from sglang_custom_amd import ops

    assert not ops.latent_prefill_attention_supported(128, 64, 128, 32, False, torch.bfloat16)     # pairs across lanes
    assert not ops.latent_prefill_attention_supported(64, 64, 128, 64, True, torch.bfloat16)
    assert not ops.latent_prefill_attention_supported(128, 64, 128, 64, True, torch.float32)


@pytest.mark.parametrize("lens", [[1], [70, 1, 129]])
@pytest.mark.parametrize("kv_far,rope_far", [(True, False), (False, True), (True, True)])
def test_rows_far_apart(lens, kv_far, rope_far):
    """Rows 2^23 elements apart, further than 32-bit offsets reach, one row (whose stride torch does not take for one) and several: the bits
    of the same rows close together."""
    from sglang_custom_amd import ops

    T, H, stride = sum(lens), 2, 1 << 23
    g = torch.Generator(device=DEV).manual_seed(T)
    q, kv, rope = (torch.randn(T, w, device=DEV, generator=g).bfloat16() for w in (H * 192, H * 256, 64))
    start = torch.tensor([sum(lens[:i]) for i in range(len(lens))], dtype=torch.int32, device=DEV)
    n, pos = torch.tensor(lens, dtype=torch.int32, device=DEV), torch.arange(T, device=DEV)

    def far(x):
        rows = torch.empty((T - 1) * stride + x.shape[1], dtype=x.dtype, device=DEV).as_strided(x.shape, (stride, 1))
        return rows.copy_(x)

    def run(kv, rope):
        assert kv.stride(0) in (H * 256, stride)
        return ops.latent_prefill_attention(q.view(T, H, 192), kv.as_strided((T, H, 256), (kv.stride(0), 256, 1)), rope, start, n, pos, None, 0,
                                            max(lens), 0.1)

    assert torch.equal(run(far(kv) if kv_far else kv, far(rope) if rope_far else rope), run(kv, rope))
