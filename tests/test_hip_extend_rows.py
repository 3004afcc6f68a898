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
