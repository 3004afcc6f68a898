"""Window attention on the matrix cores where a wave owns whole rows: every width class, ragged runs, odd output strides."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


# (dtype, query heads, kv heads, d, dv, window, pool, sink, head gate, output padding, key ranges of single tokens)
@pytest.mark.parametrize("dt,H,G,d,dv,window,pool,sink,gate,pad,splits", [
    (torch.bfloat16, 8, 2, 128, 128, 40, 8, False, True, 0, 1),
    (torch.float16, 4, 4, 64, 16, 0, 0, True, False, 3, 3),       # one head a kv head, one column tile, stores one by one
    (torch.bfloat16, 6, 2, 96, 80, 33, 0, True, True, 4, 2),      # three heads: rows that no token fills, widths inside a class
    (torch.float16, 16, 1, 160, 208, 64, 16, False, False, 0, 1),  # the widest class, a run's rows past sixteen a wave
    (torch.bfloat16, 2, 1, 32, 256, 1, 0, False, False, 1, 4),    # a window of one key
    (torch.bfloat16, 5, 1, 256, 64, 31, 31, True, False, 0, 2),
])
def test_rows_against_float64(dt, H, G, d, dv, window, pool, sink, gate, pad, splits):
    """Bound: the weights are rounded to the tensor type for P.V (u of every term over the whole denominator), the result once
    more (u of the result); the pooled rows are taken as given.  fp32 scores of up to 256 terms and __expf add less than half of that."""
    from sglang_custom_amd import ops

    g = torch.Generator().manual_seed(H * 1000 + d + dv)
    lens = [1, 2, 31, 32, 33, 65, 150]
    slots, total = [], sum(lens) + len(lens) * max(pool, 1)
    step = max(pool, 1)
    table = torch.zeros(len(lens), 160 + step, dtype=torch.int32)
    at = step
    for b, n in enumerate(lens):      # runs of slots that start on a block, so that a block's pooled row is its last slot / pool
        table[b, :n] = torch.arange(at, at + n, dtype=torch.int32)
        at += -(-n // step) * step
    k = torch.randn(at + step, G, d, generator=g).to(dt).to(DEV)
    v = torch.randn(at + step, G, dv, generator=g).to(dt).to(DEV)
    pk = torch.randn((at + step) // step + 1, G, d, generator=g).to(dt).to(DEV) if pool else None
    pv = torch.randn((at + step) // step + 1, G, dv, generator=g).to(dt).to(DEV) if pool else None
    snk = torch.randn(H, generator=g).to(DEV) if sink else None
    scale, u = d ** -0.5, torch.finfo(dt).eps / 2

    def check(req, pos, blocks, max_run, n_splits):
        T = len(req)
        q = torch.randn(T, H, d, generator=g).to(dt).to(DEV)
        hg = torch.randn(T, H, generator=g).to(dt).to(DEV) if gate else None
        out = torch.full((T, H, dv + pad), float("nan"), dtype=dt, device=DEV)[:, :, :dv]
        ops.window_attention(q, k, v, out, table.to(DEV), torch.arange(len(lens), device=DEV), torch.tensor(pos, device=DEV), snk, window, scale,
                             tok_req=torch.tensor(req, dtype=torch.int32, device=DEV), blocks=blocks, max_run=max_run, num_splits=n_splits,
                             pool=pool, pooled_k=pk, pooled_v=pv, pool_div=step if pool else 1, head_gate=hg)
        torch.cuda.synchronize()
        for t, (b, i) in enumerate(zip(req, pos)):
            lo = max(0, i - window + 1) if window else 0
            rows = table[b, lo: i + 1].long()
            ks, vs = k[rows].double(), v[rows].double()
            if pool:
                last = [e for e in range(pool - 1, i + 1, pool) if e <= i - window]
                blk = (table[b, last].long() // pool) if last else torch.zeros(0, dtype=torch.long)
                ks, vs = torch.cat([pk[blk].double(), ks]), torch.cat([pv[blk].double(), vs])
            for h in range(H):
                s = ks[:, h // (H // G)] @ q[t, h].double() * scale
                m = s.max() if snk is None else torch.maximum(s.max(), snk[h].double())
                p = (s - m).exp()
                p = p / (p.sum() + (0.0 if snk is None else (snk[h].double() - m).exp()))
                f = torch.sigmoid(hg[t, h].double()) if gate else 1.0
                want = p @ vs[:, h // (H // G)] * f
                bound = 1.5 * u * (p @ vs[:, h // (H // G)].abs() * f + want.abs()) + 1e-6
                err = (out[t, h].double() - want).abs()
                assert bool((err <= bound).all()), (b, i, h, (err / bound).max().item())

    # prefill: runs of consecutive tokens, as long as one workgroup takes them and shorter
    run = ops.window_attention_block_tokens(H, G, d, dv, dt)
    req, pos, blocks = [], [], []
    for b, n in enumerate(lens):
        start = 0 if n < 100 else n - 70
        for s in range(start, n, run):
            blocks.append((len(req), min(run, n - s)))
            req += [b] * min(run, n - s)
            pos += range(s, min(s + run, n))
    check(req, pos, torch.tensor(blocks, dtype=torch.int32, device=DEV), run, 1)
    # decode: one token each, its keys in ranges
    check(list(range(len(lens))), [n - 1 for n in lens], None, 1, splits)
