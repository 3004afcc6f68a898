"""Window attention over tiles that every row of a run sees whole (no masks there), behind ones that the window's or the triangle's edge
crosses, at the widths whose loops are laid out in full: the bound of the other widths' rows."""
import pytest
import torch
from test_hip_window_rows import test_rows_against_float64 as rows_against_float64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,H,G,d,window,pool,sink,gate,splits", [
    (torch.bfloat16, 8, 2, 128, 90, 0, True, True, 1),      # whole tiles inside the window
    (torch.float16, 4, 4, 64, 0, 0, False, False, 3),       # no window: whole from position 31 on
    (torch.bfloat16, 4, 1, 128, 10, 4, False, True, 2),     # a whole tile of averaged blocks
    (torch.float16, 4, 2, 64, 64, 2, True, False, 1),       # both
])
def test_whole_tiles(dt, H, G, d, window, pool, sink, gate, splits):
    rows_against_float64(dt, H, G, d, d, window, pool, sink, gate, 0, splits)


@pytest.mark.parametrize("dt,H,G,d,dv,window,pool,sink", [
    (torch.bfloat16, 16, 4, 128, 128, 150, 8, False),
    (torch.float16, 8, 8, 64, 64, 0, 0, True),
    (torch.float16, 8, 2, 96, 80, 170, 0, False),
])
def test_a_row_does_not_depend_on_its_block(dt, H, G, d, dv, window, pool, sink):
    """The same tokens in blocks of every length: whether a tile is whole depends on a block's first and last row, the bits do not.
    (Rows enough for a score that is rounded in one form and not in the other to show in some of the results.)"""
    from sglang_custom_amd import ops

    g = torch.Generator().manual_seed(d + window)
    n, step, DEV = 1200, max(pool, 1), "cuda"
    table = torch.arange(step, step + n, dtype=torch.int32).view(1, n).to(DEV)
    k, v, q = (torch.randn(n + 2 * step, h, w, generator=g).to(dt).to(DEV) for h, w in ((G, d), (G, dv), (H, d)))
    q = q[:n]
    pk, pv = ((torch.randn(n // step + 3, G, w, generator=g).to(dt).to(DEV) for w in (d, dv)) if pool else (None, None))
    snk = torch.randn(H, generator=g).to(DEV) if sink else None
    longest = ops.window_attention_block_tokens(H, G, d, dv, dt)
    outs = []
    for run in sorted({1, 2, max(longest // 2, 1), longest}):
        blocks = torch.tensor([(s, min(run, n - s)) for s in range(0, n, run)], dtype=torch.int32, device=DEV)
        out = torch.full((n, H, dv), float("nan"), dtype=dt, device=DEV)
        ops.window_attention(q, k, v, out, table, torch.zeros(1, dtype=torch.long, device=DEV), torch.arange(n, device=DEV), snk, window, 0.23,
                             tok_req=torch.zeros(n, dtype=torch.int32, device=DEV), blocks=blocks, max_run=run, num_splits=1, pool=pool,
                             pooled_k=pk, pooled_v=pv, pool_div=step)
        outs.append(out)
    assert len(outs) > 1 and all(torch.equal(outs[0], o) for o in outs[1:])
