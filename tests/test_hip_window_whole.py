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
