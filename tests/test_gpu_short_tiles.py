"""The decode step at head size 64, whose bfloat16 tiles are 64 tokens: contexts and windows that end on
either side of a tile, in blocks of a whole tile and more, a half, a quarter and an eighth of one."""

import pytest
import test_gpu_fused_step as step

pytestmark = pytest.mark.gpu
_pkg = step._pkg


@pytest.mark.parametrize("bs", [8, 16, 32, 64, 128])
@pytest.mark.parametrize("window,sink,small_grid", [(0, False, False), (0, False, True), (64, True, False), (65, False, True)])
def test_tile_edges(monkeypatch, bs, window, sink, small_grid):
    ctx = [0, 62, 63, 64, 65, 127, 128, 129, 700]
    step.test_fused_step_equals_update_then_decode(monkeypatch, len(ctx), 16, 2, 64, bs, ctx, False, window, sink, small_grid)
