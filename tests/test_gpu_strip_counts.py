"""Stencil visits outside the triangles' boxes against the oracle, value for
value: boxes inside one screen tile, over several, outside the frame, one tile
in all, tiles off the frame's edges, and so many tiles that the corner counters
don't fit a work-group.  sr_draw_static counts without the shared arrays."""
import pytest

from parity import assert_parity, render_gpu, render_ref
from test_gpu_wide_bins import render_static, soup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", [(128, 128), (701, 523), (700, 522), (33, 17), (350, 9), (7, 6)])
@pytest.mark.parametrize("n,size", [(3000, 4.0), (300, 60.0), (1, 2.0), (40, 500.0)])
def test_counts(ctx, n, size, tile):
    s = soup(n, 701, 523, size, seed=0x61 + n)
    s["desc"] = dict(s["desc"], tile_w=tile[0], tile_h=tile[1], stencil_test=0, stencil_op=4, stencil_wrap=1)
    print(f"{n} triangles of {size} px, tiles {tile}", flush=True)
    ref, _ = render_ref(s)
    assert (ref.stencil != 0).any()
    assert_parity(render_gpu(ctx, s), ref)
    assert_parity(render_static(ctx, s), ref)


@pytest.mark.parametrize("w,h", [(2, 2), (3, 300), (257, 2), (129, 129)])
def test_small_frames(ctx, w, h):
    s = soup(200, w, h, 30.0, seed=0x62)
    s["desc"] = dict(s["desc"], stencil_test=0, stencil_op=4, stencil_wrap=1)
    ref, _ = render_ref(s)
    assert_parity(render_gpu(ctx, s), ref)
