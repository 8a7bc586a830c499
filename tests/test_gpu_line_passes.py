"""Line plots against the oracle, bit for bit, where a pass of 256 plots holds
many of one pixel's: bundles of lines through few pixels, from one plot a tile
to many passes, both walks, both blends, depths nearer and farther in turn, a
stencil that counts plots the depth test drops, and lines on the frame's edge,
whose walks drop or wrap plots."""
import numpy as np
import pytest

from parity import assert_parity, render_gpu, render_ref
from test_gpu_lines_points import line_scene

pytestmark = pytest.mark.gpu


def bundle(n, w, h, p0, p1, spread, seed, **desc):
    """`n` lines from about p0 to about p1 (pixels)."""
    rng = np.random.default_rng(seed)
    s = line_scene(n, w, h, seed, **desc)
    p = np.stack([np.tile(p0, (n, 1)), np.tile(p1, (n, 1))], 1) + rng.normal(size=(n, 2, 2)) * spread
    s["px"] = (p[..., 0] * (2.0 / w) - 1.0).reshape(-1).astype(np.float32)
    s["py"] = (1.0 - p[..., 1] * (2.0 / h)).reshape(-1).astype(np.float32)
    return s


@pytest.mark.parametrize("aa", [0, 1])
@pytest.mark.parametrize("mode", [dict(blend=1), dict(blend=0), dict(blend=1, stencil_test=0, stencil_op=4),
                                  dict(blend=1, stencil_test=2, stencil_op=5, stencil_ref=3, stencil_wrap=1)])
@pytest.mark.parametrize("n,spread", [(1, 0.0), (16, 0.2), (40, 1.0), (600, 3.0)])
def test_bundles(ctx, n, spread, mode, aa):
    for p0, p1 in [((5.0, 5.0), (61.0, 20.0)), ((40.0, 58.0), (37.0, 3.0)), ((20.0, 20.0), (20.0, 20.0)),
                   ((1.0, 64.0), (68.0, 64.5)), ((0.4, 1.0), (0.6, 63.0)), ((68.5, 2.0), (69.0, 63.0)),
                   ((16.0, 2.0), (16.0, 61.0)), ((-9.0, 31.9), (90.0, 32.1))]:
        s = bundle(n, 70, 66, p0, p1, spread, seed=n, aa=aa, tile=(32, 50), **mode)
        ref, _ = render_ref(s)
        assert_parity(render_gpu(ctx, s), ref)


@pytest.mark.parametrize("aa", [0, 1])
def test_tiles_of_every_size(ctx, aa):
    """Screen tiles smaller and larger than the 16-pixel tiles, off their grid."""
    for tile in [(7, 9), (16, 16), (33, 500), (500, 500)]:
        s = line_scene(400, 257, 190, seed=tile[0], aa=aa, tile=tile)
        ref, _ = render_ref(s)
        assert_parity(render_gpu(ctx, s), ref)
