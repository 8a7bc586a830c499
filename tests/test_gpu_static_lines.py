"""Short lines in the fixed workspace of sr_draw_static: as many as their
records (80 bytes and, anti-aliased, four plots of 24) leave room for."""
import numpy as np
import pytest

from parity import assert_parity, render_ref
from test_gpu_lines_points import line_scene
from test_gpu_wide_bins import render_static

pytestmark = pytest.mark.gpu


def short_lines(n, aa):
    """Lines inside one pixel: two coordinates and five varyings a vertex, an item, its plots, a tile or two."""
    s = line_scene(n, 512, 512, seed=n, aa=aa)
    rng = np.random.default_rng(n)
    p = rng.integers(2, 510, (n, 1, 2)) + rng.uniform(0.1, 0.4, (n, 1, 2)) + np.array([[0.0, 0.0], [0.3, 0.2]])
    s["px"] = (p[..., 0] * (2.0 / 512) - 1.0).reshape(-1).astype(np.float32)
    s["py"] = (1.0 - p[..., 1] * (2.0 / 512)).reshape(-1).astype(np.float32)
    return s


@pytest.mark.parametrize("n,aa", [(210_000, 1), (300_000, 0)])
def test_short_lines_fit(ctx, n, aa):
    s = short_lines(n, aa)
    print(f"{n} short lines, aa {aa}", flush=True)
    ref, _ = render_ref(s)
    assert_parity(render_static(ctx, s), ref)
