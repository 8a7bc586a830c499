"""sr_draw_stats.bin_pairs of draws that are binned directly: the entries of the
draw's bins, as sr_draw_static (whose pairs are sorted) counts them."""
import numpy as np
import pytest

import softrender_hip as sr
from parity import render_gpu
from test_gpu_wide_bins import render_static, soup

pytestmark = pytest.mark.gpu

W, H = 640, 480


def at_pixels(p, **desc):
    """A scene of the triangles p [n, 3, 2], in pixels."""
    s = soup(len(p), W, H, 1.0, seed=5)
    s["px"] = (p[..., 0] * (2.0 / W) - 1.0).reshape(-1).astype(np.float32)
    s["py"] = (1.0 - p[..., 1] * (2.0 / H)).reshape(-1).astype(np.float32)
    s["desc"] = dict(s["desc"], **desc)
    return s


def tiny(n, seed):
    """`n` triangles, each inside one 8x8 tile."""
    rng = np.random.default_rng(seed)
    t = rng.integers(0, [W // 8, H // 8], (n, 1, 2)) * 8.0
    return t + np.array([[1.2, 1.1], [6.7, 2.3], [3.4, 6.6]])


def pairs(ctx, scene, static=False):
    (render_static if static else render_gpu)(ctx, scene)
    return ctx.last_stats()["bin_pairs"]


@pytest.mark.parametrize("gs", [0, 1, 2])
def test_one_entry_a_tiny_triangle(ctx, gs):
    s = at_pixels(tiny(900, 1), geometry_program=gs)
    s["pz"] = np.full_like(s["pz"], 0.5)  # inside every plane
    for static in (False, True):
        # (the clip program emits each triangle, and degenerate ones that cover nothing)
        assert pairs(ctx, s, static) == 900, static
        assert ctx.last_stats()["generated_tris"] >= (900 if gs else 0)


def test_boxes_where_visits_count(ctx):
    """A stencil that counts visits: every bin of every box."""
    rng = np.random.default_rng(2)
    p = rng.integers(1, [W - 1, H - 1], (300, 3, 2)) + rng.choice([0.25, 0.75], (300, 3, 2))
    p = p[[abs(np.linalg.det(t[1:] - t[0])) > 2000.0 for t in p]]  # (a sliver's pixels may lie outside its box)
    want = sum(int(np.prod((t.max(0).astype(int) >> 5) - (t.min(0).astype(int) >> 5) + 1)) for t in p)
    s = at_pixels(p, stencil_test=0, stencil_op=4, stencil_wrap=0)
    assert (pairs(ctx, s), pairs(ctx, s, True)) == (want, want)


def test_bins_the_triangles_meet(ctx):
    """Diagonal strips: far fewer bins than their boxes hold; asked for twice, after a clear and another draw."""
    x = np.linspace(-40.0, 40.0, 9)[:, None, None]
    p = np.array([[5.0, 5.0], [W - 9.0, H - 6.0], [W - 9.0, H - 30.0]]) + x * [1.0, 0.0]
    s = at_pixels(p)
    n = pairs(ctx, s)
    boxes = sum(int(np.prod((np.minimum(t.max(0), [W - 1, H - 1]).astype(int) >> 5) -
                            (np.maximum(t.min(0), 0).astype(int) >> 5) + 1)) for t in p)
    # bins that hold a pixel centre inside, and those that hold one within two pixels
    gx, gy = np.meshgrid(np.arange(W) + 0.5, np.arange(H) + 0.5)
    least = most = 0
    for a, b, c in p:
        d = []
        for q, r in ((a, b), (b, c), (c, a)):
            e = r - q
            d.append(((gx - q[0]) * e[1] - (gy - q[1]) * e[0]) / np.hypot(*e))
        d = np.array(d)
        d = d if (d.min(0) > 0).any() else -d
        bins = [len(set(zip((gx[m].astype(int) >> 5).tolist(), (gy[m].astype(int) >> 5).tolist())))
                for m in (d.min(0) > 0.0, d.min(0) > -2.0)]
        least, most = least + bins[0], most + bins[1]
    assert 0 < least <= n <= most < boxes, (least, n, most, boxes)
    assert ctx.last_stats()["bin_pairs"] == n
    static = pairs(ctx, s, True)
    assert n <= static < boxes
    fb = ctx.framebuffer(W, H)
    fb.clear(0)
    m = ctx.mesh(s)
    ctx.draw(fb, m, sr.make_desc(**s["desc"]), ctx.texture(*s["texture"]))
    fb.clear(0)
    assert ctx.last_stats()["bin_pairs"] == n
    m.free()
    fb.free()
