"""Triangles of every size against the oracle, bit for bit: boxes of a few 8x8
tiles, of a few bins, and of more than 32 bins (listed and emitted by whole
work-groups), needles that go to every bin of their clamped boxes, bins whose
keys hold no tile mask, and fragment queues that fill on one pixel, under each
stencil mode and blend.  sr_draw bins draws of few triangles directly,
sr_draw_static (and the batch) sorts their pairs: both are drawn."""
import numpy as np
import pytest

import scenes
import softrender_hip as sr
from parity import assert_parity, render_gpu, render_ref

pytestmark = pytest.mark.gpu

W, H = 701, 523  # 374 bins, partial bins and tiles on both edges
MODES = {
    "over": {},
    "replace": dict(blend=0),
    "count": dict(stencil_test=0, stencil_op=4, stencil_wrap=0),
    "gate": dict(stencil_test=6, stencil_op=0, stencil_ref=1),
}


def soup(n, width, height, size, seed, needle=False):
    """`n` triangles of about `size` pixels (needles: that long, a thousandth of a pixel wide)."""
    rng = np.random.default_rng(seed)
    c = rng.uniform(-0.1, 1.1, (n, 1, 2)) * (width, height)
    if needle:
        d = rng.normal(size=(n, 1, 2))
        d /= np.linalg.norm(d, axis=2, keepdims=True)
        p = c + rng.uniform(-size, size, (n, 3, 1)) * d + 1e-3 * rng.normal(size=(n, 3, 2))
    else:
        p = c + rng.normal(size=(n, 3, 2)) * size
    s = scenes.soup_scene(n, width, height, seed=seed)
    s["px"] = (p[..., 0] * (2.0 / width) - 1.0).reshape(-1).astype(np.float32)
    s["py"] = (1.0 - p[..., 1] * (2.0 / height)).reshape(-1).astype(np.float32)
    return s


def masked(s, w, h, seed):
    """The scene behind a mask: a few large flat triangles set the stencil to 1 first."""
    m = soup(12, w, h, 120.0, seed)
    fs = np.zeros(32, np.float32)
    fs[3] = 1.0
    m["desc"] = dict(m["desc"], fragment_program=0, fs_uniforms=fs, blend=0, stencil_test=0, stencil_op=3,
                     stencil_ref=1)
    return m


def render_static(ctx, scene):
    """render_gpu through sr_draw_static."""
    class Static:
        framebuffer, texture, mesh = ctx.framebuffer, ctx.texture, ctx.mesh
        draw = ctx.draw_static
    return render_gpu(Static, scene)


@pytest.mark.parametrize("mode", list(MODES))
@pytest.mark.parametrize("n,size", [(4000, 3.0), (600, 40.0), (60, 400.0), (1, 3000.0)])
def test_sizes(ctx, n, size, mode):
    s = soup(n, W, H, size, seed=0x51 + n)
    s["desc"] = dict(s["desc"], **MODES[mode])
    scene = dict(s, draws=[masked(s, W, H, 0x99), s]) if mode == "gate" else s
    print(f"{n} triangles of {size} px, {mode}", flush=True)
    ref, _ = render_ref(scene)
    assert_parity(render_gpu(ctx, scene), ref)
    assert_parity(render_static(ctx, scene), ref)


@pytest.mark.parametrize("exec_tile", [16, 32])
@pytest.mark.parametrize("mode", ["over", "gate"])
def test_sizes_other_tiles(ctx, exec_tile, mode):
    s = soup(300, W, H, 60.0, seed=0x77)
    s["desc"] = dict(s["desc"], exec_tile=exec_tile, **MODES[mode])
    scene = dict(s, draws=[masked(s, W, H, 0x9A), s]) if mode == "gate" else s
    ref, _ = render_ref(scene)
    assert_parity(render_gpu(ctx, scene), ref)


@pytest.mark.parametrize("mode", ["over", "count"])
def test_needles(ctx, mode):
    s = soup(300, 1500, 1100, 900.0, seed=0x13, needle=True)
    s["desc"] = dict(s["desc"], tile_w=96, tile_h=160, **MODES[mode])
    ref, _ = render_ref(s)
    assert_parity(render_gpu(ctx, s), ref)
    assert ctx.last_stats()["strip_slivers"] == 1
    assert_parity(render_static(ctx, s), ref)


@pytest.mark.parametrize("mode", ["over", "count"])
def test_bins_without_masks(ctx, mode):
    """More than 65,536 bins: the keys hold the bin alone."""
    w, h = 2_101_000, 2
    s = soup(2000, w, h, 60.0, seed=0x21)
    s["desc"] = dict(s["desc"], tile_w=4096, **MODES[mode])
    ref, _ = render_ref(s)
    assert (ref.depth > np.finfo(np.float32).min).any()
    assert_parity(render_gpu(ctx, s), ref)


@pytest.mark.parametrize("spread", [0.3, 3.0, 30.0])
def test_many_layers_on_few_pixels(ctx, spread):
    """700 triangles over one another, nearer and nearer: every one shades."""
    s = soup(700, 64, 48, spread, seed=0x31)
    s["px"] = s["px"] - s["px"].reshape(-1, 3).mean(1).repeat(3) + np.float32(0.13)
    s["py"] = s["py"] - s["py"].reshape(-1, 3).mean(1).repeat(3) + np.float32(0.21)
    s["pz"] = np.repeat(np.linspace(0.9, -0.9, 700), 3).astype(np.float32)
    ref, _ = render_ref(s)
    assert_parity(render_gpu(ctx, s), ref)


def test_batch_of_all_sizes(ctx):
    """Scenes of different sizes and triangle sizes in one batch, as drawn one by one."""
    items, alone, kept = [], [], []
    for k, (w, h, n, size) in enumerate([(701, 523, 40, 300.0), (64, 64, 130, 5.0), (1100, 40, 70, 90.0),
                                         (33, 700, 90, 40.0), (701, 523, 1, 2000.0), (256, 256, 3000, 4.0)]):
        s = soup(n, w, h, size, seed=0x41 + k, needle=k == 2)
        tex = ctx.texture(*s["texture"])
        fb, m, d = ctx.framebuffer(w, h), ctx.mesh(s), sr.make_desc(**s["desc"])
        items.append((fb, m, d, tex, 0xFF112233))
        one = ctx.framebuffer(w, h)
        one.clear(0xFF112233)
        ctx.draw(one, m, d, tex)
        alone.append(one.read())
        kept += [fb, m, tex, one]
    ctx.batch_draw(items)
    for (fb, *_), want in zip(items, alone):
        for a, b in zip(fb.read(), want):
            assert np.array_equal(a.view(np.uint8), b.view(np.uint8))
    for x in kept:
        x.free()


@pytest.mark.parametrize("n", [4096, 4097, 65_535, 65_536])
def test_chunks_and_limits_of_direct_binning(ctx, n):
    """A chunk of triangles and one more, the most that are binned directly and
    one more: over the frame, then all of them in one bin (the longest list)."""
    s = soup(n, 320, 200, 4.0, seed=n)
    ref, _ = render_ref(s)
    assert_parity(render_gpu(ctx, s), ref)
    s = soup(n, 320, 200, 1.5, seed=n + 1)
    s["px"], s["py"] = s["px"] * np.float32(0.04) - np.float32(0.9), s["py"] * np.float32(0.06) + np.float32(0.8)
    ref, _ = render_ref(s)
    assert_parity(render_gpu(ctx, s), ref)
