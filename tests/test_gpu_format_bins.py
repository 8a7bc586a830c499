"""The binned raster of the framebuffer formats against the oracle, bit for
bit: lists of no, one and many steps, fragments that fill the shading queue,
needles, few blended triangles (drawn one by one) and one more, every blend,
one plane and four, f32 and f64 depth, and an RGBAF32 texture under every edge
rule."""
import numpy as np
import pytest

import oracle
import scenes
import softrender_hip as sr
from test_formats import F32, RGBA8, _gpu, _oracle, _same, gbuffer_uniforms
from test_gpu_wide_bins import soup

pytestmark = pytest.mark.gpu

ONE, FOUR = ([F32], [[0.1, 0.2, 0.3, 0.5]]), ([RGBA8, F32, F32, RGBA8],
                                              [0xFF202020, [0.1, 0.2, 0.3, 0.5], [0.0, 0.0, 0.0, 1.0], 0x80FFFFFF])


@pytest.mark.parametrize("blend", [0, 1, 2])
@pytest.mark.parametrize("n,size,needle", [(1, 900.0, False), (16, 300.0, False), (17, 300.0, False),
                                           (6000, 4.0, False), (700, 60.0, False), (150, 400.0, True)])
def test_soups(ctx, n, size, needle, blend):
    s = soup(n, 333, 190, size, seed=n, needle=needle)
    s["pz"] = np.sort(s["pz"].reshape(-1, 3)[:, 0])[::-1].repeat(3).astype(np.float32)  # nearer and nearer
    tex = ctx.texture(*s["texture"])
    for (planes, colors), depth, fp in [(ONE, sr.DEPTH_F64, sr.FP_TEX_LAMBERT), (FOUR, 0, sr.FP_GBUFFER),
                                        (FOUR, sr.DEPTH_F64, sr.FP_UV_COLOR)]:
        s["desc"] = dict(s["desc"], fragment_program=fp, blend=blend, fs_uniforms=gbuffer_uniforms(0.6))
        ref, _ = _oracle(s, planes, depth=depth, colors=colors, tex=s["texture"])
        fb, got = _gpu(ctx, s, planes, depth=depth, colors=colors, tex=tex)
        fb.free()
        _same(got, ref)
    tex.free()


@pytest.mark.parametrize("edge", [0, 1, 2])
@pytest.mark.parametrize("filt", [0, 1])
def test_rgbaf32_texture(ctx, filt, edge):
    """A texture-buffer plane sampled inside and outside [0, 1]."""
    s = scenes.soup_scene(3000, 160, 100, seed=5)
    s["desc"] = dict(s["desc"], fragment_program=sr.FP_GBUFFER, blend=0, fs_uniforms=gbuffer_uniforms())
    planes, colors = FOUR
    ref, _ = _oracle(s, planes, colors=colors, tex=s["texture"])
    tex = ctx.texture(*s["texture"])
    gb, _ = _gpu(ctx, s, planes, colors=colors, tex=tex)
    s2 = soup(400, 160, 100, 20.0, seed=6)
    s2["u"], s2["v"] = (s2["u"] * np.float32(3.0) - np.float32(1.0), s2["v"] * np.float32(3.0) - np.float32(1.0))
    s2["desc"] = dict(s2["desc"], fragment_program=sr.FP_TEX_LAMBERT, blend=1, tex_filter=filt, tex_edge=edge,
                      tex_border=0x80FF4020, fs_uniforms=gbuffer_uniforms(0.6))
    want, _ = _oracle(s2, [RGBA8], colors=[0xFF000000], tex=oracle.plane_texture(ref, 1))
    plane = ctx.texture_from_fb_plane(gb, 1)
    fb, got = _gpu(ctx, s2, [RGBA8], colors=[0xFF000000], tex=plane)
    _same(got, want)
    for x in (plane, tex, gb, fb):
        x.free()
