"""Large frames whose bins hold few triangles: the bins' ends then say which
tiles have one.  Bins of none, one, sixteen, seventeen and many triangles, binned
directly, sorted (sr_draw_static) and in a batch, against the oracle bit for bit."""
import numpy as np
import pytest

import softrender_hip as sr
from parity import assert_parity, render_gpu, render_ref
from test_formats import F32, _gpu, _oracle, _same
from test_gpu_wide_bins import MODES, masked, render_static, soup

pytestmark = pytest.mark.gpu

W, H = 2100, 1000  # 66 x 32 bins


def sparse(seed, needle=False):
    """Bins of 0 to 20 small triangles in turn, and a few triangles over many bins."""
    rng = np.random.default_rng(seed)
    c = []
    for k, b in enumerate(rng.permutation(66 * 32)[:600]):
        n = [1, 2, 15, 16, 17, 20][k % 6]
        c.append(np.array([b % 66, b // 66]) * 32.0 + rng.uniform(4.0, 28.0, (n, 1, 2)))
    p = np.concatenate(c) + rng.normal(size=(sum(map(len, c)), 3, 2)) * 1.5
    big = soup(12, W, H, 150.0, seed, needle)
    s = soup(len(p) + 12, W, H, 1.0, seed)
    s["px"] = np.concatenate([(p[..., 0] * (2.0 / W) - 1.0).reshape(-1).astype(np.float32), big["px"]])
    s["py"] = np.concatenate([(1.0 - p[..., 1] * (2.0 / H)).reshape(-1).astype(np.float32), big["py"]])
    return s


@pytest.mark.parametrize("exec_tile", [0, 16, 32])
@pytest.mark.parametrize("mode", list(MODES))
def test_sparse_frames(ctx, mode, exec_tile):
    s = sparse(0x61, needle=mode == "over")
    s["desc"] = dict(s["desc"], exec_tile=exec_tile, **MODES[mode])
    scene = dict(s, draws=[masked(s, W, H, 0x99), s]) if mode == "gate" else s
    ref, _ = render_ref(scene)
    assert_parity(render_gpu(ctx, scene), ref)
    n = ctx.last_stats()["bin_pairs"]
    assert_parity(render_static(ctx, scene), ref)
    assert 0 < n <= ctx.last_stats()["bin_pairs"]  # (a sorted pair may have no tile of its bin)


def test_sparse_float_planes(ctx):
    s = sparse(0x62)
    for blend in (0, 2):
        s["desc"] = dict(s["desc"], blend=blend)
        tex = ctx.texture(*s["texture"])
        ref, _ = _oracle(s, [F32], depth=sr.DEPTH_F64, colors=[[0.1, 0.2, 0.3, 0.5]], tex=s["texture"])
        fb, got = _gpu(ctx, s, [F32], depth=sr.DEPTH_F64, colors=[[0.1, 0.2, 0.3, 0.5]], tex=tex)
        _same(got, ref)
        fb.free()
        tex.free()


def test_sparse_batch(ctx):
    """Frames of few and of many triangles a bin in one batch."""
    scenes = [sparse(0x63), soup(3, 64, 64, 9.0, seed=1), soup(2000, 300, 200, 4.0, seed=2)]
    items, kept, refs = [], [], []
    for s in scenes:
        fb, m, tex, d = ctx.framebuffer(s["width"], s["height"]), ctx.mesh(s), ctx.texture(*s["texture"]), sr.make_desc(**s["desc"])
        items.append((fb, m, d, tex, 0xFF112233))
        refs.append(render_ref(dict(s, clear=0xFF112233))[0])
        kept += [m, tex]
    ctx.batch_draw(items)
    for (fb, *_), ref in zip(items, refs):
        assert_parity(fb.read(), ref)
        fb.free()
    for x in kept:
        x.free()
