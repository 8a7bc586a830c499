"""The frames that programs built on this renderer draw, as measured cases.

Every case is one pass of such a program through softrender_hip (the binding
of the C ABI): clear, one or more draws, and the read-back of the finished
planes into pinned host memory, which is how a renderer hands a frame on.
Meshes, textures, framebuffers and pinned buffers are what a program keeps
between frames; one context (and one server) serves the whole process.

Sizes follow the repository's own workloads (512x512 sphere, 1080p frame of
1M triangles, 4K frame of clipped triangles, lines and points, batches and
served requests of 1k to 1M triangles at 256x256 to 1080p, the full example's
Fresnel frame and normal lines) and generic screen sizes, odd ones included.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "rust-softrender_amd"))
import softrender_hip as sr  # noqa: E402

F32 = np.float32
BACK = 0xFF000000


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # an icon or thumbnail of a low-poly mesh: launches and waits are everything
        dict(name="icon_64", kind="mesh", w=64, h=64, stacks=8, slices=12),
        # the sphere frame: a small mesh in a viewer, colour and depth read back
        dict(name="sphere_512", kind="mesh", w=512, h=512, stacks=32, slices=64),
        # the headline frame: a million small textured translucent triangles at 1080p
        dict(name="soup_1080p", kind="soup", w=1920, h=1080, tris=1_000_000, area=20.0, blend=1, filter=1, edge=0),
        # few large translucent triangles in many layers (particles, foliage cards) on a
        # laptop screen whose size no tile divides
        dict(name="layers_1366x768", kind="soup", w=1366, h=768, tris=20_000, area=2500.0, blend=1, filter=1, edge=1),
        # a terrain seen from the air at 4K: an indexed mesh, lit, culled, opaque; the most triangles
        dict(name="terrain_4k", kind="terrain", w=3840, h=2160, grid=1024),
        # the 4K frame of near-clipped triangles, anti-aliased lines and points with stencil counting
        dict(name="clip_4k", kind="clip", w=3840, h=2160, tris=500_000, lines=200_000, points=100_000, aa=1),
        # the full example's frame: four lights, Fresnel, tone mapping, RGBA float colour
        dict(name="example_720p", kind="example", w=1280, h=720, stacks=50, slices=100),
        # the full example's debug view: the lit model and its face normals as lines from one vertex pass
        dict(name="normals_720p", kind="normals", w=1280, h=720, stacks=100, slices=200),
        # deferred shading: a four-plane texture buffer, then a full-screen pass that samples it
        dict(name="deferred_900p", kind="deferred", w=1600, h=900, tris=60_000, area=80.0),
        # a scene seen through a stencil mask (mirror, portal, user interface clip region)
        dict(name="mask_1080p", kind="mask", w=1920, h=1080, tris=100_000, area=60.0),
        # many independent scenes rendered as one batch (data generation, previews)
        dict(name="batch_32", kind="batch", scenes=32, lo=1_000, hi=300_000),
        # a burst of requests at the rendering server over its resident meshes
        dict(name="serve_24", kind="serve", requests=24, meshes=8, lo=1_000, hi=300_000),
    ]


def _logu(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _screen(rng, lo, hi):
    """A screen of about lo to hi pixels in width, of a usual shape, odd sizes among them."""
    w = int(round(_logu(rng, lo, hi)))
    h = max(16, int(round(w * rng.choice([1.0, 9 / 16, 10 / 16, 3 / 4]))))
    return w, h


def draw(rng):
    kind = rng.choice(["mesh", "mesh", "soup", "soup", "terrain", "clip", "example", "normals", "deferred", "mask",
                       "batch", "serve"])
    if kind == "mesh":
        w, h = _screen(rng, 48, 1920)
        stacks = int(round(_logu(rng, 6, 120)))
        return dict(kind=kind, w=w, h=h, stacks=stacks, slices=2 * stacks + rng.randrange(2))
    if kind == "soup":
        w, h = _screen(rng, 200, 2560)
        area = _logu(rng, 6.0, 3000.0)
        most = min(1_000_000.0, 4.5e7 / area)
        return dict(kind=kind, w=w, h=h, tris=int(round(_logu(rng, 500, most))), area=area, blend=rng.randrange(2),
                    filter=rng.randrange(2), edge=rng.randrange(3))
    if kind == "terrain":
        w, h = _screen(rng, 400, 3840)
        return dict(kind=kind, w=w, h=h, grid=int(round(_logu(rng, 40, 1000))))
    if kind == "clip":
        w, h = _screen(rng, 400, 3840)
        return dict(kind=kind, w=w, h=h, tris=int(round(_logu(rng, 1000, 400_000))),
                    lines=int(round(_logu(rng, 500, 150_000))), points=int(round(_logu(rng, 500, 100_000))),
                    aa=rng.randrange(2))
    if kind in ("example", "normals"):
        w, h = _screen(rng, 160, 1600)
        stacks = int(round(_logu(rng, 12, 90)))
        return dict(kind=kind, w=w, h=h, stacks=stacks, slices=2 * stacks + rng.randrange(2))
    if kind == "deferred":
        w, h = _screen(rng, 200, 1920)
        return dict(kind=kind, w=w, h=h, tris=int(round(_logu(rng, 500, 60_000))), area=_logu(rng, 20.0, 150.0))
    if kind == "mask":
        w, h = _screen(rng, 200, 1920)
        return dict(kind=kind, w=w, h=h, tris=int(round(_logu(rng, 500, 100_000))), area=_logu(rng, 15.0, 150.0))
    if kind == "batch":
        return dict(kind=kind, scenes=rng.randrange(4, 33), lo=1_000, hi=int(round(_logu(rng, 5_000, 200_000))))
    return dict(kind=kind, requests=rng.randrange(4, 25), meshes=rng.randrange(2, 9), lo=1_000,
                hi=int(round(_logu(rng, 5_000, 200_000))))


# ---------------------------------------------------------------------------
# geometry and cameras (numpy, from the seed alone)
# ---------------------------------------------------------------------------
def _look_at(eye, target, up=(0.0, 1.0, 0.0)):
    eye = np.asarray(eye, np.float64)
    f = np.asarray(target, np.float64) - eye
    f /= np.linalg.norm(f)
    s = np.cross(f, np.asarray(up, np.float64))
    s /= np.linalg.norm(s)
    m = np.eye(4)
    m[0, :3], m[1, :3], m[2, :3] = s, np.cross(s, f), -f
    m[:3, 3] = -(m[:3, :3] @ eye)
    return m


def _perspective(fovy, aspect, near, far):
    """Clip z in [0, w], the near plane at 0."""
    f = 1.0 / math.tan(math.radians(fovy) / 2.0)
    p = np.zeros((4, 4))
    p[0, 0], p[1, 1] = f / aspect, f
    p[2, 2], p[2, 3], p[3, 2] = far / (near - far), near * far / (near - far), -1.0
    return p


def _rotation_y(a):
    m = np.eye(4)
    m[0, 0], m[0, 2], m[2, 0], m[2, 2] = math.cos(a), math.sin(a), -math.sin(a), math.cos(a)
    return m


def _vsu(mvp, normal3=None, model=None):
    u = np.zeros(48, F32)
    u[0:16] = np.asarray(mvp).reshape(16)
    u[16:25] = (np.eye(3) if normal3 is None else normal3).reshape(9)
    u[25:37] = (np.eye(4) if model is None else model)[:3].reshape(12)
    return u


def _viewport(w, h):
    return (0.0, 0.0, float(w), float(h), 0.0, 1.0)


def _unit(v):
    v = np.asarray(v, np.float64)
    return v / np.linalg.norm(v)


def _ball(rng, stacks, slices):
    """A bumpy UV sphere: positions, normals and a triangle list."""
    th = np.pi * np.arange(stacks + 1)[:, None] / stacks
    ph = 2.0 * np.pi * np.arange(slices + 1)[None, :] / slices
    a, b, c = rng.uniform(0.0, 2.0 * np.pi, 3)
    r = 1.0 + 0.06 * np.sin(3.0 * th + a) * np.sin(2.0 * ph + b) + 0.03 * np.cos(5.0 * th + c) + 0.0 * ph
    d = np.stack([np.sin(th) * np.cos(ph), np.cos(th) + 0.0 * ph, np.sin(th) * np.sin(ph)], -1)
    pos = (d * r[..., None]).reshape(-1, 3)
    nrm = d.reshape(-1, 3)
    row = slices + 1
    i, j = np.meshgrid(np.arange(stacks), np.arange(slices), indexing="ij")
    v00, v01, v10, v11 = i * row + j, i * row + j + 1, (i + 1) * row + j, (i + 1) * row + j + 1
    upper, lower = np.stack([v00, v10, v01], -1), np.stack([v01, v10, v11], -1)
    quads = np.stack([upper, lower], 2)
    keep = np.ones((stacks, slices, 2), bool)
    keep[0, :, 0] = False
    keep[-1, :, 1] = False
    idx = quads[keep].reshape(-1)
    return pos.astype(F32), nrm.astype(F32), idx.astype(np.uint32)


def _mesh(pos, nrm, idx, uv=None, prim=3):
    s = dict(px=pos[:, 0], py=pos[:, 1], pz=pos[:, 2], indices=idx, primitive=prim)
    if nrm is not None:
        s.update(nx=nrm[:, 0], ny=nrm[:, 1], nz=nrm[:, 2])
    if uv is not None:
        s.update(u=uv[:, 0], v=uv[:, 1])
    return s


def _cull_back(pos, idx, mvp, w, h, eye):
    """The winding of the triangles that face away from the eye (as seen on the screen)."""
    p = pos[idx].reshape(-1, 3, 3).astype(np.float64)
    t = p[np.argmin(np.linalg.norm(p.mean(1) - np.asarray(eye), axis=1))]
    c = np.c_[t, np.ones(3)] @ np.asarray(mvp).T
    x, y = (c[:, 0] / c[:, 3] + 1.0) * w / 2.0, (1.0 - c[:, 1] / c[:, 3]) * h / 2.0
    area = x[0] * y[1] + x[1] * y[2] + x[2] * y[0] - x[1] * y[0] - x[2] * y[1] - x[0] * y[2]
    return 2 if area < 0 else 1


def _soup(rng, n, w, h, area, z=(-0.99, 0.99)):
    """Equilateral triangles all over the screen in clip space, their areas
    log-normal (sigma 1) about `area` pixels, random normals and uv."""
    cx, cy = rng.uniform(-1.0, 1.0, n), rng.uniform(-1.0, 1.0, n)
    r = np.sqrt(4.0 / math.sqrt(3.0) * area * np.exp(rng.standard_normal(n))) / math.sqrt(3.0)
    t = rng.uniform(0.0, 2.0 * np.pi, n)
    p = np.empty((n, 3, 3), F32)
    for k in range(3):
        p[:, k, 0] = cx + r * np.cos(t + k * 2.0 * np.pi / 3.0) * (2.0 / w)
        p[:, k, 1] = cy + r * np.sin(t + k * 2.0 * np.pi / 3.0) * (2.0 / h)
    p[:, :, 2] = rng.uniform(z[0], z[1], n)[:, None]
    nrm = rng.random((3 * n, 3), F32) * F32(2) - F32(1)
    return p.reshape(-1, 3), nrm, rng.random((3 * n, 2), F32)


def _cloud(rng, n):
    """Triangles scattered in a unit ball, for a camera that goes round it."""
    c = rng.standard_normal((n, 3), F32)
    c *= (0.8 * np.cbrt(rng.random(n)) / np.maximum(np.linalg.norm(c, axis=1), 1e-9))[:, None].astype(F32)
    size = (0.02 * np.exp(0.5 * rng.standard_normal(n)) * math.sqrt(1e4 / max(n, 1e4))).astype(F32)
    p = c[:, None, :] + size[:, None, None] * rng.standard_normal((n, 3, 3), F32)
    return p.reshape(-1, 3), rng.random((3 * n, 3), F32) * F32(2) - F32(1), rng.random((3 * n, 2), F32)


def _orbit(rng, w, h):
    az, el, d = rng.uniform(0.0, 2.0 * np.pi), rng.uniform(-np.pi / 3, np.pi / 3), rng.uniform(2.0, 4.0)
    eye = (d * math.cos(el) * math.cos(az), d * math.sin(el), d * math.cos(el) * math.sin(az))
    return _perspective(60.0, w / h, 0.1, 100.0) @ _look_at(eye, (0.0, 0.0, 0.0))


def _checker(rng, size=1024, square=32):
    """A two-colour checkerboard with its colours from the seed."""
    y, x = np.mgrid[0:size, 0:size]
    c = rng.integers(0, 1 << 24, 2, dtype=np.uint32) | np.uint32(BACK)
    return c[(x // square + y // square) % 2].reshape(-1)


def _tex_lambert(alpha=0.8):
    fs = np.zeros(32, F32)
    fs[0:3] = _unit((0.3, 0.5, 0.8))
    fs[3:6] = (0.2, 0.8, alpha)
    return fs


def _blinn_phong(eye):
    fs = np.zeros(32, F32)
    fs[0:3], fs[3:6], fs[6:9], fs[9:13] = _unit((1, 1, 1)), eye, (0.8, 0.3, 0.2), (0.1, 0.8, 0.5, 1.0)
    return fs


LIGHTS = ((-1.0, 1.0, -1.0, 1.0, 1.0, 1.0, 9.0), (1.0, 1.0, 1.0, 0.6, 0.6, 1.0, 9.0),
          (0.0, 3.0, -1.0, 1.0, 0.3, 0.3, 25.0), (-2.0, -1.0, 1.0, 0.7, 1.0, 0.7, 25.0))


# ---------------------------------------------------------------------------
# what a program keeps
# ---------------------------------------------------------------------------
_ctx = None
_server = None


def _context():
    global _ctx
    if _ctx is None:
        _ctx = sr.Context(0)
    return _ctx


def _the_server():
    global _server
    if _server is None:
        _server = sr.Server(_context())
    return _server


class State:
    """The handles of one case, given back when the state goes."""

    def __init__(self, kind):
        self.kind = kind
        self.ctx = _context()
        self.kept = []
        self.held = []

    def keep(self, handle):
        self.kept.append(handle)
        return handle

    def mesh(self, s):
        return self.keep(self.ctx.mesh(s))

    def texture(self, rng):
        return self.keep(self.ctx.texture(1024, 1024, _checker(rng)))

    def fb(self, w, h):
        return self.keep(self.ctx.framebuffer(w, h))

    def host(self, n, dtype=torch.int32):
        return torch.empty(n, dtype=dtype, pin_memory=True)

    def release_held(self):
        for t in self.held:
            sr.lib().sr_server_release(_the_server().h, t)
        self.held = []

    def __del__(self):
        try:
            self.release_held()
            for x in reversed(self.kept):
                x.free()
        except Exception:
            pass


def _ptr(t, kind):
    return ctypes.cast(t.data_ptr(), ctypes.POINTER(kind))


def _read(fb, color, depth=None, stencil=None):
    """The planes that are wanted, into pinned memory, in one call."""
    rc = sr.lib().sr_fb_read(fb.h, _ptr(color, ctypes.c_uint32), None if depth is None else _ptr(depth, ctypes.c_float),
                             None if stencil is None else _ptr(stencil, ctypes.c_uint8))
    if rc != sr.SR_OK:
        raise sr.SoftrenderError(rc, "sr_fb_read")


def _batch_specs(rng, case):
    """(triangles, width, height) of each scene: counts log-uniform, three resolutions."""
    n = case["scenes"]
    t = np.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]), n)).round().astype(int)
    sizes = [(256, 256), (512, 512), (1920, 1080)]
    return [(int(t[i]), *sizes[i % 3]) for i in range(n)]


def _example_scene(case, seed):
    """The full example's camera, model and lights about a bumpy ball."""
    rng = np.random.default_rng(seed)
    w, h = case["w"], case["h"]
    pos, nrm, idx = _ball(rng, case["stacks"], case["slices"])
    model = _rotation_y(rng.uniform(0.0, 2.0 * np.pi))
    model[:3, :3] *= 0.7
    model[:3, 3] = (0.0, 0.25, 0.0)
    mit = np.linalg.inv(model).T
    cam = np.array([math.cos(math.radians(75.0)) * 2.0, 2.0, math.sin(math.radians(75.0)) * 2.0])
    pv = _perspective(65.0, w / h, 0.1, 1000.0) @ _look_at(cam, (0.0, 0.25, 0.0))
    return pos, nrm, idx, model, mit, cam, pv


def prepare(case, seed):
    kind = case["kind"]
    st = State(kind)
    rng = np.random.default_rng(seed)
    w, h = case.get("w"), case.get("h")
    if kind == "mesh":
        pos, nrm, idx = _ball(rng, case["stacks"], case["slices"])
        eye = (0.0, 0.0, 3.0)
        mvp = _perspective(60.0, w / h, 0.1, 100.0) @ _look_at(eye, (0.0, 0.0, 0.0))
        st.fbo, st.m = st.fb(w, h), st.mesh(_mesh(pos, nrm, idx))
        st.desc = sr.make_desc(vertex_program=sr.VP_MVP_NORMAL_WORLD, fragment_program=sr.FP_BLINN_PHONG,
                               cull=_cull_back(pos, idx, mvp, w, h, eye), vs_uniforms=_vsu(mvp),
                               fs_uniforms=_blinn_phong(eye), viewport=_viewport(w, h))
        st.color, st.depth = st.host(w * h), st.host(w * h, torch.float32)
    elif kind == "soup":
        pos, nrm, uv = _soup(rng, case["tris"], w, h, case["area"])
        st.fbo, st.m, st.tex = st.fb(w, h), st.mesh(_mesh(pos, nrm, None, uv)), st.texture(rng)
        st.desc = sr.make_desc(vertex_program=sr.VP_MVP_NORMAL_UV, fragment_program=sr.FP_TEX_LAMBERT,
                               blend=case["blend"], tex_filter=case["filter"], tex_edge=case["edge"],
                               tex_border=0xFF404040, vs_uniforms=_vsu(np.eye(4)), fs_uniforms=_tex_lambert(),
                               viewport=_viewport(w, h))
        st.color = st.host(w * h)
    elif kind == "terrain":
        g = case["grid"]
        t = np.linspace(-1.0, 1.0, g + 1)
        x, z = np.meshgrid(t, t, indexing="ij")
        y, dx, dz = 0.0 * x, 0.0 * x, 0.0 * x
        for f in (2.0, 5.0, 11.0, 23.0):  # rolling hills: a few waves each way
            a, b, c = rng.uniform(0.5, 1.0) * f, rng.uniform(-1.0, 1.0) * f, rng.uniform(0.0, 6.0)
            s = 0.12 / f
            y += s * np.sin(a * x + b * z + c)
            dx += s * a * np.cos(a * x + b * z + c)
            dz += s * b * np.cos(a * x + b * z + c)
        pos = np.stack([x, y, z], -1).reshape(-1, 3).astype(F32)
        nrm = np.stack([-dx, 1.0 + 0.0 * x, -dz], -1).reshape(-1, 3).astype(F32)
        i, j = np.meshgrid(np.arange(g), np.arange(g), indexing="ij")
        v00, v01, v10, v11 = i * (g + 1) + j, i * (g + 1) + j + 1, (i + 1) * (g + 1) + j, (i + 1) * (g + 1) + j + 1
        idx = np.stack([v00, v01, v10, v10, v01, v11], -1).reshape(-1).astype(np.uint32)
        az = rng.uniform(0.0, 2.0 * np.pi)
        eye = (1.3 * math.cos(az), 0.8, 1.3 * math.sin(az))
        mvp = _perspective(50.0, w / h, 0.1, 10.0) @ _look_at(eye, (0.0, -0.1, 0.0))
        st.fbo, st.m = st.fb(w, h), st.mesh(_mesh(pos, nrm, idx))
        st.desc = sr.make_desc(vertex_program=sr.VP_MVP_NORMAL_WORLD, fragment_program=sr.FP_BLINN_PHONG,
                               cull=_cull_back(pos, idx, mvp, w, h, eye), vs_uniforms=_vsu(mvp),
                               fs_uniforms=_blinn_phong(eye), viewport=_viewport(w, h))
        st.color = st.host(w * h)
    elif kind == "clip":
        n, nl, npt = case["tris"], case["lines"], case["points"]
        pos, nrm, uv = _soup(rng, n, w, h, 20.0, z=(0.01, 0.99))
        z = pos.reshape(n, 3, 3)[:, :, 2]  # 30% cross the near plane: one or two vertices behind it
        pick, first, two = rng.random(n) < 0.3, rng.integers(0, 3, n), rng.random(n) < 0.5
        behind = -rng.uniform(0.05, 0.6, n).astype(F32)
        for k in range(2):
            sel = np.nonzero(pick if k == 0 else pick & two)[0]
            z[sel, (first[sel] + k) % 3] = behind[sel]
        count = dict(stencil_test=0, stencil_op=4, stencil_wrap=0, viewport=_viewport(w, h), vs_uniforms=_vsu(np.eye(4)))
        length, ang = 40.0 * np.exp(0.6 * rng.standard_normal(nl)), rng.uniform(0.0, 2.0 * np.pi, nl)
        sx, sy = rng.uniform(0.0, w - 3.0, nl), rng.uniform(0.0, h - 3.0, nl)
        ex = np.clip(sx + length * np.cos(ang), 0.0, w - 3.0)
        ey = np.clip(sy + length * np.sin(ang), 0.0, h - 3.0)
        lp = np.empty((nl, 2, 3), F32)
        lp[:, 0, 0], lp[:, 1, 0] = sx * (2.0 / w) - 1.0, ex * (2.0 / w) - 1.0
        lp[:, 0, 1], lp[:, 1, 1] = 1.0 - sy * (2.0 / h), 1.0 - ey * (2.0 / h)
        lp[:, :, 2] = rng.uniform(0.02, 0.98, nl)[:, None]
        pp = np.stack([rng.uniform(-1.0, 1.0, npt), rng.uniform(-1.0, 1.0, npt), rng.uniform(0.01, 0.99, npt)], -1)
        line_fs, point_fs = np.zeros(32, F32), np.zeros(32, F32)
        line_fs[0:2], point_fs[0:4] = (0.9, 1.0), (1.0, 1.0, 0.2, 1.0)
        st.fbo, st.tex = st.fb(w, h), st.texture(rng)
        st.draws = [
            (st.mesh(_mesh(pos, nrm, None, uv)),
             sr.make_desc(vertex_program=sr.VP_MVP_NORMAL_UV, geometry_program=2, fragment_program=sr.FP_TEX_LAMBERT,
                          blend=1, tex_filter=1, fs_uniforms=_tex_lambert(), **count)),
            (st.mesh(_mesh(lp.reshape(-1, 3), None, None, rng.random((2 * nl, 2), F32), prim=2)),
             sr.make_desc(vertex_program=sr.VP_MVP_NORMAL_UV, fragment_program=sr.FP_UV_COLOR, blend=1,
                          aa_lines=case["aa"], alpha_mode=1, fs_uniforms=line_fs, **count)),
            (st.mesh(_mesh(pp.astype(F32), None, None, prim=1)),
             sr.make_desc(vertex_program=sr.VP_MVP_NORMAL_UV, fragment_program=sr.FP_FLAT, fs_uniforms=point_fs, **count)),
        ]
        st.color, st.stencil = st.host(w * h), st.host(w * h, torch.uint8)
    elif kind == "example":
        pos, nrm, idx, model, mit, cam, pv = _example_scene(case, seed)
        vsu = _vsu(pv @ model, mit[:3, :3], model)
        vsu[37:40], vsu[40:44] = mit[3, :3], model[3]
        fs = np.zeros(32, F32)
        fs[0:3], fs[3:31], fs[31] = cam, np.asarray(LIGHTS).reshape(28), 0.25
        st.fbo = st.keep(st.ctx.framebuffer_ex(w, h, [sr.COLOR_RGBAF32]))
        st.m = st.mesh(_mesh(pos, nrm, idx))
        st.desc = sr.make_desc(vertex_program=sr.VP_WORLD4_NORMAL4, fragment_program=sr.FP_FRESNEL4,
                               blend=sr.BLEND_OVER_NORMALIZED, vs_uniforms=vsu, fs_uniforms=fs, viewport=_viewport(w, h))
        st.color = st.host(4 * w * h, torch.float32)
    elif kind == "normals":
        pos, nrm, idx, model, mit, cam, pv = _example_scene(case, seed)
        vsu = _vsu(pv @ model, mit[:3, :3], model)
        gs, green = np.zeros(20, F32), np.zeros(32, F32)
        gs[:16], gs[16], green[0:4] = pv.reshape(16), 0.05, (0.0, 1.0, 0.0, 1.0)
        st.fbo, st.m = st.fb(w, h), st.mesh(_mesh(pos, nrm, idx))
        common = dict(vertex_program=sr.VP_MVP_NORMAL_WORLD, blend=1, alpha_mode=1, vs_uniforms=vsu,
                      viewport=_viewport(w, h))
        eye = np.linalg.solve(model, np.append(cam, 1.0))[:3]
        st.descs = [sr.make_desc(fragment_program=sr.FP_BLINN_PHONG, fs_uniforms=_blinn_phong(cam),
                                 cull=_cull_back(pos, idx, pv @ model, w, h, eye), **common),
                    sr.make_desc(geometry_program=4, fragment_program=sr.FP_FLAT, fs_uniforms=green, gs_uniforms=gs,
                                 aa_lines=1, **common)]
        st.color = st.host(w * h)
    elif kind == "deferred":
        pos, nrm, uv = _soup(rng, case["tris"], w, h, case["area"])
        f = sr.COLOR_RGBAF32
        st.gb = st.keep(st.ctx.framebuffer_ex(w, h, [sr.COLOR_RGBA8, f, f, sr.COLOR_RGBA8], stencil=sr.STENCIL_NONE))
        st.fbo, st.m, st.tex = st.fb(w, h), st.mesh(_mesh(pos, nrm, None, uv)), st.texture(rng)
        st.planes = [st.keep(st.ctx.texture_from_fb_plane(st.gb, p)) for p in (0, 1)]
        quad = np.array([[-1, -1, 0.5], [1, -1, 0.5], [1, 1, 0.5], [-1, -1, 0.5], [1, 1, 0.5], [-1, 1, 0.5]], F32)
        quv = np.stack([(quad[:, 0] + 1) / 2, (1 - quad[:, 1]) / 2], -1).astype(F32)
        st.quad = st.mesh(_mesh(quad, np.tile(F32([0, 0, 1]), (6, 1)), None, quv))
        base = dict(vertex_program=sr.VP_MVP_NORMAL_UV, vs_uniforms=_vsu(np.eye(4)), viewport=_viewport(w, h), tex_filter=1)
        st.desc = sr.make_desc(fragment_program=sr.FP_GBUFFER, fs_uniforms=_tex_lambert(1.0), **base)
        # the lit plane as it is, then a fifth of the normal plane over it
        full, part = np.zeros(32, F32), np.zeros(32, F32)
        full[2], full[3], full[5] = 1.0, 1.0, 1.0
        part[2], part[3], part[5] = 1.0, 1.0, 0.2
        st.compose = [(st.planes[0], sr.make_desc(fragment_program=sr.FP_TEX_LAMBERT, fs_uniforms=full, **base)),
                      (st.planes[1], sr.make_desc(fragment_program=sr.FP_TEX_LAMBERT, fs_uniforms=part, blend=1, **base))]
        st.color = st.host(w * h)
    elif kind == "mask":
        pos, nrm, uv = _soup(rng, case["tris"], w, h, case["area"])
        mpos, _, _ = _soup(rng, 48, w, h, w * h / 60.0)
        st.fbo, st.m, st.tex = st.fb(w, h), st.mesh(_mesh(pos, nrm, None, uv)), st.texture(rng)
        st.mask = st.mesh(_mesh(mpos, None, None))
        grey = np.zeros(32, F32)
        grey[0:4] = (0.1, 0.1, 0.12, 1.0)
        base = dict(vertex_program=sr.VP_MVP_NORMAL_UV, vs_uniforms=_vsu(np.eye(4)), viewport=_viewport(w, h), stencil_ref=1)
        st.desc_mask = sr.make_desc(fragment_program=sr.FP_FLAT, fs_uniforms=grey, stencil_test=0, stencil_op=3, **base)
        st.desc = sr.make_desc(fragment_program=sr.FP_TEX_LAMBERT, fs_uniforms=_tex_lambert(), blend=1, tex_filter=1,
                               stencil_test=6, stencil_op=0, **base)
        st.color, st.stencil = st.host(w * h), st.host(w * h, torch.uint8)
    elif kind == "batch":
        tex = st.texture(rng)
        st.items, st.fbs, st.colors = [], [], []
        for n, bw, bh in _batch_specs(rng, case):
            pos, nrm, uv = _soup(rng, n, bw, bh, 20.0)
            fb = st.fb(bw, bh)
            desc = sr.make_desc(vertex_program=sr.VP_MVP_NORMAL_UV, fragment_program=sr.FP_TEX_LAMBERT, blend=1,
                                tex_filter=1, vs_uniforms=_vsu(np.eye(4)), fs_uniforms=_tex_lambert(),
                                viewport=_viewport(bw, bh))
            st.items.append((fb, st.mesh(_mesh(pos, nrm, None, uv)), desc, tex, BACK))
            st.fbs.append(fb)
            st.colors.append(st.host(bw * bh))
    elif kind == "serve":
        st.server = _the_server()
        st.tex = st.texture(rng)
        counts = np.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]), case["meshes"])).round().astype(int)
        meshes = [st.mesh(_mesh(p, n, None, uv)) for p, n, uv in (_cloud(rng, int(c)) for c in counts)]
        st.requests = []
        for i in range(case["requests"]):
            rw, rh = [(512, 512), (1920, 1080)][i % 2]
            desc = sr.make_desc(vertex_program=sr.VP_MVP_NORMAL_UV, fragment_program=sr.FP_TEX_LAMBERT, blend=1,
                                tex_filter=1, vs_uniforms=_vsu(_orbit(rng, rw, rh)), fs_uniforms=_tex_lambert(),
                                viewport=_viewport(rw, rh))
            st.requests.append((meshes[int(rng.integers(len(meshes)))], desc, rw, rh))
    else:
        raise ValueError(kind)
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(st):
    kind, ctx = st.kind, st.ctx
    if kind == "mesh":
        st.fbo.clear(BACK, -1.0)
        ctx.draw(st.fbo, st.m, st.desc)
        _read(st.fbo, st.color, st.depth)
        return [st.color, st.depth]
    if kind == "soup":
        st.fbo.clear(BACK)
        ctx.draw(st.fbo, st.m, st.desc, st.tex)
        st.fbo.read_color_into(st.color.data_ptr())
        return [st.color]
    if kind == "terrain":
        st.fbo.clear(0xFFC09060)
        ctx.draw(st.fbo, st.m, st.desc)
        st.fbo.read_color_into(st.color.data_ptr())
        return [st.color]
    if kind == "clip":
        st.fbo.clear(BACK)
        for m, desc in st.draws:
            ctx.draw(st.fbo, m, desc, st.tex)
        _read(st.fbo, st.color, None, st.stencil)
        return [st.color, st.stencil]
    if kind == "example":
        st.fbo.clear_ex([(0.01, 0.01, 0.01, 1.0)])
        ctx.draw(st.fbo, st.m, st.desc)
        planes = (ctypes.c_void_p * 1)(st.color.data_ptr())
        rc = sr.lib().sr_fb_read_ex(st.fbo.h, planes, None, None)
        if rc != sr.SR_OK:
            raise sr.SoftrenderError(rc, "sr_fb_read_ex")
        return [st.color]
    if kind == "normals":
        st.fbo.clear(BACK)
        ctx.draw_chains(st.fbo, st.m, st.descs)
        st.fbo.read_color_into(st.color.data_ptr())
        return [st.color]
    if kind == "deferred":
        st.gb.clear_ex([BACK, 0.0, 0.0, BACK])
        ctx.draw(st.gb, st.m, st.desc, st.tex)
        st.fbo.clear(BACK)
        for plane, desc in st.compose:
            ctx.draw(st.fbo, st.quad, desc, plane)
        st.fbo.read_color_into(st.color.data_ptr())
        return [st.color]
    if kind == "mask":
        st.fbo.clear(BACK)
        ctx.draw(st.fbo, st.mask, st.desc_mask)
        ctx.draw(st.fbo, st.m, st.desc, st.tex)
        _read(st.fbo, st.color, None, st.stencil)
        return [st.color, st.stencil]
    if kind == "batch":
        ctx.batch_draw(st.items)
        for fb, color in zip(st.fbs, st.colors):
            fb.read_color_into(color.data_ptr())
        return st.colors
    # serve: the completions' pinned pixels are used in place and given back
    # before the next burst
    st.release_held()
    where = {}
    for i, (m, desc, w, h) in enumerate(st.requests):
        where[st.server.submit(m, desc, w, h, st.tex)] = i
    out = [None] * len(where)
    buf, n = (sr.Completion * 64)(), ctypes.c_uint32()
    while where:
        rc = sr.lib().sr_server_poll(st.server.h, buf, 64, ctypes.byref(n), -1)
        if rc != sr.SR_OK:
            raise sr.SoftrenderError(rc, "sr_server_poll")
        for c in buf[:n.value]:
            st.held.append(c.ticket)
            if c.status != sr.SR_OK:
                raise sr.SoftrenderError(c.status, "served request")
            out[where.pop(c.ticket)] = np.ctypeslib.as_array(c.rgba, shape=(c.width * c.height,)).view(np.int32)
    return out


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
PER_VERTEX, PER_TRIANGLE, PER_PIXEL = 60.0, 40.0, 60.0  # operations: transform; edges and box; test, shade and blend once
TEXTURE = 4 * 1024 * 1024


def _ball_tris(case):
    return 2 * case["slices"] * (case["stacks"] - 1)


def _work(vertices, vertex_bytes, indices, tris, pixels, fb_bytes, textures=0):
    return dict(bytes=vertices * vertex_bytes + 4.0 * indices + pixels * fb_bytes + textures,
                flops=PER_VERTEX * vertices + PER_TRIANGLE * tris + PER_PIXEL * pixels)


def work(case):
    """Vertices, indices and texture read once, the planes written once and read back once (those that are)."""
    kind = case["kind"]
    px = case.get("w", 0) * case.get("h", 0)
    if kind in ("mesh", "example", "normals"):
        t = _ball_tris(case)
        v = (case["stacks"] + 1) * (case["slices"] + 1)
        fb = {"mesh": 16, "example": 36, "normals": 12}[kind]
        return _work(v, 24, 3 * t, t, px, fb)
    if kind == "soup":
        return _work(3 * case["tris"], 32, 0, case["tris"], px, 12, TEXTURE)
    if kind == "terrain":
        v, t = (case["grid"] + 1) ** 2, 2 * case["grid"] ** 2
        return _work(v, 24, 3 * t, t, px, 12)
    if kind == "clip":
        v = 3 * case["tris"] + 2 * case["lines"] + case["points"]
        return _work(v, 24, 0, case["tris"] + case["lines"], px, 14, TEXTURE)
    if kind == "deferred":
        return _work(3 * case["tris"], 32, 0, case["tris"], px, 44 + 20 + 12, TEXTURE)
    if kind == "mask":
        return _work(3 * case["tris"], 32, 0, case["tris"], px, 14, TEXTURE)
    n = case["scenes"] if kind == "batch" else case["requests"]
    mean = (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"])
    sizes = [256 * 256, 512 * 512, 1920 * 1080] if kind == "batch" else [512 * 512, 1920 * 1080]
    px = sum(sizes[i % len(sizes)] for i in range(n))
    kept = n if kind == "batch" else case["meshes"]
    return dict(bytes=kept * mean * 96 + px * 12.0 + TEXTURE,
                flops=n * mean * (3 * PER_VERTEX + PER_TRIANGLE) + PER_PIXEL * px)


# ---------------------------------------------------------------------------
# the same frames in 64 bits
# ---------------------------------------------------------------------------
def _screen64(pos, mvp, w, h):
    """Screen x, y, z of each vertex: y down, z in (-1, -0.5) and larger when nearer."""
    c = np.c_[pos.astype(np.float64), np.ones(len(pos))] @ np.asarray(mvp, np.float64).T
    n = c[:, :3] / c[:, 3:]
    return np.stack([(n[:, 0] + 1.0) * w / 2.0, (1.0 - n[:, 1]) * h / 2.0, -0.5 * n[:, 2] - 0.5], -1)


def _raster64(scr, idx, w, h, keep, far):
    """Depth and, per pixel, the last triangle that passed and its barycentrics."""
    depth = np.full((h, w), far)
    tri = np.full((h, w), -1)
    bary = np.zeros((h, w, 3))
    for t, (a, b, c) in enumerate(scr[idx].reshape(-1, 3, 3)):
        if not keep[t]:
            continue
        x0, x1 = max(0, int(min(a[0], b[0], c[0]))), min(w - 1, int(max(a[0], b[0], c[0])))
        y0, y1 = max(0, int(min(a[1], b[1], c[1]))), min(h - 1, int(max(a[1], b[1], c[1])))
        det = (b[1] - c[1]) * (a[0] - c[0]) + (c[0] - b[0]) * (a[1] - c[1])
        if x0 > x1 or y0 > y1 or det == 0.0:
            continue
        dx, dy = np.arange(x0, x1 + 1)[None, :] + 0.5 - c[0], np.arange(y0, y1 + 1)[:, None] + 0.5 - c[1]
        u = ((b[1] - c[1]) * dx + (c[0] - b[0]) * dy) / det
        v = ((c[1] - a[1]) * dx + (a[0] - c[0]) * dy) / det
        q = 1.0 - u - v
        z = a[2] * u + b[2] * v + c[2] * q
        at = (slice(y0, y1 + 1), slice(x0, x1 + 1))
        ok = (u >= 0) & (v >= 0) & (q >= 0) & (z < 0) & (z >= depth[at])
        depth[at][ok] = z[ok]
        tri[at][ok] = t
        bary[at][ok] = np.stack([u, v, q], -1)[ok]
    return depth, tri, bary


def _unit_rows(v):
    return v / np.sqrt((v * v).sum(-1, keepdims=True))


def exact(case, seed):
    """Depth of a mesh frame and the float colours of an example frame; the
    other outputs are bytes, which stay as they are."""
    kind, w, h = case["kind"], case.get("w"), case.get("h")
    if kind not in ("mesh", "example") or _ball_tris(case) > 60_000:
        return None
    rng = np.random.default_rng(seed)
    if kind == "mesh":
        pos, _, idx = _ball(rng, case["stacks"], case["slices"])
        eye = (0.0, 0.0, 3.0)
        mvp = (_perspective(60.0, w / h, 0.1, 100.0) @ _look_at(eye, (0.0, 0.0, 0.0))).astype(F32)
        scr = _screen64(pos, mvp, w, h)
        x, y = scr[idx][:, 0].reshape(-1, 3), scr[idx][:, 1].reshape(-1, 3)
        area = (x * np.roll(y, -1, 1) - np.roll(x, -1, 1) * y).sum(1)
        keep = area >= 0 if _cull_back(pos, idx, mvp, w, h, eye) == 1 else area < 0
        return [None, _raster64(scr, idx, w, h, keep, -1.0)[0].reshape(-1)]
    pos, nrm, idx, model, mit, cam, pv = _example_scene(case, seed)
    mvp, model, mit = (m.astype(F32).astype(np.float64) for m in (pv @ model, model, mit))
    scr = _screen64(pos, mvp, w, h)
    _, tri, bary = _raster64(scr, idx, w, h, np.ones(len(idx) // 3, bool), -np.inf)
    wp = np.c_[pos.astype(np.float64), np.ones(len(pos))] @ model.T
    wn = _unit_rows(np.c_[nrm.astype(np.float64), np.zeros(len(nrm))] @ mit.T)
    hit = tri >= 0
    vid, b = idx.reshape(-1, 3)[tri[hit]], bary[hit][:, :, None]
    p, n = (wp[vid] * b).sum(1), (wn[vid] * b).sum(1)
    view = _unit_rows(np.append(cam.astype(F32), 1.0) - p)
    col = np.zeros((len(p), 3))
    grey, f0 = 0.25 ** 2.2, ((1.0 - 1.45) / (1.0 + 1.45)) ** 2
    for light in np.asarray(LIGHTS, F32).astype(np.float64):
        d = np.append(light[:3], 1.0) - p
        dist = np.sqrt((d * d).sum(-1))
        d = d / dist[:, None]
        half = _unit_rows(d + view)
        dot = lambda a, c: np.clip((a * c).sum(-1), 0.0, 1.0)  # noqa: E731
        f = f0 + (1.0 - f0) * (1.0 - dot(view, half)) ** 5
        amount = f * dot(n, half) ** 64 + (1.0 - f) * dot(d, n) * 0.7 * grey
        col += (light[6] / dist ** 2 * amount)[:, None] * light[3:6]
    tone = (col * (2.51 * col + 0.03)) / (col * (2.43 * col + 0.59) + 0.14)
    out = np.tile([0.01, 0.01, 0.01, 1.0], (h, w, 1))
    out[hit] = np.c_[tone ** (1.0 / 2.2), np.ones(len(p))]
    return [out.reshape(-1)]
