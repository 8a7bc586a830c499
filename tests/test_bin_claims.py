"""What binning and the raster's 4x4 groups leave out, checked on the CPU by
brute force: a numpy float64 restatement of row_bins and cover_planes
(sr_kernels.hip) and of group_cover (sr_raster.hip) against every pixel whose
centre passes the coverage test of triangle.rs:104-113 in float32.  Also the
float form of the unorm table (unorm8, sr_device.hpp)."""
import numpy as np
import pytest

from test_strip_reach import passing_pixels

f32, f64 = np.float32, np.float64
W, H = 300, 220


def records(x, y):
    """The f32 fields of a triangle record, and its box (setup's rounding)."""
    x1, x2, x3 = (f32(v) for v in x)
    y1, y2, y3 = (f32(v) for v in y)
    det = ((y2 - y3) * (x1 - x3)) + ((x3 - x2) * (y1 - y3))
    box = (int(np.floor(np.clip(min(x), -1, W))), int(np.floor(np.clip(max(x), -1, W))),
           int(np.floor(np.clip(min(y), -1, H))), int(np.floor(np.clip(max(y), -1, H))))
    with np.errstate(all="ignore"):
        R = f64(1.0) / f64(det)
    return R, f64(x3), f64(y3), f64(y2 - y3), f64(x3 - x2), f64(y3 - y1), f64(x1 - x3), box


def group_cover(rec, X, Y):
    R, x3, y3, e23y, e23x, e31y, e31x, _ = rec
    with np.errstate(all="ignore"):
        ua, ub, va, vb = e23y * R, e23x * R, e31y * R, e31x * R
        dx, dy = X + 0.5 - x3, Y + 0.5 - y3
        DX, DY = max(abs(dx), abs(dx + 7)), max(abs(dy), abs(dy + 7))
        tu, tv = abs(ua) * DX + abs(ub) * DY, abs(va) * DX + abs(vb) * DY
        tiny = 2.0 ** -100 + 2.0 ** -140 * abs(R)
        u0, v0 = ua * dx + ub * dy, va * dx + vb * dy
        wa, wb = -(ua + va), -(ub + vb)
        best = lambda a, b: 3.0 * (max(a, 0.0) + max(b, 0.0))
        u = u0 + best(ua, ub) + (2.0 ** -18 * tu + tiny)
        v = v0 + best(va, vb) + (2.0 ** -18 * tv + tiny)
        w = 1.0 - u0 - v0 + best(wa, wb) + (2.0 ** -18 * (tu + tv + 1.0) + tiny)
        m = 0
        for g in range(4):
            ox, oy = 4.0 * (g & 1), 4.0 * (g >> 1)
            if not (u + (ua * ox + ub * oy) < 0 or v + (va * ox + vb * oy) < 0 or w + (wa * ox + wb * oy) < 0):
                m |= 1 << g
    return m


def row_runs(rec):
    """Per bin row of the clamped box: the first and last bin kept (row_bins), or
    None where the box misses the framebuffer."""
    R, x3, y3, e23y, e23x, e31y, e31x, (X0, X1, Y0, Y1) = rec
    px0, px1, py0, py1 = max(X0, 0), min(X1, W - 1), max(Y0, 0), min(Y1, H - 1)
    if px0 > px1 or py0 > py1:
        return {}
    with np.errstate(all="ignore"):
        ox, oy = 0.5 - x3, 0.5 - y3
        ua, ub, uc = e23y * R, e23x * R, (e23y * ox + e23x * oy) * R
        va, vb, vc = e31y * R, e31x * R, (e31y * ox + e31x * oy) * R
        wa, wb, wc = -(ua + va), -(ub + vb), (1.0 - uc) - vc
        mu = mv = au = av = 0.0
        for k in range(4):
            dx, dy = (px1 if k & 1 else px0) + ox, (py1 if k & 2 else py0) + oy
            mu = max(mu, (abs(e23y * dx) + abs(e23x * dy)) * abs(R))
            mv = max(mv, (abs(e31y * dx) + abs(e31x * dy)) * abs(R))
            au, av = max(au, abs((e23y * dx + e23x * dy) * R)), max(av, abs((e31y * dx + e31x * dy) * R))
        xm, ym, s = px1 + 1.0, py1 + 1.0, 2.0 ** -18
        eu = 2.0 ** -48 * (abs(ua) * xm + abs(ub) * ym + abs(uc) + mu + 1)
        ev = 2.0 ** -48 * (abs(va) * xm + abs(vb) * ym + abs(vc) + mv + 1)
        ew = 2.0 ** -48 * (abs(wa) * xm + abs(wb) * ym + abs(wc)) + eu + ev
        planes = ((ua, ub, uc, s * (mu + au + 1) + eu), (va, vb, vc, s * (mv + av + 1) + ev),
                  (wa, wb, wc, s * (mu + mv + au + av + 3) + ew))
    runs = {}
    for by in range(py0 >> 5, (py1 >> 5) + 1):
        lo, hi = px0 >> 5, px1 >> 5
        y0, y1 = max(py0, by * 32), min(py1, by * 32 + 31)
        for a, b, k, d in planes:
            with np.errstate(all="ignore"):
                r = -d - (b * (y1 if b > 0 else y0) + k)
                if a > 0:
                    q = r / a - 1.0
                    if q > px1:
                        hi = -1
                    elif q > px0:
                        lo = max(lo, int(np.floor(q)) >> 5)
                elif a < 0:
                    q = r / a + 1.0
                    if q < px0:
                        hi = -1
                    elif q < px1:
                        hi = min(hi, int(np.floor(q)) >> 5)
                elif r > 0:
                    hi = -1
        runs[by] = (lo, hi)
    return runs


def triangles(kind, n, seed):
    rng = np.random.default_rng(seed)
    c = rng.uniform(-20, [W + 20, H + 20], (n, 1, 2))
    if kind == "sliver":  # long, a fraction of a pixel wide
        d = rng.normal(size=(n, 1, 2))
        d /= np.linalg.norm(d, axis=2, keepdims=True)
        t = rng.uniform(-300, 300, (n, 3, 1))
        p = c + t * d + 10.0 ** rng.uniform(-5, -0.5, (n, 1, 1)) * rng.normal(size=(n, 3, 2))
    elif kind == "lattice":  # edges and vertices exactly on pixel centres
        p = np.round(c + rng.normal(size=(n, 3, 2)) * 12) + 0.5
    else:
        p = c + rng.normal(size=(n, 3, 2)) * {"tiny": 0.7, "small": 6.0, "large": 150.0, "far": 4e6}[kind]
    return p[..., 0].astype(f32), p[..., 1].astype(f32)


@pytest.mark.parametrize("kind", ["tiny", "small", "large", "far", "sliver", "lattice"])
def test_groups_and_rows_keep_every_passing_pixel(kind):
    x, y = triangles(kind, 150, seed=len(kind))
    kept = skipped = passed = 0
    for t in range(len(x)):
        rec = records(x[t], y[t])
        if not abs(rec[0]) < np.inf:
            continue
        px, py = passing_pixels(x[t], y[t], W, H)
        passed += px.size
        X0, X1, Y0, Y1 = rec[7]
        inside = (px >= X0) & (px <= X1) & (py >= Y0) & (py <= Y1)  # strip pixels have bins of their own
        runs = row_runs(rec)
        for qx, qy in {(int(a) >> 5, int(b) >> 5) for a, b in zip(px[inside], py[inside])}:
            assert runs[qy][0] <= qx <= runs[qy][1], (kind, t, qx, qy, runs[qy])
        hit = {}
        for a, b in zip(px.tolist(), py.tolist()):
            g = (a >> 2 & 1) | (b >> 2 & 1) << 1
            hit[(a & ~7, b & ~7)] = hit.get((a & ~7, b & ~7), 0) | 1 << g
        tiles = {(a, b) for a in range(max(X0, 0) & ~7, min(X1, W - 1) + 1, 8)
                 for b in range(max(Y0, 0) & ~7, min(Y1, H - 1) + 1, 8)} if len(hit) < 200 else set()
        for tile in tiles | set(hit):
            m = group_cover(rec, *tile)
            assert hit.get(tile, 0) & ~m == 0, (kind, t, tile)
            kept += bin(m).count("1")
            skipped += 4 - bin(m).count("1")
    assert passed > 0
    if kind in ("small", "lattice"):
        assert skipped > kept // 2, (kept, skipped)  # the test leaves something out


def test_unorm8_equals_the_table():
    i = np.arange(256, dtype=f64)
    hi, lo = f64(f32(float.fromhex("0x1.010102p-8"))), f32(float.fromhex("-0x1.fdfdfep-33"))
    small = (i.astype(f32) * lo).astype(f64)
    # i * hi needs 32 bits and the sum fewer than 53: float64 holds it exactly, so one rounding as in a fused sum
    assert np.array_equal((i * hi + small).astype(f32), (i.astype(f32) / f32(255.0)))
    back = np.floor((i.astype(f32) / f32(255.0)) * f32(255.0) + f32(0.5))
    assert np.array_equal(back, i)
