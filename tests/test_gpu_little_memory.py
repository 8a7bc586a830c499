"""Draws on a device without room for the larger of two workspaces take the
smaller one and equal the oracle.  A process of its own, in which allocations
above a limit fail."""
import ctypes
import os
import shutil
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))
MIB = 1 << 20


def few_triangles():
    """Lists for direct binning: 30,000 triangles times 256 bins, 31 MB."""
    from test_gpu_wide_bins import soup
    return soup(30_000, 512, 512, 4.0, seed=7), 16 * MIB


def tiny_screen_tiles():
    """Strip counts of 511 x 511 screen tiles: 11 arrays of a MiB and 8 without the shared ones (and a quarter over)."""
    from test_gpu_wide_bins import soup
    s = soup(300, 512, 512, 30.0, seed=8)
    s["desc"] = dict(s["desc"], tile_w=1, tile_h=1, stencil_test=0, stencil_op=4, stencil_wrap=0)
    return s, 12 * MIB


SCENES = {"direct lists": few_triangles, "strip arrays": tiny_screen_tiles}


@pytest.mark.parametrize("what", list(SCENES))
def test_draw(what, tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host compiler")
    shim = str(tmp_path / "malloc_limit.so")
    subprocess.run([cxx, "-shared", "-fPIC", "-O1", "-o", shim, os.path.join(HERE, "cpp", "malloc_limit.cpp")], check=True)
    r = subprocess.run([sys.executable, "-u", os.path.abspath(__file__), shim, what], capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr


def main(shim, what):
    limit = ctypes.CDLL(shim, mode=ctypes.RTLD_GLOBAL)
    limit.malloc_limit.argtypes = [ctypes.c_void_p, ctypes.c_size_t]
    import conftest  # noqa: F401  (the import paths)
    import softrender_hip as sr
    sr.lib()  # loads the library, and the HIP runtime with it
    with open("/proc/self/maps") as maps:
        hip = next(line.split()[-1] for line in maps if "libamdhip64" in line)
    real = ctypes.cast(ctypes.CDLL(hip).hipMalloc, ctypes.c_void_p)
    limit.malloc_limit(real, ~0 & (2 ** 64 - 1))
    from parity import assert_parity, render_gpu, render_ref
    ctx = sr.Context(0)
    scene, most = SCENES[what]()
    limit.malloc_limit(real, most)
    print(f"{what}: allocations above {most} bytes fail", flush=True)
    got = [render_gpu(ctx, scene) for _ in range(2)]
    assert limit.malloc_refused() > 0
    ref, _ = render_ref(scene)
    for g in got:
        assert_parity(g, ref)
    limit.malloc_limit(real, ~0 & (2 ** 64 - 1))
    assert_parity(render_gpu(ctx, scene), ref)
    ctx.close()


if __name__ == "__main__":
    main(*sys.argv[1:])
