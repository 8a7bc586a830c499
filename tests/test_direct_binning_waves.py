"""k_bin_direct's work-group, its waves as far apart as its barriers let them be.

The kernel's own source runs on the CPU, a fiber a thread: one wave at a time
goes on until it stands at a barrier, in an order of the test's choice.  All
waves have to stand at the same barrier each time (a wave that reads a word
another one already wrote for the next chunk goes elsewhere), and every bin's
list is the triangles whose box holds it, in order."""
import os
import re
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = os.path.join(ROOT, "rust-softrender_amd", "csrc", "sr_kernels.hip")
HOST = os.path.join(ROOT, "tests", "cpp", "direct_waves.cpp")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host compiler")
    text = open(SOURCE).read()
    sizes = re.search(r"^constexpr uint32_t DIRECT_THREADS = .*$", text, re.M)
    kernel = re.search(r"^__global__ __launch_bounds__\(DIRECT_THREADS\) void k_bin_direct\(.*?^}$", text, re.M | re.S)
    assert sizes and kernel
    out = tmp_path_factory.mktemp("direct_waves")
    (out / "kernel.inc").write_text(sizes.group(0) + "\n" + kernel.group(0) + "\n")
    subprocess.run([cxx, "-std=c++17", "-O1", "-I", str(out), "-o", str(out / "run"), HOST], check=True)
    return str(out / "run")


def boxes(kind, n, rng):
    """Per triangle its bin box (columns and rows, inclusive; lo > hi: none) on a 3 x 2 grid of bins."""
    x0, y0 = rng.integers(0, 3, n), rng.integers(0, 2, n)
    x1, y1 = np.minimum(x0 + rng.integers(0, 2, n), 2), np.minimum(y0 + rng.integers(0, 2, n), 1)
    if kind == "chunks apart":  # bin 0 meets only the second chunk, bin 5 only the last triangle
        x0, x1, y0, y1 = np.full(n, 1), np.full(n, 1), np.zeros(n, int), np.zeros(n, int)
        x0[4096:8192:3] = x1[4096:8192:3] = 0
        x0[-1] = x1[-1] = 2
        y0[-1] = y1[-1] = 1
    elif kind == "culled":
        x0[rng.random(n) < 0.7] = 9
    return x0, x1, y0, y1


@pytest.mark.parametrize("order", ["up", "down"])
@pytest.mark.parametrize("kind,n", [("any", 1), ("any", 700), ("any", 4097), ("chunks apart", 4096), ("chunks apart", 4098),
                                    ("chunks apart", 12_289), ("culled", 9000)])
def test_waves_meet_at_every_barrier(program, kind, n, order, tmp_path):
    x0, x1, y0, y1 = boxes(kind, n, np.random.default_rng(n))
    path = tmp_path / "boxes"
    np.stack([x0 | x1 << 16, y0 | y1 << 16], 1).astype(np.uint32).tofile(path)
    for b in range(6):
        r = subprocess.run([program, str(path), str(n), "3", str(b), order], capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, (kind, n, b, r.stderr)
        bx, by = b % 3, b // 3
        want = np.nonzero((x0 <= bx) & (bx <= x1) & (y0 <= by) & (by <= y1))[0]
        assert np.array_equal(np.array(r.stdout.split(), dtype=np.int64), want), (kind, n, b)
