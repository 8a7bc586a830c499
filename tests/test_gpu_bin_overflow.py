"""Draws whose pairs are sorted and do not fit the buffers a fresh context
guesses (room for 4 a triangle and 4,096, and a quarter over): some triangles'
pairs fit and some do not, nothing is drawn, the buffers grow, all pairs (those
of triangles over more than 32 bins among them) are emitted again and the draw
equals the oracle."""
import os
import re

import pytest

import softrender_hip as sr
from parity import assert_parity, render_gpu, render_ref
from test_gpu_wide_bins import soup

pytestmark = pytest.mark.gpu

W, H, N, SIZE = 640, 480, 66_000, 75.0
INTERNAL = os.path.join(os.path.dirname(sr.__file__), "csrc", "sr_internal.hpp")


@pytest.mark.parametrize("mode", [{}, dict(stencil_test=0, stencil_op=4, stencil_wrap=0)])
def test_sorted_pairs_overflow_and_draw_again(mode):
    most = int(re.search(r"constexpr uint32_t DIRECT_TRIS = (\d+);", open(INTERNAL).read()).group(1))
    assert N > most  # more triangles than are ever binned directly
    s = soup(N, W, H, SIZE, seed=0xB1)
    s["desc"] = dict(s["desc"], **mode)
    ref, _ = render_ref(s)
    ctx = sr.Context(0)
    try:
        got = render_gpu(ctx, s)
        pairs = ctx.last_stats()["bin_pairs"]
        assert pairs > (4 * N + 4096) * 5 // 4, pairs
        assert_parity(got, ref)
        assert_parity(render_gpu(ctx, s), ref)  # the grown buffers hold it at once
        assert ctx.last_stats()["bin_pairs"] == pairs
    finally:
        ctx.close()
