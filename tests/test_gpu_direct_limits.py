"""The most triangles that are binned directly, and one more, in frames of few
and of more bins: against the oracle, bit for bit."""
import pytest

from parity import assert_parity, render_gpu, render_ref
from test_gpu_wide_bins import soup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,most", [(64, 64, 8192 + 512 * 4), (20, 16, 8192 + 512), (320, 200, 32768)])
@pytest.mark.parametrize("more", [0, 1])
def test_limits(ctx, w, h, most, more):
    s = soup(most + more, w, h, 5.0, seed=most)
    ref, _ = render_ref(s)
    assert_parity(render_gpu(ctx, s), ref)
    s["desc"] = dict(s["desc"], blend=0, stencil_test=0, stencil_op=4, stencil_wrap=1)
    ref, _ = render_ref(s)
    assert_parity(render_gpu(ctx, s), ref)
