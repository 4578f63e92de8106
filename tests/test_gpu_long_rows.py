"""Signals whose row is so long that its element counts, or the products of counts that an index is
worked out from, leave 32 bits: what the kernels count in 64 bits there, and the sizes on either side
of the line.  Data movement is exact."""
import numpy as np
import pytest

from util import announce, run_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("c,w,wo", [(1, 40000, 80000), (8, 40000, 80000), (8, 40000, 60001), (3, 40000, 60001), (5, 70000, 30001),
                                    (8, 16384, 65535), (8, 16384, 65537), (3, 16384, 65536)])
@pytest.mark.parametrize("mode", [{}, {"fp16": True}], ids=["fp32", "fp16"])
def test_nearest_resize_of_a_long_row(c, w, wo, mode):
    """(whole factors in vectors and by elements, ragged factors up and down, W * Wo at 2^30)"""
    announce("resize %d x %d -> %d %s" % (c, w, wo, mode))
    x = (np.arange(2 * c * w, dtype=np.int64) % 2039).astype(np.float32).reshape(2, c, 1, w)

    def build(b):
        b.output(b.resize_nearest(b.arg("x", x.shape), (1, wo), name="y"), "y")
    got, want = run_both(build, {"x": x}, **mode)
    assert np.array_equal(got["y"], want["y"])
