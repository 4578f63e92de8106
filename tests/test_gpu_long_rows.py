"""Signals whose row is so long that its element counts, or the products of counts that an index is
worked out from, leave 32 bits: what the kernels count in 64 bits there, and the sizes on either side
of the line.  Data movement is exact."""
import numpy as np
import pytest

from util import announce, run_both, run_hip

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


def test_pooling_of_an_image_beyond_2g_positions():
    """One channel, 32769 x 65535 results: checked in rows from the start, the middle and the end."""
    H, W = 32770, 65536
    assert (H - 1) * (W - 1) > 2 ** 31
    announce("pool %d x %d" % (H, W))
    row = lambda h: ((np.arange(W) * 13 + h * 7) % 2039).astype(np.float32)
    x = np.empty((1, 1, H, W), np.float32)
    period = np.stack([row(h) for h in range(2039)])   # (rows repeat: 2039 is prime)
    for h in range(0, H, 2039):
        x[0, 0, h:h + 2039] = period[:H - h]

    def build(b):
        b.output(b.maxpool(b.arg("x", x.shape), (2, 2), (1, 1), (0, 0, 0, 0), name="y"), "y")
    got = run_hip(build, {"x": x})["y"]
    assert got.shape == (1, 1, H - 1, W - 1)
    for h in (0, 1, H // 2, 32767, H - 2):
        two = np.maximum(row(h), row(h + 1))
        assert np.array_equal(got[0, 0, h], np.maximum(two[1:], two[:-1])), h
