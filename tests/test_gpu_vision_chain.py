"""Operators between convolutions on channels-last tensors: the layout change at the first
element-wise operator, BatchNorm with its activation, results stored as channel slices of
a Concat, reductions of odd channel counts (split over the reduced axis where the columns
are few), the conversion of a channels-last result to its declared type in one launch, and
results written into the caller's device buffers.  Sizes at the edges of the vectors (odd
channels, one channel), the tiles (64 positions, 64 channels) and the reduction's slices."""
import numpy as np
import pytest

import __graft_entry__ as entry
from util import announce, run_hip, run_ref

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 3), (2, 3, 7), (1, 162, 67), (3, 25, 39), (2, 64, 16), (5, 96, 33), (1, 8, 150), (2, 130, 8), (4, 65, 9)]
KW = {"fp32": {}, "fp16": {"fp16": True}, "bf16": {"bf16": "performance"}}
TOL = {"fp32": 1e-4, "fp16": 2e-2, "bf16": 6e-2}


def build_chain(n, c, hw):
    r = np.random.default_rng(c)
    m, v, g, o = (t.astype(np.float32) for t in (r.standard_normal(c), r.random(c) + 0.5, r.standard_normal(c), r.standard_normal(c)))

    def build(b):
        x = b.arg("x", (n, c, hw, hw))
        y = b.batchnorm(x, b.const("m", m), b.const("v", v), 1e-5, b.const("g", g), b.const("o", o), name="bn")
        y = b.leaky_relu(y, 0.1, name="act")
        p = b.maxpool(y, (3, 3), (2, 2), (1, 1, 1, 1), name="mp")
        a = b.avgpool(y, (2, 2), (1, 1), (0, 0, 0, 0), name="ap")
        up = b.resize_nearest(p, (hw, hw), name="up")
        s = b.sigmoid(b.avgpool(y, (1, 1), (1, 1), (0, 0, 0, 0), name="id"), name="gate")
        b.output(b.concat([up, b.add(y, x, name="res"), s], 1, name="cat"), "cat")
        b.output(b.softmax(b.reshape(b.reduce_mean(a, (2, 3), True, name="gap"), (n, c), name="flat"), -1, name="prob"), "prob")
        b.output(b.reduce_max(y, (2, 3), True, name="peak"), "peak")
        b.output(b.reduce_l2(y, (2, 3), True, 0.0, name="l2"), "l2")
    return build


@pytest.mark.parametrize("mode", list(KW))
@pytest.mark.parametrize("size", SIZES)
def test_chain(size, mode):
    n, c, hw = size
    announce("vision chain %s %s" % (size, mode))
    build = build_chain(n, c, hw)
    feeds = {"x": np.random.default_rng(1).standard_normal((n, c, hw, hw)).astype(np.float32)}
    want = run_ref(build, feeds)
    got = run_hip(build, feeds, **KW[mode])
    for k in want:
        assert got[k].shape == want[k].shape
        d = float(np.max(np.abs(got[k] - want[k])))
        assert d <= TOL[mode] * max(1.0, float(np.max(np.abs(want[k])))), (k, d)
    # the same bits when every argument and result is bound to device memory, replayed
    odla = entry.load().odla
    hb = odla.HipBuilder(**KW[mode])
    build(hb)
    s = hb.session()
    s.bind_device_io(feeds)
    for _ in range(3):
        s.execute()
        dev = s.fetch_device_outputs()
        for k in want:
            assert np.array_equal(dev[k], got[k]), k
    s.close()
    hb.destroy()
