"""Operators within a plane as one launch: windows and element-wise instructions at the edges of
their rows (fewer than four results, one more than a multiple of four), several planes per
workgroup with a ragged last chunk, planes that fill the LDS, every kind of window, values with
several places to go, and the graphs that have to keep their other routes."""
import numpy as np
import pytest

import __graft_entry__ as entry
from test_plan_layernorm_cpu import steps_of
from util import announce, run_both

pytestmark = pytest.mark.gpu

KW = {"fp32": {}, "fp16": {"fp16": True}, "bf16": {"bf16": "performance"}}
EPS = {"fp32": 2.0 ** -23, "fp16": 2.0 ** -11, "bf16": 2.0 ** -8}


def check(build, feeds, mode, steps, ops=8, grouped=True):
    """`ops` roundings of values of the result's size, and one more for the sums; `steps`: launches of the plan."""
    got, want = run_both(build, feeds, **KW[mode])
    names = steps_of(entry.load().odla, build, **KW[mode])
    assert any(m.startswith("planes(") for m in names) == grouped, names
    if steps is not None:
        assert len(names) == steps, names
    for k in want:
        assert got[k].shape == want[k].shape
        scale = max(1.0, float(np.max(np.abs(want[k]))))
        assert float(np.max(np.abs(got[k] - want[k]))) <= (ops + 1) * EPS[mode] * scale, (k, mode)


def image(*shape, seed=3):
    return np.random.default_rng(seed).standard_normal(shape).astype(np.float32)


WINDOWS = [("max", (2, 2), (2, 2), 0), ("max", (3, 3), (2, 2), 1), ("max", (3, 3), (1, 1), 1), ("max", (5, 3), (2, 1), 1), ("avg", (1, 1), (1, 1), 0),
           ("avg", (2, 2), (1, 1), 0), ("avg", (2, 2), (2, 2), 0), ("avg", (3, 3), (2, 2), 1), ("avg", (3, 3), (2, 2), 0), ("avg", (4, 2), (3, 2), 1)]


@pytest.mark.parametrize("mode", KW)
@pytest.mark.parametrize("kind,window,step,pad", WINDOWS)
def test_windows(kind, window, step, pad, mode):
    for n, c, h, w in ((1, 1, 6, 5), (2, 3, 9, 7), (1, 37, 8, 11), (3, 130, 6, 6), (1, 2, 64, 67), (1, 5, 150, 33)):
        announce("plane windows %s %s %s %s" % (mode, kind, window, (n, c, h, w)))

        def build(b):
            x = b.arg("x", (n, c, h, w))
            pool = b.maxpool if kind == "max" else b.avgpool
            y = pool(b.leaky_relu(x, 0.25, name="a"), window, step, (pad,) * 4, name="p")
            b.output(y, "pool")
            b.output(b.reduce_mean(y, (2, 3), True, name="m"), "mean")

        check(build, {"x": image(n, c, h, w)}, mode, 1)


@pytest.mark.parametrize("mode", KW)
@pytest.mark.parametrize("kind,window,step,pad", WINDOWS)
def test_mean_of_a_pool_that_nothing_else_reads(kind, window, step, pad, mode):
    """The pool's own result is no result of the plan."""
    for n, c, h, w in ((1, 1, 6, 5), (2, 3, 9, 7), (1, 37, 8, 11), (3, 130, 6, 6)):
        announce("plane mean %s %s %s %s" % (mode, kind, window, (n, c, h, w)))

        def build(b):
            pool = b.maxpool if kind == "max" else b.avgpool
            y = pool(b.leaky_relu(b.arg("x", (n, c, h, w)), 0.25, name="a"), window, step, (pad,) * 4, name="p")
            b.output(b.reduce_mean(y, (2, 3), True, name="m"), "mean")

        check(build, {"x": image(n, c, h, w)}, mode, 1)


@pytest.mark.parametrize("mode", KW)
@pytest.mark.parametrize("kind", ["max", "avg"])
@pytest.mark.parametrize("window,step", [(1, 11), (1, 12), (1, 22), (2, 11), (2, 12)])
def test_steps_beyond_ten(kind, window, step, mode):
    """Small windows with steps whose digits, behind the window's, are those of a compiled window."""
    for n, c, h, w in ((1, 3, 48, 48), (2, 5, 36, 91)):
        announce("plane steps %s %s %d %d %s" % (mode, kind, window, step, (n, c, h, w)))

        def build(b):
            pool = b.maxpool if kind == "max" else b.avgpool
            y = pool(b.leaky_relu(b.arg("x", (n, c, h, w)), 0.25, name="a"), (window,) * 2, (step,) * 2, (0,) * 4, name="p")
            b.output(y, "pool")
            b.output(b.reduce_mean(y, (2, 3), True, name="m"), "mean")

        check(build, {"x": image(n, c, h, w)}, mode, 1)


@pytest.mark.parametrize("mode", KW)
def test_places_and_shapes(mode):
    """A value that is a result, a part of two Concats and read by a window; resizes up, down and to odd sizes."""
    for n, c, h, w in ((1, 3, 5, 4), (2, 6, 13, 9), (1, 16, 40, 31), (2, 65, 7, 7)):
        announce("plane places %s %s" % (mode, (n, c, h, w)))

        def build(b):
            x, z = b.arg("x", (n, c, h, w)), b.arg("z", (n, c, h, w))
            s = b.mul(b.sub(x, z, name="d"), x, name="s")
            y = b.relu(s, name="y")
            b.output(y, "y")
            b.output(b.concat([y, s], 1, name="c1"), "c1")
            b.output(b.concat([s, b.maxpool(y, (3, 3), (1, 1), (1, 1, 1, 1), name="p"), y], 1, name="c2"), "c2")
            b.output(b.resize_nearest(y, (2 * h + 1, 3 * w), name="up"), "up")
            b.output(b.resize_nearest(y, (max(1, h // 2), max(1, w // 3)), name="down"), "down")

        check(build, {"x": image(n, c, h, w), "z": image(n, c, h, w, seed=4)}, mode, 1)


@pytest.mark.parametrize("mode", KW)
def test_batchnorm_chunks(mode):
    """Affine maps across the planes of a chunk, the last chunk ragged; planes of exactly four elements; the largest planes."""
    r = np.random.default_rng(8)
    for n, c, h, w in ((3, 517, 2, 2), (2, 61, 7, 7), (1, 7, 75, 75), (1, 3, 190, 200)):
        announce("plane batchnorm %s %s" % (mode, (n, c, h, w)))
        m, v, g, o = (t.astype(np.float32) for t in (r.standard_normal(c), r.random(c) + 0.5, r.standard_normal(c), r.standard_normal(c)))

        def build(b):
            x = b.arg("x", (n, c, h, w))
            y = b.sigmoid(b.batchnorm(x, b.const("m", m), b.const("v", v), 1e-5, b.const("g", g), b.const("o", o), name="bn"), name="act")
            b.output(b.avgpool(y, (2, 2), (1, 1), (0, 0, 0, 0), name="p"), "p")
            b.output(b.add(y, x, name="r"), "r")

        check(build, {"x": image(n, c, h, w)}, mode, 1)


def test_other_routes():
    """Planes beyond the LDS, and values that a convolution reads, run as before."""
    def tall(b):
        y = b.relu(b.arg("x", (1, 2, 310, 300)), name="a")
        b.output(b.maxpool(y, (3, 3), (2, 2), (1, 1, 1, 1), name="p"), "p")

    check(tall, {"x": image(1, 2, 310, 300)}, "fp32", None, grouped=False)
    w = image(8, 8, 1, 1)

    def net(b):
        y = b.maxpool(b.relu(b.arg("x", (2, 8, 12, 12)), name="a"), (2, 2), (2, 2), (0, 0, 0, 0), name="p")
        b.output(b.conv(y, b.const("w", w), name="c"), "c")

    check(net, {"x": image(2, 8, 12, 12)}, "fp32", None, ops=32, grouped=False)
