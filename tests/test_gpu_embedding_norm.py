"""Rows of a table plus positions, normalised by one launch, against the launches it stands for (the same graph with the
sum as a result too); a LayerNorm whose only reader is the caller writes fp32; forms that keep their launches."""
import numpy as np
import pytest

from test_plan_layernorm_cpu import steps_of
from util import announce, run_hip, run_ref

pytestmark = pytest.mark.gpu

MODES = {"fp32": {}, "fp16": {"fp16": True}, "bf16": {"bf16": "performance"}, "bf16acc": {"bf16": "accuracy"}}


def embedding(shape, h, pos_shape, words=37, swap=False, sum_too=False, more=False, scale=True):
    r = np.random.default_rng(h + len(pos_shape))
    table = r.standard_normal((words, h)).astype(np.float32)
    pos = r.standard_normal(pos_shape).astype(np.float32)
    g, o = (1 + 0.2 * r.standard_normal(h)).astype(np.float32), (0.1 * r.standard_normal(h)).astype(np.float32)

    def build(b):
        t = b.gather(b.const("table", table), b.arg("ids", shape, np.int32), 0, name="rows")
        p = b.const("pos", pos)
        t = b.add(p, t, name="sum") if swap else b.add(t, p, name="sum")
        y = b.layernorm(t, 1, 1e-5, b.const("g", g) if scale else None, b.const("o", o) if scale else None, name="ln")
        if sum_too:
            b.output(t, "sum")
        if more:
            y = b.relu(y, name="act")
        b.output(y, "y")

    ids = r.integers(-words, words, shape).astype(np.int32)
    ids.flat[0], ids.flat[-1] = words + 5, -words - 3      # (beyond the table: its nearest row)
    return build, {"ids": ids}


@pytest.mark.parametrize("mode", sorted(MODES))
@pytest.mark.parametrize("shape,h,pos_shape,swap,more", [((1, 41), 768, (41, 768), False, False), ((3, 7), 64, (7, 64), True, True), ((2, 5, 3), 520, (3, 520), False, True),
                                                         ((6,), 1024, (1024,), False, False), ((2, 9), 256, (2, 9, 256), True, False), ((70, 33), 8, (1, 33, 8), False, True)])
def test_embedding_is_one_launch(odla, mode, shape, h, pos_shape, swap, more):
    announce("embedding %s %s x %d %s" % (mode, shape, h, pos_shape))
    kw = MODES[mode]
    one, feeds = embedding(shape, h, pos_shape, swap=swap, more=more, scale=h != 64)
    apart, _ = embedding(shape, h, pos_shape, swap=swap, more=more, scale=h != 64, sum_too=True)
    assert any(s.startswith("embed+layernorm") for s in steps_of(odla, one, **kw))
    assert any(s.startswith("gather") for s in steps_of(odla, apart, **kw))
    np.testing.assert_array_equal(run_hip(one, feeds, **kw)["y"], run_hip(apart, feeds, **kw)["y"])


@pytest.mark.parametrize("mode", ["fp16", "bf16"])
@pytest.mark.parametrize("rows,h", [(1, 8), (41, 768), (300, 1032), (5, 2048), (3, 2056), (4, 36)])
def test_last_layernorm_writes_the_declared_type(odla, mode, rows, h):
    announce("last layernorm %s %d x %d" % (mode, rows, h))
    r = np.random.default_rng(rows + h)
    x = r.standard_normal((rows, h)).astype(np.float32)
    g = (1 + 0.2 * r.standard_normal(h)).astype(np.float32)

    def build(extra):
        def b_(b):
            t = b.layernorm(b.arg("x", x.shape), 1, 1e-5, b.const("g", g), None, name="ln")
            b.output(t, "y")
            if extra:
                b.output(b.relu(t, name="r"), "r")
        return b_

    kw = MODES[mode]
    whole = h % 8 == 0 and h <= 2048
    assert any(s.startswith("out.cast") for s in steps_of(odla, build(False), **kw)) != whole
    got, apart = run_hip(build(False), {"x": x}, **kw)["y"], run_hip(build(True), {"x": x}, **kw)["y"]
    np.testing.assert_array_equal(got, apart)
    assert np.max(np.abs(got - run_ref(build(False), {"x": x})["y"])) <= (2.0 ** -9 if mode == "fp16" else 2.0 ** -6) * 6


@pytest.mark.parametrize("form", ["sum_too", "arg_pos", "two_axes"])
def test_forms_that_keep_their_launches(odla, form):
    r = np.random.default_rng(3)
    table, pos, ids = r.standard_normal((9, 64)).astype(np.float32), r.standard_normal((5, 64)).astype(np.float32), r.integers(0, 9, (2, 5)).astype(np.int32)
    feeds = {"ids": ids}

    def build(b):
        t = b.gather(b.const("table", table), b.arg("ids", ids.shape, np.int32), 0, name="rows")
        p = b.arg("pos", pos.shape) if form == "arg_pos" else b.const("pos", pos)
        t = b.add(t, p, name="sum")
        if form == "two_axes":
            n = (np.ones((5, 64), np.float32), np.zeros((5, 64), np.float32))
        else:
            n = (np.ones(64, np.float32), np.zeros(64, np.float32))
        b.output(b.layernorm(t, 2 if form == "two_axes" else 1, 1e-5, b.const("g", n[0]), b.const("o", n[1]), name="ln"), "y")
        if form == "sum_too":
            b.output(t, "sum")

    if form == "arg_pos":
        feeds["pos"] = pos
    assert not any(s.startswith("embed") for s in steps_of(odla, build))
    np.testing.assert_allclose(run_hip(build, feeds)["y"], run_ref(build, feeds)["y"], rtol=1e-4, atol=1e-5)
