"""Two pointwise convolutions in one launch (64 channels to 128 or 256 with residual and activation, those to 64 or
128) against the oracle and, to the bit, against the two launches: ragged pixel counts, one pixel, more tiles than wavefronts; the
wide result is read elsewhere too; forms that stay apart."""
import numpy as np
import pytest

from test_plan_layernorm_cpu import steps_of
from util import announce, run_hip, run_ref

pytestmark = pytest.mark.gpu

MODES = {"fp16": ({"fp16": True}, 2.0 ** -11), "bf16": ({"bf16": "performance"}, 2.0 ** -8)}


def builder(n, h, w, wide, narrow, residual, act, stride=1, narrow_residual=False):
    r = np.random.default_rng(n * 31 + h * 7 + w + wide + narrow)
    k1 = (r.standard_normal((wide, 64, 1, 1)) / 8).astype(np.float32)
    k2 = (r.standard_normal((narrow, wide, 1, 1)) / 16).astype(np.float32)
    b1, b2 = r.standard_normal(wide).astype(np.float32), r.standard_normal(narrow).astype(np.float32)
    feeds = {"x": r.standard_normal((n, 64, h, w)).astype(np.float32)}
    if residual:
        feeds["r"] = r.standard_normal((n, wide, h, w)).astype(np.float32)

    def build(b):
        t = b.conv(b.arg("x", feeds["x"].shape), b.const("k1", k1), b.const("b1", b1), name="c1")
        if residual:
            t = b.add(t, b.arg("r", feeds["r"].shape), name="s")
        if act[0]:
            t = b.relu(t, name="y_act")
        z = b.conv(t, b.const("k2", k2), b.const("b2", b2) if narrow != 64 else None, stride=(stride, stride), name="c2")
        if act[1]:
            z = b.relu(z, name="z_act")
        b.output(t, "y")
        b.output(z, "z")
    return build, feeds


def one_order(monkeypatch, pixels):
    """Fewer pixels than one launch is ever taken for: the layers' own launches would be small tiles, which split K
    between wavefronts.  The tiles that walk K in one order, as one launch of both does, stand in for them."""
    if pixels < 1 << 15:
        monkeypatch.setenv("ODLA_HIP_WREG_KSPLIT", "0")


def rides(odla, build, kw):
    return any("+" in s for s in steps_of(odla, build, **kw) if s.startswith("conv:"))


@pytest.mark.parametrize("mode", sorted(MODES))
@pytest.mark.parametrize("n,h,w,wide,narrow,residual,act", [(1, 1, 1, 256, 64, True, (1, 1)), (2, 5, 7, 256, 128, True, (1, 1)), (1, 31, 33, 128, 64, False, (0, 1)), (3, 56, 56, 256, 64, True, (1, 1)),
                                                            (7, 56, 55, 256, 128, False, (1, 0)), (30, 56, 56, 256, 64, True, (0, 0)), (25, 57, 60, 128, 128, True, (1, 1)), (600, 4, 4, 256, 64, False, (1, 1))])
def test_two_layers_in_one_launch(odla, monkeypatch, mode, n, h, w, wide, narrow, residual, act):
    announce("pair %s %d x %d x %d, %d then %d" % (mode, n, h, w, wide, narrow))
    kw, eps = MODES[mode]
    one_order(monkeypatch, n * h * w)
    build, feeds = builder(n, h, w, wide, narrow, residual, act)
    monkeypatch.setenv("ODLA_HIP_PAIR_MIN_PIXELS", "1")
    assert rides(odla, build, kw)
    got = run_hip(build, feeds, **kw)
    monkeypatch.setenv("ODLA_HIP_PAIR_MIN_PIXELS", str(1 << 40))
    assert not rides(odla, build, kw)
    apart, want = run_hip(build, feeds, **kw), run_ref(build, feeds)
    for name, k in (("y", 64), ("z", wide)):
        # operands of k products and the result rounded once each (the second layer's operand is the first's result)
        bound = eps * (2 * np.sqrt(k) + 4) * max(1.0, float(np.max(np.abs(want[name]))))
        assert np.max(np.abs(got[name] - want[name])) <= bound
        np.testing.assert_array_equal(got[name], apart[name])


def shortcut(n, h, w, wide, narrow, act=False, twice=False):
    r = np.random.default_rng(n * 13 + h + w + wide)
    shape = (n, 64, h, w)
    ks = [(r.standard_normal((c, i, 1, 1)) * s).astype(np.float32) for c, i, s in ((wide, 64, 0.1), (64, 64, 0.12), (wide, 64, 0.1), (narrow, wide, 0.06))]
    bs = [r.standard_normal(k.shape[0]).astype(np.float32) for k in ks]

    def build(b):
        x = b.arg("x", shape)
        x = b.relu(b.maxpool(x, (3, 3), (1, 1), (1, 1, 1, 1), name="front"), name="front_act")
        conv = lambda t, k, name: b.conv(t, b.const("k%d" % k, ks[k]), b.const("b%d" % k, bs[k]), name=name)
        s = conv(x, 0, "short")
        if act:
            s = b.relu(s, name="short_act")
        t = b.relu(conv(x, 1, "c1"), name="c1_act")
        y = b.relu(b.add(conv(t, 2, "c2"), s, name="sum"), name="y_act")
        b.output(y, "y")
        b.output(b.relu(conv(y, 3, "c3"), name="z_act"), "z")
        if twice:
            b.output(b.relu(s, name="s2"), "s")
    return build, {"x": r.standard_normal(shape).astype(np.float32)}


@pytest.mark.parametrize("mode", sorted(MODES))
@pytest.mark.parametrize("n,h,w,wide,narrow,form", [(1, 1, 1, 256, 64, ""), (2, 5, 7, 128, 64, ""), (3, 56, 56, 256, 64, ""), (23, 57, 55, 256, 64, ""), (41, 45, 47, 128, 64, ""),
                                                    (2, 20, 21, 256, 128, "apart"), (2, 20, 21, 256, 64, "act"), (2, 20, 21, 256, 64, "twice")])
def test_the_residual_is_a_layer_too(odla, monkeypatch, mode, n, h, w, wide, narrow, form):
    """Three layers in one launch; apart (the residual is written and read) where it does not fit or is read elsewhere."""
    announce("pair with shortcut %s %d x %d x %d, %d then %d %s" % (mode, n, h, w, wide, narrow, form))
    kw, eps = MODES[mode]
    one_order(monkeypatch, n * h * w)
    build, feeds = shortcut(n, h, w, wide, narrow, form == "act", form == "twice")
    monkeypatch.setenv("ODLA_HIP_PAIR_MIN_PIXELS", "1")
    names = steps_of(odla, build, **kw)
    assert any(s.count("+") == (1 if form else 2) for s in names if s.startswith("conv:")) and ("conv:short" in names) == (form in ("apart", "twice"))
    got = run_hip(build, feeds, **kw)
    monkeypatch.setenv("ODLA_HIP_PAIR_MIN_PIXELS", str(1 << 40))
    apart, want = run_hip(build, feeds, **kw), run_ref(build, feeds)
    for name in want:
        size = max(1.0, float(np.max(np.abs(want[name]))))
        # three roundings of operands and results in a row
        assert np.max(np.abs(got[name] - want[name])) <= 3 * eps * (2 * np.sqrt(wide) + 4) * size
        np.testing.assert_array_equal(got[name], apart[name])


@pytest.mark.parametrize("form", ["fp32", "accuracy", "stride", "wide_512", "narrow_96"])
def test_forms_that_stay_apart(odla, monkeypatch, form):
    monkeypatch.setenv("ODLA_HIP_PAIR_MIN_PIXELS", "1")
    kw = {"fp32": {}, "accuracy": {"bf16": "accuracy"}}.get(form, {"fp16": True})
    build, feeds = builder(2, 12, 10, 512 if form == "wide_512" else 256, 96 if form == "narrow_96" else 64, True, (1, 1), stride=2 if form == "stride" else 1)
    assert not rides(odla, build, kw)
    got, want = run_hip(build, feeds, **kw), run_ref(build, feeds)
    for name in want:
        assert np.max(np.abs(got[name] - want[name])) <= 3e-2 * max(1.0, float(np.max(np.abs(want[name]))))
