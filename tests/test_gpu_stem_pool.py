"""A 7x7 / stride 2 convolution over three channels, ReLU and 3x3 / stride 2 maximum in one launch: odd and even
images, images smaller than a filter, strips of one, two and four pooled rows, more than four column groups; against
the oracle (fp16, bf16) and, to the bit, its integer accumulation and requantisation (int8)."""
import numpy as np
import pytest

import __graft_entry__ as entry
from stem_concat_graphs import CONCATS, concat_graph
from test_plan_layernorm_cpu import steps_of
from util import announce, run_hip, run_ref

pytestmark = pytest.mark.gpu

#        N, H, W
SIZES = [(1, 2, 2), (1, 3, 7), (2, 9, 11), (2, 45, 37), (3, 64, 50), (1, 224, 224), (13, 237, 237), (5, 33, 400),
         (40, 97, 96), (300, 58, 61)]


def data(n, h, w, seed):
    r = np.random.default_rng(seed)
    x = r.standard_normal((n, 3, h, w)).astype(np.float32)
    k = (r.standard_normal((64, 3, 7, 7)) * 0.12).astype(np.float32)
    return x, k, r.standard_normal(64).astype(np.float32) * 0.3


def builder(shape, k, bias):
    def build(b):
        t = b.conv(b.arg("x", shape), b.const("w", k), None if bias is None else b.const("b", bias), (2, 2), (3, 3, 3, 3), name="y")
        t = b.maxpool(b.relu(t, name="t"), (3, 3), (2, 2), (1, 1, 1, 1), name="p")
        b.output(b.relu(t, name="out_relu"), "out")
    return build


def one_launch(odla, build, **kw):
    return any(s.startswith("stem:") for s in steps_of(odla, build, **kw))


@pytest.mark.parametrize("mode", ["fp16", "bf16"])
@pytest.mark.parametrize("n,h,w", SIZES)
def test_stem_pool_float(odla, n, h, w, mode):
    announce("stem and pool %s %d x %d x %d" % (mode, n, h, w))
    x, k, bias = data(n, h, w, h * 7 + w)
    kw = {"fp16": {"fp16": True}, "bf16": {"bf16": "performance"}}[mode]
    build = builder(x.shape, k, None if h == 45 else bias)
    assert one_launch(odla, build, **kw)
    got, want = run_hip(build, {"x": x}, **kw)["out"], run_ref(build, {"x": x})["out"]
    # operands of 147 products and the result rounded once each, largest of nine
    eps = 2.0 ** -11 if mode == "fp16" else 2.0 ** -8
    assert got.shape == want.shape
    assert np.max(np.abs(got - want)) <= eps * (2 * np.sqrt(147) + 1) * max(1.0, float(np.max(np.abs(want))))


@pytest.mark.parametrize("n,h,w", SIZES)
@pytest.mark.parametrize("y_rng", [(-2.5, 4.0), (0.0, 3.0)])
def test_stem_pool_int8(odla, n, h, w, y_rng):
    announce("stem and pool int8 %d x %d x %d" % (n, h, w))
    ref, models = entry.load_oracle(), entry.load().models
    x, k, bias = data(n, h, w, h * 5 + w)
    x = (x * 1.5 + 0.3).astype(np.float32)
    x_rng = (float(x.min()), float(x.max()))
    x_qp, y_qp = ref.act_qparams(*x_rng), ref.act_qparams(*y_rng)
    entries = [(name, *models.act_qparams(*rng), *rng, None) for name, rng in (("x", x_rng), ("t", y_rng))]
    wt = k.reshape(64, -1)
    entries.append(("w", 1.0, 0, float(wt.min()), float(wt.max()), list(zip(wt.min(axis=1).tolist(), wt.max(axis=1).tolist()))))
    table = odla.quant_table(entries)

    def build(b):
        t = b.conv(b.arg("x", x.shape), b.const("w", k), b.const("b", bias), (2, 2), (3, 3, 3, 3), name="y")
        b.output(b.maxpool(b.relu(t, name="t"), (3, 3), (2, 2), (1, 1, 1, 1), name="p"), "out")

    assert one_launch(odla, build, quant_table=table)
    got = run_hip(build, {"x": x}, quant_table=table)["out"]
    q, _ = ref.qconv(ref.quantize_act(x, *x_qp), x_qp, k, bias, y_qp, (2, 2), (3, 3, 3, 3), relu=True)
    c = ref.dequantize_act(q, *y_qp)
    p = np.pad(c, ((0, 0), (0, 0), (1, 2), (1, 2)), constant_values=-np.inf)
    ho, wo = got.shape[2:]
    want = np.max([p[:, :, i:i + 2 * ho:2, j:j + 2 * wo:2][:, :, :ho, :wo] for i in range(3) for j in range(3)], axis=0)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("mode", ["fp16", "int8"])
def test_stem_pool_infinities_and_nan(odla, mode):
    """Infinite pixels saturate as the largest levels do; results that are no number count as zero."""
    announce("stem and pool, infinite pixels %s" % mode)
    models = entry.load().models
    x, k, bias = data(2, 50, 46, 9)
    k = np.abs(k) if mode == "fp16" else k
    kw = {"fp16": True}
    if mode == "int8":
        entries = [(name, *models.act_qparams(*rng), *rng, None) for name, rng in (("x", (-2.0, 3.0)), ("t", (0.0, 4.0)))]
        wt = k.reshape(64, -1)
        entries.append(("w", 1.0, 0, float(wt.min()), float(wt.max()), list(zip(wt.min(axis=1).tolist(), wt.max(axis=1).tolist()))))
        kw = {"quant_table": odla.quant_table(entries)}

    def build(b):
        t = b.conv(b.arg("x", x.shape), b.const("w", k), b.const("b", bias), (2, 2), (3, 3, 3, 3), name="y")
        b.output(b.maxpool(b.relu(t, name="t"), (3, 3), (2, 2), (1, 1, 1, 1), name="p"), "out")

    assert one_launch(odla, build, **kw)
    special, plain = x.copy(), x.copy()
    special[0, 1, 20, 20], plain[0, 1, 20, 20] = np.inf, 1e30
    special[1, 2, 30, 11], plain[1, 2, 30, 11] = -np.inf, -1e30
    if mode == "int8":
        special[0, 0, 5, 5], plain[0, 0, 5, 5] = np.nan, -1e30
        assert np.array_equal(run_hip(build, {"x": special}, **kw)["out"], run_hip(build, {"x": plain}, **kw)["out"])
        return
    got = run_hip(build, {"x": special}, **kw)["out"]
    want = run_hip(build, {"x": x}, **kw)["out"]
    hit = np.isinf(got)
    assert not np.isnan(got).any() and hit[0].any() and not hit[1].any()
    # pooled rows and columns within reach of the pixel: 2 p - 1 .. 2 p + 1 of convolution rows 2 r - 3 .. 2 r + 3
    far = np.ones_like(hit)
    far[0, :, 4:7, 4:7] = far[1, :, 6:10, 1:5] = False
    assert np.array_equal(got[far], want[far])


def test_the_convolution_is_read_elsewhere_too(odla):
    """A second reader of the activation, or another window, keeps the launches apart."""
    x, k, bias = data(2, 40, 40, 3)

    def both(b):
        t = b.relu(b.conv(b.arg("x", x.shape), b.const("w", k), b.const("b", bias), (2, 2), (3, 3, 3, 3), name="y"), name="t")
        b.output(b.maxpool(t, (3, 3), (2, 2), (1, 1, 1, 1), name="p"), "p")
        b.output(b.relu(t, name="u"), "u")

    def window(b):
        t = b.relu(b.conv(b.arg("x", x.shape), b.const("w", k), b.const("b", bias), (2, 2), (3, 3, 3, 3), name="y"), name="t")
        b.output(b.maxpool(t, (2, 2), (2, 2), (0, 0, 0, 0), name="p"), "p")

    for build in (both, window):
        assert not one_launch(odla, build, fp16=True)
        got, want = run_hip(build, {"x": x}, fp16=True), run_ref(build, {"x": x})
        for name in want:
            assert np.max(np.abs(got[name] - want[name])) <= 2e-2 * max(1.0, float(np.max(np.abs(want[name]))))


@pytest.mark.parametrize("mode", ["fp16", "bf16"])
@pytest.mark.parametrize("n,h,w", [(1, 3, 7), (2, 45, 37), (40, 97, 96)])
@pytest.mark.parametrize("parts,one", CONCATS)
def test_stem_pool_as_a_part_of_a_concat(odla, parts, one, n, h, w, mode):
    """The pooled pixels are a slice of the Concat's, in front of, behind and between other parts."""
    announce("stem and pool in a concat %s %d x %d x %d %s" % (mode, n, h, w, parts))
    kw = {"fp16": {"fp16": True}, "bf16": {"bf16": "performance"}}[mode]
    build, feeds = concat_graph(n, h, w, parts)
    assert one_launch(odla, build, **kw) == one
    got, want = run_hip(build, feeds, **kw)["out"], run_ref(build, feeds)["out"]
    # operands of 147 products and the result rounded once each, largest of nine
    eps = 2.0 ** -11 if mode == "fp16" else 2.0 ** -8
    assert np.max(np.abs(got - want)) <= eps * (2 * np.sqrt(147) + 1) * max(1.0, float(np.max(np.abs(want))))
