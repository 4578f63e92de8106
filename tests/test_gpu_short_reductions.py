"""Means over short axes with few columns (a global pool behind a backbone): whole and ragged column groups, axes below
and above the length from which they are cut into slices, fp32 / fp16 against 64-bit sums and 8-bit ones to the bit;
and a classifier's result that a later launch reads, written in the caller's buffer."""
import ctypes

import numpy as np
import pytest

import __graft_entry__ as entry
from test_plan_layernorm_cpu import steps_of
from util import announce, run_hip, run_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp16", [False, True])
@pytest.mark.parametrize("outer,length,inner", [(1, 8, 16), (1, 49, 2048), (3, 49, 528), (13, 64, 2048), (2, 33, 136), (1, 127, 1000), (1, 128, 1000),
                                                (5, 100, 72), (40, 49, 512), (257, 32, 64)])
def test_mean_over_a_short_axis(odla, outer, length, inner, fp16):
    announce("short mean %d x %d x %d fp16=%s" % (outer, length, inner, fp16))
    x = np.random.default_rng(length * 7 + inner).standard_normal((outer, length, inner)).astype(np.float32)

    def build(b):
        t = b.arg("x", x.shape)
        b.output(b.reduce_mean(t, (1,), False, name="m"), "y")

    got = run_hip(build, {"x": x}, fp16=fp16)["y"]
    x64 = (x.astype(np.float16) if fp16 else x).astype(np.float64)
    # sums of `length` terms in 32 bits, and the stored result's rounding
    bound = length * 2.0 ** -24 * np.abs(x64).mean(1).max() + (2.0 ** -11 * np.abs(x64.mean(1)).max() if fp16 else 2.0 ** -23)
    assert np.max(np.abs(got - x64.mean(1))) <= bound


@pytest.mark.parametrize("n,hw,c", [(1, 3, 64), (1, 7, 2048), (13, 8, 512), (2, 7, 528), (3, 11, 64), (2, 12, 256), (300, 7, 64)])
def test_mean_of_8_bit_levels(odla, n, hw, c):
    announce("8-bit mean %d x %d^2 x %d" % (n, hw, c))
    ref, models = entry.load_oracle(), entry.load().models
    r = np.random.default_rng(hw * 5 + c)
    x = r.standard_normal((n, 16, hw, hw)).astype(np.float32)
    k = (r.standard_normal((c, 16, 1, 1)) * 0.3).astype(np.float32)
    x_rng, y_rng = (float(x.min()), float(x.max())), (-2.0, 3.0)
    x_qp, y_qp = ref.act_qparams(*x_rng), ref.act_qparams(*y_rng)
    entries = [(name, *models.act_qparams(*rng), *rng, None) for name, rng in (("x", x_rng), ("c", y_rng))]
    wt = k.reshape(c, -1)
    entries.append(("w", 1.0, 0, float(wt.min()), float(wt.max()), list(zip(wt.min(axis=1).tolist(), wt.max(axis=1).tolist()))))
    table = odla.quant_table(entries)

    def build(b):
        t = b.conv(b.arg("x", x.shape), b.const("w", k), None, (1, 1), (0, 0, 0, 0), name="c")
        b.output(b.reduce_mean(t, (2, 3), True, name="m"), "y")

    got = run_hip(build, {"x": x}, quant_table=table)["y"].reshape(n, c)
    q, _ = ref.qconv(ref.quantize_act(x, *x_qp), x_qp, k, np.zeros(c, np.float32), y_qp, (1, 1), (0, 0, 0, 0), relu=False)
    scale, zp = np.float32(y_qp[0]), int(y_qp[1])
    total = np.asarray(q).astype(np.int64).reshape(n, c, -1).sum(2) - zp * hw * hw
    want = (total.astype(np.float32) / np.float32(hw * hw)) * scale
    assert np.array_equal(got, want)


@pytest.mark.parametrize("rows", [3, 200, 300])
def test_scores_that_a_later_launch_reads(odla, rows):
    """The product is written where the caller bound it; the probabilities come from there."""
    announce("scores in place, %d rows" % rows)
    r = np.random.default_rng(rows)
    w = (r.standard_normal((2048, 1000)) * 0.02).astype(np.float32)

    def build(b):
        t = b.gemm(b.arg("x", (rows, 2048)), b.const("w", w), name="mm")
        b.output(t, "scores")
        b.output(b.softmax(t, -1, name="sm"), "prob")

    if rows >= 200:
        assert any(s.startswith("gemm.sum") for s in steps_of(odla, build))
    hb = odla.HipBuilder()
    build(hb)
    s = hb.session(True)
    for _ in range(3):
        feeds = {"x": r.standard_normal((rows, 2048)).astype(np.float32)}
        want = run_ref(build, feeds)
        s.bind_device_io(feeds)
        s.execute()
        for name, (p, shape, dt) in s.dev_out.items():
            got = np.empty(shape, dt)
            assert s.L.odla_CopyMemory(got.ctypes.data_as(ctypes.c_void_p), p, got.nbytes, odla.ODLA_MEMCPY_D2H) == 0
            np.testing.assert_allclose(got, want[name], rtol=2e-4, atol=2e-5)
    s.close()
    hb.destroy()
