"""The 128-channel tiles of 96 and 128 rows and their epilogue in the accumulator layout: rows past the last one, 32-channel blocks
past the last channel, every activation it branches on, a residual requested ahead of the K loop,
results addressed as attention heads, and the borders that keep the epilogue by rows."""
import math

import numpy as np
import pytest

import test_gpu_int8 as q8
from test_gpu_taps_kernel import run_logged
from util import announce, run_both

pytestmark = pytest.mark.gpu

MODES = {"fp32": {}, "fp16": {"fp16": True}, "bf16": {"bf16": "performance"}, "bf16acc": {"bf16": "accuracy"}}
EPS = {"fp32": 2.0 ** -24, "fp16": 2.0 ** -11, "bf16": 2.0 ** -9, "bf16acc": 2.0 ** -9}


def tolerance(mode, k, want):
    # operands rounded (rms 1 products, k / sqrt(k)^2 = 1 in all: five deviations of two roundings),
    # result and residual rounded, 32-bit sums; no activation here has a slope above 1.13
    return 1.13 * 5 * (2 * EPS[mode] + 2.0 ** -24 * np.sqrt(k)) + 2 * EPS[mode] * np.max(np.abs(want)) + 4e-7


def tile_forms(seen):
    return [s for s in seen if ": tiles of " in s]


@pytest.mark.parametrize("rows", ["96", "128"])
@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("act", ["none", "relu", "gelu", "sigmoid", "tanh"])
def test_ragged_tiles(rows, mode, act, monkeypatch):
    monkeypatch.setenv("ODLA_HIP_WREG_ROWS", rows)
    monkeypatch.setenv("ODLA_HIP_IGEMM_TILE", "wreg")
    r = np.random.default_rng(5)
    for m, n, k in ((1, 32, 64), (95, 96, 128), (97, 64, 64), (129, 160, 192), (300, 128, 64), (200, 100, 128)):
        announce("tile epilogue %s %s %s" % (mode, act, (m, n, k)))
        x = r.standard_normal((m, k)).astype(np.float32)
        w, bias = (r.standard_normal((k, n)) / np.sqrt(k)).astype(np.float32), r.standard_normal((n,)).astype(np.float32)

        def build(b):
            y = b.gemm(b.arg("x", (m, k)), b.const("w", w), b.const("b", bias), False, False, 1.0, 1.0, name="g")
            b.output(y if act == "none" else getattr(b, act)(y, name="o"), "o")

        (got, want), seen = run_logged(lambda: run_both(build, {"x": x}, **MODES[mode]))
        assert any("kernel 128x128w" in s for s in seen), [s for s in seen if "kernel" in s]
        form = tile_forms(seen)
        assert form and all("tiles of %s rows" % rows in s and ("accumulator" in s) == (n % 32 == 0) for s in form), form
        assert np.max(np.abs(got["o"] - want["o"])) <= tolerance(mode, k, want["o"]), (m, n, k)


@pytest.mark.parametrize("rows,groups", [("96", "0"), ("96", "2"), ("128", "0"), ("128", "2")])
@pytest.mark.parametrize("mode", MODES)
def test_residual_and_activation_in_either_order(mode, rows, groups, monkeypatch):
    """One K group and two (an even number of stages; an odd one keeps one)."""
    monkeypatch.setenv("ODLA_HIP_WREG_ROWS", rows)
    monkeypatch.setenv("ODLA_HIP_WREG_KSPLIT", groups)
    monkeypatch.setenv("ODLA_HIP_IGEMM_TILE", "wreg")
    r = np.random.default_rng(6)
    for m, n, k in ((1, 32, 256), (95, 96, 512), (193, 224, 192), (130, 100, 1024)):
        announce("tile epilogue %s residual %s" % (mode, (m, n, k)))
        x, res = r.standard_normal((m, k)).astype(np.float32), r.standard_normal((m, n)).astype(np.float32)
        w, bias = (r.standard_normal((k, n)) / np.sqrt(k)).astype(np.float32), r.standard_normal((n,)).astype(np.float32)

        def build(b):
            v, t = b.arg("x", (m, k)), b.arg("res", (m, n))
            y = b.gemm(v, b.const("w", w), b.const("b", bias), False, False, 1.0, 1.0, name="g")
            b.output(b.relu(b.add(y, t, name="a"), name="out1"), "relu")
            y2 = b.gemm(v, b.const("w2", w[:, ::-1].copy()), b.const("b2", bias), False, False, 1.0, 1.0, name="h")
            b.output(b.add(b.leaky_relu(y2, 0.25, name="l"), t, name="out2"), "late")

        (got, want), seen = run_logged(lambda: run_both(build, {"x": x, "res": res}, **MODES[mode]))
        assert any("kernel 128x128w" in s for s in seen), [s for s in seen if "kernel" in s]
        form = tile_forms(seen)
        stages = k * (4 if mode == "fp32" else 2) // 128
        assert form and all("tiles of %s rows" % rows in s and ("residual ahead" in s) == (n % 32 == 0) and
                            ("2 K groups" in s) == (groups == "2" and stages % 2 == 0) for s in form), form
        for key in want:
            assert np.max(np.abs(got[key] - want[key])) <= tolerance(mode, k, want[key]), (m, n, k, key)


@pytest.mark.parametrize("batch", [4, 5, 8, 9])
def test_residual_on_either_side_of_the_resident_workgroups(batch, monkeypatch):
    """256 workgroups, one per compute unit (residual ahead, in the accumulator layout), and more (by rows)."""
    monkeypatch.setenv("ODLA_HIP_IGEMM_TILE", "wreg")
    r = np.random.default_rng(7)
    x = r.standard_normal((batch, 64, 91, 90)).astype(np.float32)
    res = r.standard_normal((batch, 128, 91, 90)).astype(np.float32)
    w = (r.standard_normal((128, 64, 1, 1)) / 8).astype(np.float32)

    def build(b):
        y = b.conv(b.arg("x", x.shape), b.const("w", w), name="c")
        b.output(b.relu(b.add(y, b.arg("res", res.shape), name="a"), name="o"), "o")

    (got, want), seen = run_logged(lambda: run_both(build, {"x": x, "res": res}, fp16=True))
    form = tile_forms(seen)
    assert form and all(s.endswith("residual ahead" if batch == 4 else "results by rows") for s in form), form
    assert np.max(np.abs(got["o"] - want["o"])) <= tolerance("fp16", 64, want["o"])


@pytest.mark.parametrize("dims", [(1, 128, 8, 8, 64), (3, 128, 9, 7, 96), (2, 512, 5, 5, 160), (2, 256, 7, 7, 256)])
@pytest.mark.parametrize("groups", ["0", "2"])
def test_8bit_residual_block_in_tiles_of_96_rows(dims, groups, odla, ref, monkeypatch):
    """Bit-equal to the oracle."""
    monkeypatch.setenv("ODLA_HIP_IGEMM_TILE", "wreg")
    monkeypatch.setenv("ODLA_HIP_WREG_ROWS", "96")
    monkeypatch.setenv("ODLA_HIP_WREG_KSPLIT", groups)
    q8.test_q8_residual_fused_equals_unfused_equals_oracle(dims, 0, odla, ref, monkeypatch)


@pytest.mark.parametrize("mode", ["fp16", "bf16", "bf16acc"])
def test_projection_into_heads(mode, monkeypatch):
    """[B * S, heads * d] stored as [B, heads, S, d]."""
    monkeypatch.setenv("ODLA_HIP_IGEMM_TILE", "wreg")
    monkeypatch.setenv("ODLA_HIP_FUSED_ATTENTION", "0")
    r = np.random.default_rng(4)
    for bs, s, heads, d in ((2, 7, 2, 32), (1, 141, 2, 64), (3, 33, 8, 8)):
        h = heads * d
        x = r.standard_normal((bs * s, h)).astype(np.float32)
        w = (r.standard_normal((h, h)) / np.sqrt(h)).astype(np.float32)

        def build(b):
            y = b.gemm(b.arg("x", (bs * s, h)), b.const("w", w), None, False, False, 1.0, 0.0, name="q")
            t = b.transpose(b.reshape(y, (bs, s, heads, d), name="r"), (0, 2, 1, 3), name="t")
            b.output(b.tanh(t, name="o"), "o")

        got, want = run_both(build, {"x": x}, **MODES[mode])
        assert np.max(np.abs(got["o"] - want["o"])) <= tolerance(mode, h, want["o"]), (bs, s, heads, d)


@pytest.mark.parametrize("mode", ["fp16", "bf16"])
@pytest.mark.parametrize("tiles", ["", "1", "3"])
def test_nine_taps_of_one_vector(mode, tiles, monkeypatch):
    """3 x 3 filters over three channels (one 16-byte vector) in the short-tap kernel, at most 32 results."""
    monkeypatch.setenv("ODLA_HIP_IGEMM_TILE", "taps")
    if tiles:
        monkeypatch.setenv("ODLA_HIP_LEAN_TILES", tiles)
    r = np.random.default_rng(9)
    for n, h, w_, o, stride, pad in ((1, 5, 5, 32, 1, 1), (2, 31, 29, 32, 1, 1), (3, 26, 27, 17, 2, 1), (1, 40, 33, 8, 1, 0), (2, 3, 3, 32, 1, 2)):
        announce("nine taps %s %s" % (mode, (n, h, w_, o, stride, pad)))
        x = r.standard_normal((n, 3, h, w_)).astype(np.float32)
        w = (r.standard_normal((o, 3, 3, 3)) / np.sqrt(27)).astype(np.float32)
        bias = r.standard_normal((o,)).astype(np.float32)

        def build(b):
            y = b.conv(b.arg("x", x.shape), b.const("w", w), b.const("b", bias), (stride, stride), (pad,) * 4, (1, 1), 1, name="c")
            b.output(b.leaky_relu(y, 0.1, name="o"), "o")

        (got, want), seen = run_logged(lambda: run_both(build, {"x": x}, **MODES[mode]))
        assert any(s.endswith("kernel 128x64t") for s in seen) or stride == 2, [s for s in seen if "kernel" in s]
        assert np.max(np.abs(got["o"] - want["o"])) <= tolerance(mode, 27, want["o"]), (n, h, w_, o, stride, pad)


def test_gelu_over_its_range():
    """Against the exact function in 64 bits; infinities and NaN as x (1 + erf(x / sqrt 2)) / 2 has them."""
    special = np.array([np.inf, -np.inf, np.nan, 0.0, -0.0, 1e-30, -1e-30, 3e38, -3e38, 1e10, -1e10, 5.65, -5.65], np.float32)
    r = np.random.default_rng(8)
    x = np.concatenate([np.linspace(-14, 14, 200001), r.standard_normal(50000), special]).astype(np.float32)
    got = run_both(lambda b: b.output(b.gelu(b.arg("x", x.shape), False, name="o"), "o"), {"x": x})[0]["o"]
    n = x.size - special.size
    v = x[:n].astype(np.float64)
    want = v * 0.5 * np.array([math.erfc(-t / math.sqrt(2.0)) for t in v])
    err = np.abs(got[:n] - want)
    assert err.max() <= 4e-7
    near = v >= -5.65
    assert np.all(err[near] <= 4e-6 * np.abs(want[near]))
    tail = got[n:]
    assert tail[0] == np.inf and np.isnan(tail[1]) and np.isnan(tail[2])
    assert np.all(tail[3:5] == 0) and not np.signbit(tail[3]) and np.signbit(tail[4])
    assert np.allclose(tail[5:7], [5e-31, -5e-31], rtol=1e-6) and np.allclose(tail[[7, 9, 11]], special[[7, 9, 11]], rtol=1e-7)
    assert np.all(tail[[8, 10]] == 0) and -4.6e-8 * 1.00001 <= tail[12] <= -4.5e-8
