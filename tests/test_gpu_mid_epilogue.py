"""The 64 x 64 tile's epilogue: blocks of 32 channels that end inside the result or past it, rows
whose pitch allows no vectors, a residual in every result type, results addressed as attention
heads, and the 8-bit residual block bit-equal to the oracle."""
import numpy as np
import pytest

import test_gpu_int8 as q8
from test_gpu_taps_kernel import run_logged
from util import announce, run_both

pytestmark = pytest.mark.gpu

MODES = {"fp32": {}, "fp16": {"fp16": True}, "bf16": {"bf16": "performance"}, "bf16acc": {"bf16": "accuracy"}}


@pytest.mark.parametrize("dims", [(1, 32, 8, 8, 64), (3, 64, 9, 7, 96), (2, 128, 5, 5, 160), (2, 64, 6, 6, 256)])
def test_8bit_residual_block(dims, odla, ref, monkeypatch):
    monkeypatch.setenv("ODLA_HIP_IGEMM_TILE", "mid")
    q8.test_q8_residual_fused_equals_unfused_equals_oracle(dims, 0, odla, ref, monkeypatch)


@pytest.mark.parametrize("mode", MODES)
def test_residual_and_activation_in_either_order(mode, monkeypatch):
    monkeypatch.setenv("ODLA_HIP_IGEMM_TILE", "mid")
    r = np.random.default_rng(2)
    eps = {"fp32": 2.0 ** -24, "fp16": 2.0 ** -11, "bf16": 2.0 ** -9, "bf16acc": 2.0 ** -9}[mode]
    for m, n, k in ((1, 32, 64), (63, 64, 72), (65, 96, 128), (130, 33, 256), (200, 100, 64), (64, 8, 512)):
        announce("mid epilogue %s %s" % (mode, (m, n, k)))
        x, res = r.standard_normal((m, k)).astype(np.float32), r.standard_normal((m, n)).astype(np.float32)
        w, bias = (r.standard_normal((k, n)) / np.sqrt(k)).astype(np.float32), r.standard_normal((n,)).astype(np.float32)

        def build(b):
            v, t = b.arg("x", (m, k)), b.arg("res", (m, n))
            y = b.gemm(v, b.const("w", w), b.const("b", bias), False, False, 1.0, 1.0, name="g")
            b.output(b.relu(b.add(y, t, name="a"), name="out1"), "relu")
            y2 = b.gemm(v, b.const("w2", w[:, ::-1].copy()), b.const("b2", bias), False, False, 1.0, 1.0, name="h")
            b.output(b.add(b.leaky_relu(y2, 0.25, name="l"), t, name="out2"), "late")

        (got, want), seen = run_logged(lambda: run_both(build, {"x": x, "res": res}, **MODES[mode]))
        assert any(s.endswith("kernel 64x64") for s in seen), [s for s in seen if "kernel" in s]
        for key in want:
            # operands rounded (rms 1 products, k / sqrt(k)^2 = 1 in all: five deviations of two roundings),
            # result and residual rounded, 32-bit sums
            tol = 5 * (2 * eps + 2.0 ** -24 * np.sqrt(k)) + 2 * eps * np.max(np.abs(want[key]))
            assert np.max(np.abs(got[key] - want[key])) <= tol, (m, n, k, key)


@pytest.mark.parametrize("mode", ["fp16", "bf16", "bf16acc"])
def test_projection_into_heads(mode, monkeypatch):
    """[B * S, heads * d] stored as [B, heads, S, d]."""
    monkeypatch.setenv("ODLA_HIP_IGEMM_TILE", "mid")
    monkeypatch.setenv("ODLA_HIP_FUSED_ATTENTION", "0")
    r = np.random.default_rng(4)
    for bs, s, heads, d in ((2, 7, 3, 32), (1, 41, 2, 64), (3, 33, 2, 8)):
        h = heads * d
        x = r.standard_normal((bs * s, h)).astype(np.float32)
        w = (r.standard_normal((h, h)) / np.sqrt(h)).astype(np.float32)

        def build(b):
            y = b.gemm(b.arg("x", (bs * s, h)), b.const("w", w), None, False, False, 1.0, 0.0, name="q")
            t = b.transpose(b.reshape(y, (bs, s, heads, d), name="r"), (0, 2, 1, 3), name="t")
            b.output(b.tanh(t, name="o"), "o")

        got, want = run_both(build, {"x": x}, **MODES[mode])
        eps = 2.0 ** -11 if mode == "fp16" else 2.0 ** -9
        assert np.max(np.abs(got["o"] - want["o"])) <= 5 * 2 * eps + 2 * eps * 4, (bs, s, heads, d)
