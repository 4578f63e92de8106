"""The small-tile implicit-GEMM kernels (16x16 and 32x32 tiles with K split over a
workgroup's wavefronts, 64x64 tiles with both operands in LDS), forced for every
launch: the convolution sweeps and requantisation cases at the parity bar of the
other kernels, and products at the edges of the tiles and of the K split (one row,
fewer K steps than wavefronts, a partial last step, ragged rows and columns)."""
import numpy as np
import pytest

import test_gpu_conv_sweep as sweep
import test_gpu_int8 as q8
from test_gpu_taps_kernel import run_logged
from util import announce, run_both

pytestmark = pytest.mark.gpu

TILES = {"slim1": "16x16k16", "slim2": "32x32k8", "mid": "64x64"}


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("mode", ["fp32", "fp16", "bf16"])
def test_float_convolution_sweep(tile, mode, monkeypatch):
    monkeypatch.setenv("ODLA_HIP_IGEMM_TILE", tile)
    sweep.test_random_convolutions(mode)


@pytest.mark.parametrize("tile", TILES)
def test_int8_sweep_and_requantisation(tile, monkeypatch, odla, ref):
    monkeypatch.setenv("ODLA_HIP_IGEMM_TILE", tile)
    sweep.test_random_convolutions_int8()
    for case in q8.Q8_CONV_CASES:
        q8.test_q8_conv_accumulators_and_requant(case, odla, ref)


EDGES = [(1, 16, 16), (1, 1000, 2048), (15, 17, 40), (16, 16, 64), (17, 33, 72), (31, 65, 1024), (33, 32, 1032), (64, 64, 128),
         (65, 63, 3072), (129, 200, 264)]


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("mode", ["fp32", "fp16", "bf16"])
def test_product_edges(tile, mode, monkeypatch):
    """[M, K] x [K, N] + bias -> GELU, and the same with a residual and LeakyReLU."""
    monkeypatch.setenv("ODLA_HIP_IGEMM_TILE", tile)
    r = np.random.default_rng(9)
    tol = {"fp32": 1e-4, "fp16": 2e-2, "bf16": 6e-2}[mode]
    for M, N, K in EDGES:
        announce("%s %s %s" % (tile, mode, (M, N, K)))
        x = r.standard_normal((M, K)).astype(np.float32)
        w = (r.standard_normal((K, N)) / np.sqrt(K)).astype(np.float32)
        bias = r.standard_normal((N,)).astype(np.float32)
        res = r.standard_normal((M, N)).astype(np.float32)

        def build(b):
            v, t = b.arg("x", (M, K)), b.arg("res", (M, N))
            y = b.gemm(v, b.const("w", w), b.const("b", bias), False, False, 1.0, 1.0, name="g")
            b.output(b.gelu(y, False, name="gelu"), "gelu")
            y2 = b.add(b.gemm(v, b.const("w2", w), None, False, False, 1.0, 0.0, name="h"), t, name="hr")
            b.output(b.leaky_relu(y2, 0.1, name="leaky"), "leaky")

        (got, want), seen = run_logged(lambda: run_both(build, {"x": x, "res": res}, fp16=mode == "fp16", bf16=mode == "bf16"))
        if K * (4 if mode == "fp32" else 2) < 2048:   # (longer ones may be planned as split products)
            assert any(m.endswith("kernel " + TILES[tile]) for m in seen), [m for m in seen if "kernel" in m]
        for k in want:
            assert np.max(np.abs(got[k] - want[k])) <= tol * max(1.0, float(np.max(np.abs(want[k])))), (M, N, K, k)
