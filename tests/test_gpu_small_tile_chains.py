"""The small-tile kernels at every length of a wavefront's share of K: none, fewer steps than a
batch, a batch, what lies between two and three, with a remainder and a partial last step; filters
of one tap and of nine, whose padding taps read nothing."""
import numpy as np
import pytest

from test_gpu_taps_kernel import run_logged
from util import announce, run_both

pytestmark = pytest.mark.gpu

# wavefronts of a workgroup, K steps of a batch
TILES = {"slim1": ("16x16k16", 16, 5), "slim2": ("32x32k8", 8, 3)}


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("mode,step", [("fp16", 32), ("fp32", 16)])
@pytest.mark.parametrize("taps", [1, 3])
def test_every_share_of_k(tile, mode, step, taps, monkeypatch):
    monkeypatch.setenv("ODLA_HIP_IGEMM_TILE", tile)
    kernel, waves, u = TILES[tile]
    r = np.random.default_rng(11)
    eps = {"fp16": 2.0 ** -11, "fp32": 2.0 ** -24}[mode]
    steps = sorted({waves * s + e for s in (0, 1, u - 1, u, u + 1, 2 * u - 1, 2 * u, 2 * u + 1, 3 * u, 4 * u + 1) for e in (0, waves // 2 + 1)} - {0})
    for n in steps:
        # whole steps, and a channel count that leaves the last one partial (8 of 16-byte vectors)
        for short in ((0, step // 4) if n % 2 else (0,)):
            c = max(step // 4, (n * step) // (taps * taps) // step * step - short)
            announce("%s %s taps %d steps %d channels %d" % (tile, mode, taps, n, c))
            k = c * taps * taps
            x = r.standard_normal((2, c, 3, 5)).astype(np.float32)
            w = (r.standard_normal((24, c, taps, taps)) / np.sqrt(k)).astype(np.float32)
            p = taps // 2

            def build(b):
                b.output(b.conv(b.arg("x", x.shape), b.const("w", w), b.const("b", w[:, 0, 0, 0].copy()), (1, 1), (p, p, p, p), name="y"), "out")

            (got, want), seen = run_logged(lambda: run_both(build, {"x": x}, fp16=mode == "fp16"))
            assert any(m.endswith("kernel " + kernel) for m in seen), [m for m in seen if "kernel" in m]
            # operands and result rounded once each (rms 1, |w| sums of k products of size 1/sqrt(k):
            # five standard deviations of the rounding errors), 32-bit sums in any order
            assert np.max(np.abs(got["out"] - want["out"])) <= 5 * (2 * eps + 2.0 ** -24 * np.sqrt(k)) + eps * np.max(np.abs(want["out"])), (n, c)
