"""The one-launch attention kernel at sequence lengths that fill no 32-key block and at lengths
beyond one 128-key tile (running maximum and sum over the tiles): one launch per block, at the
parity bar of the lengths it served first."""
import numpy as np
import pytest

import test_gpu_attention as att
from util import announce, run_hip, run_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["bf16", "fp16", "bf16acc"])
@pytest.mark.parametrize("S", [1, 7, 31, 33, 41, 127, 129, 160, 255, 257, 384, 512, 600])
def test_attention_length(S, mode):
    att.test_attention_block((2, 3, S, 64, "div", True, True, True), mode)


def test_attention_tiles_masked_away():
    """Whole tiles of masked keys, in front and behind, with -inf as the mask value."""
    B, heads, S, d = 3, 2, 400, 64
    build = att.build_attention(B, heads, S, d, "div", True, True)
    f = att.feeds_for(B, heads, S, d, True, True, 3)
    f["mask"][:] = 0.0
    f["mask"][0, ..., :300] = -np.inf
    f["mask"][1, ..., 100:] = -np.inf
    announce("attention masked tiles")
    got = run_hip(build, f, bf16="performance")["out"]
    want = run_ref(build, f)["out"]
    assert np.all(np.isfinite(got))
    assert float(np.max(np.abs(got - want))) <= 2e-2 * max(1.0, float(np.max(np.abs(want))))


def test_long_sequence_is_one_launch(odla):
    build = att.build_attention(1, 2, 200, 64, "div", True, True)
    hb = odla.HipBuilder(bf16="performance")
    build(hb)
    n = hb.plan_summary()["launches"]
    hb.destroy()
    assert n <= 8, n   # conversions of the four arguments and the result beside it
