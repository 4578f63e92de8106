"""The one-launch attention at the edges of its tiles: sequences around multiples of its 32-key blocks, of
its tiles of 96 and 128 keys and of a workgroup's 128 queries, with few workgroups (two groups of
wavefronts share the tiles) and many (one); masks of -10000, of the type's lowest value and of -infinity."""
import numpy as np
import pytest
import torch

from test_gpu_attention import build_attention
from util import run_hip

pytestmark = pytest.mark.gpu


def reference(f, scale):
    q, k, v = (f[n].astype(np.float64) for n in ("q", "k", "v"))
    s = q @ k.transpose(0, 1, 3, 2) * scale + f["mask"].astype(np.float64)
    e = np.exp(s - s.max(-1, keepdims=True))
    c = (e / e.sum(-1, keepdims=True)) @ v
    return c.transpose(0, 2, 1, 3).reshape(c.shape[0], c.shape[2], -1)


CASES = [(2, 2, s) for s in (1, 31, 33, 64, 65, 97, 127, 128, 129, 191, 192, 193, 255, 257, 384, 385, 511)]
CASES += [(11, 12, s) for s in (129, 300, 384)]   # more than 128 workgroups


@pytest.mark.parametrize("mode", ["bf16", "bf16acc", "fp16"])
@pytest.mark.parametrize("mask", ["some", "lowest", "inf"])
@pytest.mark.parametrize("B,heads,S", CASES)
def test_tiles(B, heads, S, mask, mode):
    print("attention tiles", B, heads, S, mask, mode, flush=True)
    r = np.random.default_rng(S)
    f = {n: r.standard_normal((B, heads, S, 64)).astype(np.float32) for n in ("q", "k", "v")}
    keep = r.random((B, 1, 1, S)) < 0.7
    keep[..., 0] = True
    lowest = {"bf16": -3.3895314e38, "bf16acc": float(np.finfo(np.float32).min), "fp16": -65504.0}[mode]
    low = {"some": -10000.0, "lowest": lowest, "inf": -np.inf}[mask]
    f["mask"] = np.where(keep, 0.0, low).astype(np.float32)
    if mask == "lowest":
        f["mask"][0] = low   # nothing but masked keys: their plain mean (fp16: their own softmax)
    kw = {"bf16": {"bf16": "performance"}, "bf16acc": {"bf16": "accuracy"}, "fp16": {"fp16": True}}[mode]
    got = run_hip(build_attention(B, heads, S, 64, "div", True, True, True), f, **kw)["out"]
    # operands as the plan stores them
    eps = 2.0 ** -11 if mode == "fp16" else 2.0 ** -8
    stored = torch.float16 if mode == "fp16" else torch.bfloat16
    g = {n: torch.from_numpy(a).to(stored).float().numpy() if n != "mask" or mode != "bf16acc" else a for n, a in f.items()}
    if mask == "lowest" and mode != "fp16":
        g["q"] = g["q"].copy()
        g["q"][0] = 0.0          # (no score shows beside such a mask in 32 bits)
    want = np.maximum(reference(g, 0.125), 0)
    assert np.all(np.isfinite(got))
    # probabilities and the result are rounded once each; |v| stays below 5
    assert np.max(np.abs(got - want)) <= 3 * eps * 5


@pytest.mark.parametrize("mode", ["bf16", "bf16acc"])
@pytest.mark.parametrize("B,heads,S", [(2, 2, 31), (2, 2, 128), (2, 2, 300), (11, 12, 300)])
def test_masks_near_the_lowest_value_differ(B, heads, S, mode):
    """Two mask values, both below what a product with log2(e) leaves finite: the larger one decides."""
    print("attention mask near the lowest value", B, heads, S, mode, flush=True)
    r = np.random.default_rng(S)
    f = {n: r.standard_normal((B, heads, S, 64)).astype(np.float32) for n in ("q", "k", "v")}
    keep = r.random((B, 1, 1, S)) < 0.3
    keep[..., -1] = True
    for low, high in ((-3.3e38, -2.5e38), (-2.5e38, -8e37), (-1e38, -8e37), (2.5e38, 3.3e38)):
        f["mask"] = np.where(keep, high, low).astype(np.float32)
        kw = {"bf16": {"bf16": "performance"}, "bf16acc": {"bf16": "accuracy"}}[mode]
        got = run_hip(build_attention(B, heads, S, 64, "div", True, True, True), f, **kw)["out"]
        # (no score shows beside such a mask in 32 bits)
        v = torch.from_numpy(f["v"]).to(torch.bfloat16).double().numpy()
        w = keep[:, :, 0, :, None] / keep.sum(-1)[..., None]
        mean = (v * w).sum(2)                                     # [B, heads, 64]
        want = np.maximum(np.broadcast_to(mean.reshape(B, 1, heads * 64), got.shape), 0)
        # probabilities and the result are rounded once each; |v| stays below 5
        assert np.max(np.abs(got - want)) <= 3 * 2.0 ** -8 * 5
