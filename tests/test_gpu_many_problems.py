"""Batches of more products than one grid holds in its third dimension (65535): batched matrix
products with a residual, results of merged heads (whose groups a launch keeps whole) and a
convolution of as many groups.  fp32 within 1e-5 of the largest value (sums of at most 64 terms,
2^-24 each), fp16 plans within 2e-3 (operands and results rounded to 2^-11)."""
import numpy as np
import pytest

from util import announce, run_both, run_hip

pytestmark = pytest.mark.gpu

MODES = {"fp32": ({}, 1e-5), "fp16": ({"fp16": True}, 2e-3)}


def close(build, feeds, mode):
    kw, tol = MODES[mode]
    got, want = run_both(build, feeds, **kw)
    for n in want:
        scale = np.abs(want[n]).max()
        assert np.abs(got[n] - want[n]).max() <= tol * scale, n
        assert np.abs(got[n].ravel()[-8:] - want[n].ravel()[-8:]).max() <= tol * scale, n


@pytest.mark.parametrize("mode", list(MODES))
@pytest.mark.parametrize("n,m,k,c,residual", [(65535, 2, 16, 8, False), (65536, 2, 16, 8, True), (65537, 1, 64, 8, False),
                                               (70001, 3, 16, 5, True), (131073, 1, 8, 8, False)])
def test_batched_product(n, m, k, c, residual, mode):
    announce("products %d x [%d, %d, %d] residual=%s %s" % (n, m, k, c, residual, mode))
    r = np.random.default_rng(n)
    feeds = {"x": r.standard_normal((n, m, k)).astype(np.float32), "w": r.standard_normal((n, k, c)).astype(np.float32)}
    if residual:
        feeds["z"] = r.standard_normal((n, m, c)).astype(np.float32)

    def build(b):
        y = b.batch_matmul(b.arg("x", (n, m, k)), b.arg("w", (n, k, c)), name="p")
        b.output(b.relu(b.add(y, b.arg("z", (n, m, c)), name="s"), name="y") if residual else y, "y")
    close(build, feeds, mode)


@pytest.mark.parametrize("mode", list(MODES))
@pytest.mark.parametrize("batch,heads", [(7000, 12), (2, 33000), (1, 66001)])
def test_merged_heads(batch, heads, mode):
    announce("merged heads %d x %d %s" % (batch, heads, mode))
    S, d = 2, 8
    r = np.random.default_rng(heads)
    feeds = {"p": r.standard_normal((batch, heads, S, 16)).astype(np.float32), "v": r.standard_normal((batch, heads, 16, d)).astype(np.float32)}

    def build(b):
        y = b.batch_matmul(b.arg("p", (batch, heads, S, 16)), b.arg("v", (batch, heads, 16, d)), name="ctx")
        b.output(b.reshape(b.transpose(y, (0, 2, 1, 3), name="t"), (batch, S, heads * d), name="r"), "y")
    close(build, feeds, mode)


@pytest.mark.parametrize("mode", list(MODES))
def test_convolution_groups(mode):
    G, cg = 66001, 8
    announce("convolution of %d groups %s" % (G, mode))
    r = np.random.default_rng(G)
    w, bias = (r.standard_normal((G * cg, cg, 1, 1)) * 0.4).astype(np.float32), r.standard_normal(G * cg).astype(np.float32)
    x = r.standard_normal((2, G * cg, 1, 2)).astype(np.float32)

    def build(b):
        b.output(b.conv(b.arg("x", x.shape), b.const("w", w), b.const("b", bias), (1, 1), (0, 0, 0, 0), group=G, name="y"), "y")
    kw, tol = MODES[mode]
    got = run_hip(build, {"x": x}, **kw)["y"]
    want = np.matmul(w.reshape(G, cg, cg).astype(np.float64), x.reshape(2, G, cg, 2).astype(np.float64)) + bias.reshape(G, cg, 1)
    assert np.abs(got - want.reshape(got.shape)).max() <= tol * np.abs(want).max()
