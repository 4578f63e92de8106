"""Products of few columns, a row per workgroup: every number of wavefronts and columns the
kernel is compiled for, at the edges of its ranges, against sums in 64 bits."""
import numpy as np
import pytest

from util import run_hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("columns", [1, 4, 5, 8, 9, 12, 13, 16])
@pytest.mark.parametrize("depth", [256, 260, 512, 516, 1024, 1028, 4096, 4100, 8196])
def test_row_products(depth, columns):
    print("row product", depth, columns, flush=True)
    r = np.random.default_rng(depth * 100 + columns)
    for rows in (1, 37):
        a = r.standard_normal((rows, depth)).astype(np.float32)
        w = r.standard_normal((depth, columns)).astype(np.float32)
        bias = r.standard_normal(columns).astype(np.float32)

        def build(b):
            b.output(b.gemm(b.arg("a", a.shape), b.const("w", w), b.const("bias", bias), name="y"), "y")

        got = run_hip(build, {"a": a})["y"].astype(np.float64)
        a64, w64 = a.astype(np.float64), w.astype(np.float64)
        # the longest chain of roundings: a thread of 64 adds its terms one by one, then six exchanges of lanes,
        # up to three of wavefronts and the bias
        chain = -(-depth // 256) * 4 + 10
        bound = chain * 2.0 ** -24 * (np.abs(a64) @ np.abs(w64) + np.abs(bias))
        assert np.all(np.abs(got - (a64 @ w64 + bias)) <= bound)


@pytest.mark.parametrize("rows", [1023, 1024, 4096])
@pytest.mark.parametrize("columns,depth", [(3, 260), (16, 1028), (10, 2048), (16, 2052)])
def test_many_rows(depth, columns, rows):
    """One wavefront a row from 1024 rows on, up to a depth of 2048."""
    print("row product of many rows", rows, depth, columns, flush=True)
    r = np.random.default_rng(depth * 100 + columns)
    a = r.standard_normal((rows, depth)).astype(np.float32)
    w = r.standard_normal((depth, columns)).astype(np.float32)

    def build(b):
        b.output(b.softmax(b.gemm(b.arg("a", a.shape), b.const("w", w), None, name="y"), -1, name="s"), "s")
        b.output(b.gemm(b.arg("c", a.shape), b.const("v", w), None, name="z"), "z")

    got = run_hip(build, {"a": a, "c": a})
    y = a.astype(np.float64) @ w.astype(np.float64)
    # (as above)
    bound = (-(-depth // 256) * 4 + 10) * 2.0 ** -24 * (np.abs(a.astype(np.float64)) @ np.abs(w.astype(np.float64)))
    assert np.all(np.abs(got["z"] - y) <= bound)
    e = np.exp(y - y.max(-1, keepdims=True))
    p = e / e.sum(-1, keepdims=True)
    # a probability moves by its own logit's error and the largest one's, and by the last places of exponential, sum and quotient
    assert np.all(np.abs(got["s"] - p) <= p * (2 * bound.max(-1, keepdims=True) + 32 * 2.0 ** -24) + 2.0 ** -126)
