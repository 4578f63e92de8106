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
