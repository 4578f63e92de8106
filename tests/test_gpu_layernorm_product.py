"""A LayerNorm in front of a product of few rows, computed by the product's own launch: rows at the
edges of the 16- and 32-row tiles, channel counts that give a wavefront one, two and three steps of
K (and ones that stay apart), with and without scale and offset, a residual that reads the
normalised rows too, and three products over the same rows.  Tolerances: storage type."""
import numpy as np
import pytest

import __graft_entry__ as entry
from util import announce, run_hip, run_ref

pytestmark = pytest.mark.gpu

KW = {"fp32": {}, "fp16": {"fp16": True}, "bf16": {"bf16": "performance"}, "bf16acc": {"bf16": "accuracy"}}
TOL = {"fp32": 1e-4, "fp16": 1e-2, "bf16": 4e-2, "bf16acc": 2e-2}


def build_block(rows, c, affine):
    r = np.random.default_rng(c + rows)
    w = [(r.standard_normal((c, n)) * c ** -0.5).astype(np.float32) for n in (c, c, c, 72)]
    g, o = (r.standard_normal(c).astype(np.float32) for _ in range(2))

    def build(b):
        x = b.arg("x", (1, rows, c))
        n = lambda t, name: b.layernorm(t, 1, 1e-5, *([b.const(name + ".g", g), b.const(name + ".o", o)] if affine else []), name=name)
        mm = lambda t, i, name: b.gemm(t, b.const(name + ".w", w[i]), None, False, False, 1.0, 0.0, name=name)
        h = n(x, "n0")
        q = b.add(b.add(mm(h, 0, "q"), mm(h, 1, "k"), name="qk"), mm(h, 2, "v"), name="qkv")
        h2 = n(b.add(q, h, name="res"), "n1")
        b.output(b.gelu(mm(h2, 3, "f"), False, name="act"), "y")
        b.output(h2, "h2")
    return build


@pytest.mark.parametrize("mode", list(KW))
@pytest.mark.parametrize("rows,c,affine", [(1, 768, True), (15, 512, True), (16, 256, False), (17, 1024, True), (33, 768, False), (41, 768, True),
                                           (64, 544, True), (96, 1536, True), (7, 1568, True), (31, 64, True), (5, 200, True)])
def test_layernorm_rides_in_the_product(rows, c, affine, mode):
    announce("layernorm + product %d x %d affine=%s %s" % (rows, c, affine, mode))
    build = build_block(rows, c, affine)
    feeds = {"x": np.random.default_rng(3).standard_normal((1, rows, c)).astype(np.float32) + 0.5}
    want, got = run_ref(build, feeds), run_hip(build, feeds, **KW[mode])
    for name in want:
        err = np.abs(got[name] - want[name]).max() / np.abs(want[name]).max()
        assert err <= TOL[mode], (name, err)
