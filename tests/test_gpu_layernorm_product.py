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


def forms(rows, c):
    """Graphs in which the product with the LayerNorm in its launch is not the rows' only reader."""
    r = np.random.default_rng(rows * c)
    w = {n: (r.standard_normal((c, n)) * c ** -0.5).astype(np.float32) for n in (c, 256, 72)}
    norm = lambda b, t, name: b.layernorm(t, 1, 1e-5, name=name)
    mm = lambda b, t, n, name: b.gemm(t, b.const(name + ".w", w[n]), None, False, False, 1.0, 0.0, name=name)

    def two_widths(b):
        h = norm(b, b.arg("x", (rows, c)), "h")
        b.output(mm(b, h, c, "q"), "q")
        b.output(mm(b, h, 256, "k"), "k")

    def three_widths_and_the_rows(b):
        h = norm(b, b.arg("x", (rows, c)), "h")
        b.output(b.gelu(mm(b, h, c, "q"), False, name="act"), "q")
        b.output(mm(b, h, 256, "k"), "k")
        b.output(mm(b, h, 72, "v"), "v")
        b.output(h, "rows")

    def residual(b):
        h = norm(b, b.arg("x", (rows, c)), "h")
        b.output(b.add(mm(b, h, c, "p"), h, name="y"), "y")

    def addend_of_a_view(b):
        h = b.reshape(norm(b, b.arg("x", (rows, c)), "h"), (1, rows, c), name="v")
        b.output(b.gemm(h, b.const("p.w", w[c]), h, False, False, 1.0, 1.0, name="y"), "y")

    def residual_in_front_of_the_norm(b):
        x = b.arg("x", (rows, c))
        b.output(b.add(mm(b, norm(b, x, "h"), c, "p"), x, name="y"), "y")

    def outer_product(b):
        h = norm(b, b.arg("x", (rows, c)), "h")
        b.output(b.gemm(h, h, None, False, True, 1.0, 0.0, name="y"), "y")

    return {f.__name__: f for f in (two_widths, three_widths_and_the_rows, residual, addend_of_a_view, residual_in_front_of_the_norm, outer_product)}


@pytest.mark.parametrize("mode", list(KW))
@pytest.mark.parametrize("rows,c", [(1, 768), (41, 768), (17, 512)])
@pytest.mark.parametrize("form", list(forms(1, 64)))
def test_other_readers_of_the_rows(form, rows, c, mode):
    """Two inputs through one context: what the second leaves is not what the first left."""
    announce("readers of layernorm rows: %s %d x %d %s" % (form, rows, c, mode))
    build = forms(rows, c)[form]
    feeds = [{"x": (np.random.default_rng(s).standard_normal((rows, c)) * (1 + s)).astype(np.float32)} for s in (0, 1)]
    hb = entry.load().odla.HipBuilder(**KW[mode])
    try:
        build(hb)
        s = hb.session()
        try:
            got = [s.run(f) for f in feeds]
        finally:
            s.close()
    finally:
        hb.destroy()
    for f, g in zip(feeds, got):
        want = run_ref(build, f)
        for name in want:
            err = np.abs(g[name] - want[name]).max() / np.abs(want[name]).max()
            assert err <= TOL[mode], (name, err)


@pytest.mark.parametrize("mode", ["fp32", "bf16"])
def test_a_plan_outlives_its_tuning_environment(mode, monkeypatch):
    """Launches that are made anew on every execution keep the kernels of the plan."""
    announce("plan and environment %s" % mode)
    monkeypatch.setenv("ODLA_HIP_GRAPH_MIN_STEPS", "1000")
    build = forms(41, 768)["three_widths_and_the_rows"]
    feeds = {"x": np.random.default_rng(5).standard_normal((41, 768)).astype(np.float32)}
    hb = entry.load().odla.HipBuilder(**KW[mode])
    try:
        build(hb)
        s = hb.session()
        try:
            first = s.run(feeds)
            monkeypatch.setenv("ODLA_HIP_IGEMM_TILE", "128x64")
            second = s.run(feeds)
        finally:
            s.close()
    finally:
        hb.destroy()
    for name in first:
        assert np.array_equal(first[name], second[name]), name
