"""Plans of graphs whose products read the rows of a LayerNorm, lowered on the host: which launch
computes what.  A product of few rows takes the LayerNorm in front of it into its own launch; every
other reader of the rows keeps a launch of its own behind that one."""
import ctypes

import numpy as np
import pytest

MODES = {"fp32": {}, "fp16": {"fp16": True}, "bf16": {"bf16": "performance"}, "bf16acc": {"bf16": "accuracy"}}


def steps_of(odla, build, **kw):
    """The names of a plan's launches, in order."""
    L = odla.load_library()
    seen = []
    cb = ctypes.CFUNCTYPE(None, ctypes.c_char_p, ctypes.c_int, ctypes.c_char_p, ctypes.c_int, ctypes.c_char_p)(
        lambda f, l, fn, lvl, msg: seen.append(msg.decode()))
    hb = odla.HipBuilder(**kw)
    L.odla_SetLogger(ctypes.cast(cb, ctypes.c_void_p))
    L.odla_SetLogLevel(5)   # ODLA_LOG_LEVEL_DEBUG
    try:
        build(hb)
        launches = hb.plan_summary()["launches"]
    finally:
        L.odla_SetLogLevel(2)
        L.odla_SetLogger(None)
        hb.destroy()
    steps = [m[len("step "):] for m in seen if m.startswith("step ")]
    assert len(steps) == launches
    return steps


def weight(b, name, *shape):
    return b.const(name, np.random.default_rng(len(name) + shape[-1]).standard_normal(shape).astype(np.float32))


def product(b, x, name, k, n):
    return b.gemm(x, weight(b, name + ".w", k, n), None, False, False, 1.0, 0.0, name=name)


def position(steps, name):
    """Index of the first launch of the product `name` (which may take a LayerNorm along)."""
    at = [i for i, s in enumerate(steps) for part in s.split("+") if part.startswith("gemm") and part.split(":")[-1] == name]
    assert at, (name, steps)
    return at[0]


@pytest.mark.parametrize("mode", list(MODES))
@pytest.mark.parametrize("widths", [(768, 256), (256, 768), (768, 256, 512), (3072, 768)])
def test_every_product_over_the_rows_has_its_launch(odla, widths, mode):
    def build(b):
        h = b.layernorm(b.arg("x", (41, 768)), 1, 1e-5, name="h")
        for i, n in enumerate(widths):
            b.output(product(b, h, "p%d" % i, 768, n), "y%d" % i)

    steps = steps_of(odla, build, **MODES[mode])
    assert sum("layernorm" in s for s in steps) == 1, steps
    norm = [i for i, s in enumerate(steps) if "layernorm" in s][0]
    for i in range(len(widths)):
        assert position(steps, "p%d" % i) >= norm, steps


# products that read the normalised rows a second time, as their residual or their right operand
def residual(b, rows):
    h = b.layernorm(b.arg("x", (rows, 768)), 1, 1e-5, name="h")
    b.output(b.add(product(b, h, "p", 768, 768), h, name="y"), "y")


def addend(b, rows):
    h = b.layernorm(b.arg("x", (rows, 768)), 1, 1e-5, name="h")
    b.output(b.gemm(h, weight(b, "p.w", 768, 768), h, False, False, 1.0, 1.0, name="y"), "y")


def residual_view(b, rows):
    h = b.layernorm(b.arg("x", (rows, 768)), 1, 1e-5, name="h")
    v = b.reshape(h, (1, rows, 768), name="v")
    b.output(b.add(product(b, v, "p", 768, 768), v, name="y"), "y")


def residual_behind_activation(b, rows):
    h = b.layernorm(b.arg("x", (rows, 768)), 1, 1e-5, name="h")
    b.output(b.add(b.relu(product(b, h, "p", 768, 768), name="r"), h, name="y"), "y")


def outer_product(b, rows):
    h = b.layernorm(b.arg("x", (rows, 768)), 1, 1e-5, name="h")
    b.output(b.gemm(h, h, None, False, True, 1.0, 0.0, name="y"), "y")


TWICE = [residual, addend, residual_view, residual_behind_activation, outer_product]


@pytest.mark.parametrize("mode", list(MODES))
@pytest.mark.parametrize("rows", [1, 41])
@pytest.mark.parametrize("build", TWICE, ids=lambda f: f.__name__)
def test_rows_read_twice_are_written_by_a_launch_in_front(odla, build, rows, mode):
    steps = steps_of(odla, lambda b: build(b, rows), **MODES[mode])
    assert [s for s in steps if "layernorm" in s] == ["layernorm:h"], steps
    assert steps.index("layernorm:h") < position(steps, "y"), steps


@pytest.mark.parametrize("mode", list(MODES))
def test_residual_of_the_rows_in_front_of_the_norm_still_rides(odla, mode):
    def build(b):
        x = b.arg("x", (41, 768))
        h = b.layernorm(x, 1, 1e-5, name="h")
        b.output(b.add(product(b, h, "p", 768, 768), x, name="y"), "y")

    assert "layernorm+gemm:y" in steps_of(odla, build, **MODES[mode])
