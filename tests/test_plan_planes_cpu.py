"""Chains of plane operators, lowered on the host: one launch where that is the faster form, the
operators one by one where few large planes, or windows that are not compiled, would keep a few
compute units busy for longer than all the separate launches take."""
import numpy as np
import pytest

from test_plan_layernorm_cpu import steps_of

KW = {"fp32": {}, "fp16": {"fp16": True}}


def pool(b, x, n, c, h):
    b.output(b.maxpool(b.relu(x, name="r"), (2, 2), (2, 2), (0,) * 4, name="p"), "p")


def norm(b, x, n, c, h):
    k = lambda name, v: b.const(name, np.full((c,), v, np.float32))
    y = b.sigmoid(b.batchnorm(x, k("m", 0.1), k("v", 1.5), 1e-5, k("g", 0.7), k("o", 0.2), name="bn"), name="act")
    b.output(b.avgpool(y, (2, 2), (1, 1), (0,) * 4, name="p"), "p")
    b.output(b.add(y, x, name="s"), "s")


def average7(b, x, n, c, h):
    b.output(b.avgpool(b.relu(x, name="r"), (7, 7), (1, 1), (3,) * 4, name="p"), "p")


def upscale(b, x, n, c, h):
    b.output(b.resize_nearest(b.relu(x, name="r"), (2 * h, 2 * h), name="u"), "u")


def long_chain(b, x, n, c, h):
    k = lambda name, v: b.const(name, np.full((c,), v, np.float32))
    y = b.leaky_relu(b.batchnorm(x, k("m", 0.1), k("v", 1.5), 1e-5, k("g", 0.7), k("o", 0.2), name="bn"), 0.1, name="act")
    up = b.resize_nearest(b.maxpool(y, (3, 3), (2, 2), (1,) * 4, name="p"), (h, h), name="up")
    b.output(b.concat([up, b.add(y, x, name="s")], 1, name="cat"), "cat")
    b.output(b.reduce_mean(b.avgpool(y, (2, 2), (1, 1), (0,) * 4, name="a"), (2, 3), True, name="gap"), "gap")


# us per call as separate launches / as one, MI355X
CASES = [(pool, "fp16", 1, 4, 150, True),         # 25.0 / 17.7
         (pool, "fp16", 1, 4, 280, False),        # 25.9 / 28.5
         (pool, "fp16", 1, 16, 280, False),       # 25.0 / 29.4
         (pool, "fp16", 1, 64, 280, True),        # 31.6 / 30.1
         (pool, "fp32", 1, 1, 150, True),         # 18.9 / 18.0
         (pool, "fp32", 1, 1, 195, False),        # 19.0 / 22.3
         (norm, "fp32", 1, 1, 110, True),         # 24.4 / 23.8
         (norm, "fp32", 1, 1, 150, False),        # 24.6 / 29.1
         (norm, "fp16", 1, 1, 195, False),        # 34.6 / 41.6
         (norm, "fp16", 1, 8, 195, True),         # 46.8 / 42.4
         (norm, "fp16", 1, 8, 230, False),        # 48.0 / 52.3
         (norm, "fp16", 1, 32, 230, True),        # 62.6 / 53.0
         (norm, "fp16", 1, 16, 280, False),       # 56.0 / 64.5
         (average7, "fp16", 1, 64, 28, True),     # 38.5 / 27.5
         (average7, "fp32", 1, 1, 28, False),     # 22.6 / 27.2
         (average7, "fp16", 1, 64, 75, False),    # 38.9 / 88.2
         (average7, "fp16", 64, 96, 75, False),   # 306.7 / 376.8
         (upscale, "fp16", 1, 64, 150, True),     # 32.3 / 27.7
         (upscale, "fp16", 1, 16, 195, False),    # 28.4 / 36.5
         (upscale, "fp16", 64, 96, 75, True),     # 413.6 / 156.4
         (long_chain, "fp16", 1, 3, 150, True), (long_chain, "fp32", 1, 512, 150, True), (long_chain, "fp16", 64, 96, 75, True)]


@pytest.mark.parametrize("chain,mode,n,c,h,one", CASES, ids=["%s-%s-%d-%d-%d" % (f.__name__, m, n, c, h) for f, m, n, c, h, _ in CASES])
def test_one_launch_where_it_is_the_faster_form(odla, chain, mode, n, c, h, one):
    steps = steps_of(odla, lambda b: chain(b, b.arg("x", (n, c, h, h)), n, c, h), **KW[mode])
    assert any(s.startswith("planes(") for s in steps) == one, steps
