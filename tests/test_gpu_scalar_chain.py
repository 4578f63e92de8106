"""Operators with one constant each behind the conversion of an argument: one launch, every step rounded as the stored
value would be (bit for bit); infinities, NaN, division by zero; forms that keep their launches."""
import numpy as np
import pytest
import torch

from test_plan_layernorm_cpu import steps_of
from util import announce, run_hip

pytestmark = pytest.mark.gpu

MODES = {"fp32": ({}, torch.float32), "fp16": ({"fp16": True}, torch.float16), "bf16": ({"bf16": "performance"}, torch.bfloat16), "bf16acc": ({"bf16": "accuracy"}, torch.float32)}
# operator, constant, constant on the left
CHAINS = {"mask": [("sub", 1.0, True), ("mul", -10000.0, False)],
          "five": [("mul", 0.3, False), ("add", 0.7, True), ("div", 3.0, False), ("sub", 0.11, False), ("mul", 2.0, True)],
          "divided": [("div", 1.0, True), ("mul", 0.1, False)],
          "one": [("add", 0.1, False)]}


def builder(shape, chain, also=()):
    def build(b):
        t = b.arg("x", shape)
        for k, (op, c, lhs) in enumerate(chain):
            cv = b.const("c%d" % k, np.full((1,), c, np.float32))
            t = getattr(b, op)(cv, t, name="t%d" % k) if lhs else getattr(b, op)(t, cv, name="t%d" % k)
            if k in also or k == len(chain) - 1:
                b.output(t, "y%d" % k)
    return build


def expected(x, chain, dtype):
    def rounded(t):
        return t.to(dtype).float()
    t = rounded(torch.from_numpy(x))
    for op, c, lhs in chain:
        cv = rounded(torch.tensor(c))
        l, r = (cv, t) if lhs else (t, cv)
        t = rounded({"add": torch.add, "sub": torch.sub, "mul": torch.mul, "div": torch.div}[op](l, r))
    return t.numpy()


@pytest.mark.parametrize("mode", sorted(MODES))
@pytest.mark.parametrize("chain", sorted(CHAINS))
@pytest.mark.parametrize("shape", [(1, 1, 1, 1), (2, 1, 1, 41), (3, 2, 5, 7), (64, 1, 1, 128), (1, 1, 300, 1031), (5, 13)])
def test_chain_of_scalars(odla, mode, chain, shape):
    announce("scalar chain %s %s %s" % (mode, chain, shape))
    kw, dtype = MODES[mode]
    x = np.random.default_rng(sum(shape)).standard_normal(shape).astype(np.float32)
    flat = x.reshape(-1)
    flat[:1] = 0.0
    if flat.size > 3:
        flat[1:4] = np.inf, -np.inf, np.nan
    build = builder(shape, CHAINS[chain])
    if len(shape) == 4:
        names = steps_of(odla, build, **kw)
        converts = dtype != torch.float32
        assert any(s.startswith("scalars(") for s in names) == (converts or len(CHAINS[chain]) > 1)
        assert not any(s.startswith("cast:") for s in names)
    got = run_hip(build, {"x": x}, **kw)["y%d" % (len(CHAINS[chain]) - 1)]
    if len(shape) == 4:
        np.testing.assert_array_equal(got, expected(x, CHAINS[chain], dtype))
    else:
        np.testing.assert_allclose(got, expected(x, CHAINS[chain], dtype), rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("mode", sorted(MODES))
def test_a_step_that_is_read_elsewhere_ends_the_launch(odla, mode):
    kw, dtype = MODES[mode]
    chain = CHAINS["five"]
    x = np.random.default_rng(1).standard_normal((2, 3, 4, 5)).astype(np.float32)
    got = run_hip(builder(x.shape, chain, also=(1, 2)), {"x": x}, **kw)
    for k in (1, 2, 4):
        np.testing.assert_array_equal(got["y%d" % k], expected(x, chain[:k + 1], dtype))


@pytest.mark.parametrize("mode", sorted(MODES))
@pytest.mark.parametrize("act", ["relu", "leaky", "clamp"])
@pytest.mark.parametrize("n", [1, 2, 3, 5])
def test_an_activation_takes_the_value_before_it_is_rounded(odla, n, act, mode):
    announce("scalar chain and activation %s %d %s" % (mode, n, act))
    kw, dtype = MODES[mode]
    chain = CHAINS["five"][:n]
    x = np.random.default_rng(n).standard_normal((3, 2, 50, 41)).astype(np.float32)

    def build(b):
        t = b.arg("x", x.shape)
        for k, (op, c, lhs) in enumerate(chain):
            cv = b.const("c%d" % k, np.full((1,), c, np.float32))
            t = getattr(b, op)(cv, t, name="t%d" % k) if lhs else getattr(b, op)(t, cv, name="t%d" % k)
        b.output({"relu": lambda: b.relu(t, name="act"), "leaky": lambda: b.leaky_relu(t, 0.3, name="act"),
                  "clamp": lambda: b.clamp(t, -0.4, 0.4, name="act")}[act](), "y")

    v = torch.from_numpy(expected(x, chain[:-1], dtype)) if n > 1 else torch.from_numpy(x).to(dtype).float()
    op, c, lhs = chain[-1]
    cv = torch.tensor(c).to(dtype).float()
    l, r = (cv, v) if lhs else (v, cv)
    v = {"add": torch.add, "sub": torch.sub, "mul": torch.mul, "div": torch.div}[op](l, r)
    v = {"relu": lambda: torch.relu(v), "leaky": lambda: torch.where(v > 0, v, v * torch.tensor(0.3)),
         "clamp": lambda: torch.clamp(v, -0.4, 0.4)}[act]()
    np.testing.assert_array_equal(run_hip(build, {"x": x}, **kw)["y"], v.to(dtype).float().numpy())
