"""Plans of operators with one constant each in front of an activation, lowered on the host: the activation stays in
the launch of the operator in front of it, which applies it to the value as it is before it is rounded."""
import numpy as np
import pytest

from test_plan_layernorm_cpu import MODES, steps_of

ACTS = {"relu": lambda b, t: b.relu(t, name="act"), "leaky": lambda b, t: b.leaky_relu(t, 0.3, name="act"),
        "clamp": lambda b, t: b.clamp(t, -0.5, 0.5, name="act")}


def scalars_and_act(b, shape, act, ops):
    t = b.arg("x", shape)
    for i, (op, c) in enumerate(ops):
        t = getattr(b, op)(t, b.const("c%d" % i, np.full((1,), c, np.float32)), name="t%d" % i)
    b.output(ACTS[act](b, t), "y")


OPS = [("mul", 0.3), ("add", 0.7), ("sub", 0.11), ("mul", 1.7), ("add", -0.2), ("div", 3.0)]


@pytest.mark.parametrize("mode", sorted(MODES))
@pytest.mark.parametrize("act", sorted(ACTS))
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 6])
def test_activation_rides_with_the_last_operator(odla, n, act, mode):
    steps = steps_of(odla, lambda b: scalars_and_act(b, (2, 3, 5, 7), act, OPS[:n]), **MODES[mode])
    steps = [s for s in steps if not s.startswith("out.cast")]
    assert not any(s.startswith("unary") for s in steps), steps
    assert steps[-1] == "binary:act", steps
    # up to four operators in front of it and the conversion of the argument are one launch
    in_front = n - 1 + (mode in ("fp16", "bf16"))
    assert len(steps) == (1 + (in_front > 0) if n <= 5 else 3), steps
