"""Plans in which an element-wise group could ride in the launch of an earlier one, lowered on the
host: it does so only behind the last launch that stores to what it reads."""
import pytest

from fused_join_graphs import GRAPHS
from test_plan_layernorm_cpu import steps_of


@pytest.mark.parametrize("mode", [{}, {"fp16": True}], ids=["fp32", "fp16"])
@pytest.mark.parametrize("name", GRAPHS)
def test_the_reader_of_a_concat_follows_all_of_its_parts(odla, name, mode):
    build, _, want = GRAPHS[name]
    steps = [s.split("(")[0] for s in steps_of(odla, build, **mode) if not s.startswith(("cast", "out.cast"))]
    assert steps == want


def test_groups_that_read_finished_values_still_share_a_launch(odla):
    def build(b):
        x, z = b.arg("x", (64, 100, 64)), b.arg("z", (16, 1000, 64))
        b.output(b.relu(b.tanh(b.add(x, x, name="a"), name="t"), name="u"), "u")
        b.output(b.tanh(b.mul(z, z, name="c"), name="v"), "v")

    assert [s.split("(")[0] for s in steps_of(odla, build)] == ["fused:u"]
