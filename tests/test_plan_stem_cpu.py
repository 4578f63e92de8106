"""Plans of a network stem whose pool is one part of a channel Concat (two-branch stems), lowered on the host: the
stem's launch writes its slice where a pixel's slice holds whole 16-byte vectors, otherwise the launches stay apart."""
import pytest

from stem_concat_graphs import CONCATS, concat_graph
from test_plan_layernorm_cpu import steps_of


@pytest.mark.parametrize("mode", [{"fp16": True}, {"bf16": "performance"}], ids=["fp16", "bf16"])
@pytest.mark.parametrize("parts,one", CONCATS)
def test_pool_in_front_of_a_concat(odla, parts, one, mode):
    steps = steps_of(odla, concat_graph(2, 40, 38, parts)[0], **mode)
    assert any(s.startswith("stem:") for s in steps) == one, steps
    assert any(s.startswith("maxpool:p") for s in steps) != one, steps
    assert not any(s.startswith("concat:") for s in steps), steps
