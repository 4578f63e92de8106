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


@pytest.mark.parametrize("rows,joins", [(1024, True), (65536, False)])
def test_offsets_of_64_bits_stay_out_of_a_launch_that_leaves_best_scores(odla, rows, joins):
    """The launch of a detector's scores leaves the best ones in its 32-bit form only: a group of 4 GiB
    behind the suppression has a launch of its own, one of 64 MiB rides along."""
    import __graft_entry__ as entry
    yolo = entry.load().models_yolo

    def build(b):
        heads = [b.arg("head%d" % i, (1, 3 * 85, 224 // s, 224 // s)) for i, s in enumerate((32, 16, 8))]
        b.output(yolo.yolo_postprocess(b, heads, 1, 224, 80, 100, 0.45, 0.3), "detections")
        x = b.arg("x", (rows, 1024, 16))
        gate = b.sigmoid(b.slice(x, (0, 0, 0), (rows, 1024, 1), name="g"), name="sg")
        b.output(b.mul(b.sigmoid(x, name="sx"), gate, name="y"), "y")

    steps = steps_of(odla, build)
    assert any(s.startswith("nms.best") for s in steps)
    assert any(s.startswith("fused:y") for s in steps) != joins, steps
