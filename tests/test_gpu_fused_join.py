"""Element-wise groups that read a Concat of several launches' parts: the values, over several
replays of the captured launches.

Tolerance: fp32 graphs 1e-5 of the largest expected magnitude, fp16 storage 2e-2 absolute on O(1) data."""
import pytest

from fused_join_graphs import GRAPHS
from test_gpu_fused_eltwise import check
from util import announce, run_hip, run_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["fp32", "fp16"])
@pytest.mark.parametrize("name", GRAPHS)
def test_the_reader_of_a_concat_sees_all_of_its_parts(name, mode):
    announce("reader of a Concat %s %s" % (name, mode))
    build, feeds, _ = GRAPHS[name]
    check(run_hip(build, feeds, repeats=3, fp16=mode == "fp16"), run_ref(build, feeds), 1e-5 if mode == "fp32" else 2e-2)
