"""Small arguments in ordinary host memory that several launches read: the sequence's first launches copy them.
Byte counts with and without a remainder of 16, up to the largest that takes this way and one above, new data and
new buffers in every execution, captured or not; the bytes arrive as they are."""
import numpy as np
import pytest

import __graft_entry__ as entry
from test_gpu_device_args import capture_log
from util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("use_graph", [True, False])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 255, 257, 1023, 4099, 262143, 262144, 262145])
def test_arguments_read_twice(n, use_graph):
    announce("host copy %d graph=%s" % (n, use_graph))
    odla = entry.load().odla
    L, seen = odla.load_library(), []
    hb = odla.HipBuilder()
    x, z = hb.arg("x", (1, n)), hb.arg("z", (1, 7))
    # matrices of one column are copies of the rows: several launches read both arguments
    for k, t in enumerate((x, z)):
        for i in range(4):
            hb.output(hb.transpose(hb.concat([t, t], 0, name="c%d%d" % (k, i)), (1, 0), name="t%d%d" % (k, i)), "o%d%d" % (k, i))
    callback = capture_log(L, seen)
    try:
        s = hb.session(use_graph)
        r = np.random.default_rng(n)
        for _ in range(3):
            seen.clear()
            feeds = {"x": r.standard_normal((1, n)).astype(np.float32), "z": r.standard_normal((1, 7)).astype(np.float32)}
            feeds["x"][0, -1] = np.float32(np.inf)
            got = s.run(feeds)
            # up to 1 MiB
            assert any("'x' is copied by the first launches" in m for m in seen) == (4 * n <= 1 << 20), seen
            assert any("'z' is copied by the first launches" in m for m in seen), seen
            for k, name in enumerate("xz"):
                want = np.concatenate([feeds[name], feeds[name]], 0).T
                for i in range(4):
                    np.testing.assert_array_equal(got["o%d%d" % (k, i)], want)
        s.close()
    finally:
        L.odla_SetLogLevel(2)
        L.odla_SetLogger(None)
        del callback
        hb.destroy()
