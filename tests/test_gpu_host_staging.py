"""Arguments and results in ordinary host memory.  Small ones pass through page-locked room of the
context (read and written there by the launch itself where it touches every element once, copied
otherwise), larger ones straight between the caller's memory and the device: sizes around the
limits (1 MiB in, 128 KiB out), one argument below and one above, rows of a small product, and
executions that alternate between host and device buffers and between inputs."""
import ctypes

import numpy as np
import pytest

import __graft_entry__ as entry
from util import announce, run_ref

pytestmark = pytest.mark.gpu


def product(rows):
    w = (np.random.default_rng(1).standard_normal((256, 8)) * 0.1).astype(np.float32)

    def build(b):
        x = b.arg("x", (rows, 256))
        b.output(b.softmax(b.gemm(x, b.const("w", w), name="mm"), -1, name="sm"), "y")
    return build


def pair(rows):
    def build(b):
        x, z = b.arg("x", (rows, 64)), b.arg("z", (1, 64))
        s = b.add(x, z, name="s")
        b.output(s, "s")
        b.output(b.reduce_mean(s, (0,), True, name="m"), "m")
    return build


def image(rows):
    w = (np.random.default_rng(2).standard_normal((8, 3, 3, 3)) * 0.2).astype(np.float32)

    def build(b):
        b.output(b.relu(b.conv(b.arg("x", (rows, 3, 16, 16)), b.const("w", w), pad=(1, 1, 1, 1), name="c"), name="r"), "y")
    return build


@pytest.mark.parametrize("use_graph", [True, False])
@pytest.mark.parametrize("make,rows", [(product, r) for r in (1, 3, 1024, 1025, 4096)] +
                         [(pair, r) for r in (1, 511, 512, 513, 4096, 4097)] + [(image, r) for r in (1, 2, 16, 341, 342)])
def test_host_buffers_of_every_size(make, rows, use_graph):
    announce("host buffers %s %d rows graph=%s" % (make.__name__, rows, use_graph))
    build = make(rows)
    hb = entry.load().odla.HipBuilder()
    build(hb)
    s, device = hb.session(use_graph), hb.session(use_graph)
    r = np.random.default_rng(rows)
    kept = []
    for _ in range(4):
        feeds = {n: r.standard_normal(shape).astype(np.float32) for n, (h, shape, dt) in hb.args.items()}
        want = run_ref(build, feeds)
        kept.append((want, s.run(feeds)))
    # device buffers through the same context, then host arrays again
    device.bind_device_io(feeds)
    for name, (h, shape, dt) in hb.outs.items():
        assert s.L.odla_BindToOutput(h, device.dev_out[name][0], s.ctx) == 0
    s.execute()
    for name, (p, shape, dt) in device.dev_out.items():
        got = np.empty(shape, dt)
        assert s.L.odla_CopyMemory(got.ctypes.data_as(ctypes.c_void_p), p, got.nbytes, entry.load().odla.ODLA_MEMCPY_D2H) == 0
        kept.append(({name: want[name]}, {name: got}))
    kept.append((want, s.run(feeds)))
    for want, got in kept:   # (also: a later execution leaves earlier results alone)
        for name in want:
            np.testing.assert_allclose(got[name], want[name], rtol=1e-4, atol=1e-4)
    s.close()
    device.close()
    hb.destroy()
