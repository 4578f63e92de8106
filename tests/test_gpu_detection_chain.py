"""What follows a detector's heads: element-wise groups that read in front of a Transpose and write
into a Concat over several groups, and non-maximum suppression in blocks of 64 candidates.

Tolerance: fp32 graphs 1e-5 of the largest expected magnitude, fp16 storage 2e-2 absolute on O(1) data;
the suppression's indices are whole numbers and equal the oracle's."""
import numpy as np
import pytest

from test_gpu_fused_eltwise import check, fused, run_with_steps
from util import announce, run_both, run_ref

pytestmark = pytest.mark.gpu


def decode(b, n, sizes, classes, anchors=3):
    """Heads [n, anchors * (5 + classes), g] -> [n, boxes, 2] and [n, classes, boxes] over all heads."""
    per_box, per_class = [], []
    for i, g in enumerate(sizes):
        h = b.arg("h%d" % i, (n, anchors * (5 + classes), g))
        t = b.reshape(h, (n, anchors, 5 + classes, g), name="r%d" % i)
        t = b.transpose(t, (0, 1, 3, 2), name="t%d" % i)
        t = b.reshape(t, (n, anchors * g, 5 + classes), name="s%d" % i)
        part = lambda k0, k1, nm: b.slice(t, (0, 0, k0), (n, anchors * g, k1), name="%s%d" % (nm, i))
        pos = b.const("p%d" % i, np.tile(np.arange(g, dtype=np.float32), anchors).reshape(1, anchors * g, 1))
        cx = b.add(b.sigmoid(part(0, 1, "x"), name="sx%d" % i), pos, name="cx%d" % i)
        cy = b.add(b.exp(part(1, 2, "y"), name="ey%d" % i), pos, name="cy%d" % i)
        per_box.append(b.concat([cx, cy], 2, name="b%d" % i))
        score = b.mul(b.sigmoid(part(5, 5 + classes, "c"), name="sc%d" % i), b.sigmoid(part(4, 5, "o"), name="so%d" % i), name="m%d" % i)
        per_class.append(b.transpose(score, (0, 2, 1), name="q%d" % i))
    b.output(b.concat(per_box, 1, name="boxes"), "boxes")
    b.output(b.concat(per_class, 2, name="scores"), "scores")


# one head; several of which one is tiny; rows that are not 16-byte multiples; more than 2^22 points,
# where a scattered store would not pay but this one is not scattered; more heads than a launch takes
@pytest.mark.parametrize("mode,n,sizes,classes", [("fp32", 1, (7,), 1), ("fp32", 2, (169, 4, 1), 9), ("fp16", 3, (64, 65), 80),
                                                  ("fp32", 4, (6000, 12), 80), ("fp32", 1, tuple(range(5, 15)), 3)])
def test_decode_reads_the_heads_and_writes_the_concat(mode, n, sizes, classes):
    announce("decode %s n %d heads %s classes %d" % (mode, n, sizes, classes))
    r = np.random.default_rng(3)
    feeds = {"h%d" % i: r.standard_normal((n, 3 * (5 + classes), g)).astype(np.float32) for i, g in enumerate(sizes)}
    build = lambda b: decode(b, n, sizes, classes)
    got, steps = run_with_steps(build, feeds, fp16=(mode == "fp16"))
    check(got, run_ref(build, feeds), 1e-5 if mode == "fp32" else 2e-2)
    assert not [s for s in steps if s.startswith(("transpose:", "concat:", "slice:"))], steps
    if mode == "fp32" and len(sizes) > 1:   # (no conversion of a later head stands between them)
        assert len(fused(steps)) < 2 * len(sizes), steps


def test_a_transposed_value_with_another_reader_exists_as_well():
    """A Transpose read by a group and by something else; one whose dims the group cannot follow."""
    announce("transposed value, several readers")
    r = np.random.default_rng(4)
    x = r.standard_normal((6, 10, 8)).astype(np.float32)

    def build(b):
        v = b.arg("x", x.shape)
        t = b.transpose(v, (0, 2, 1), name="t")
        b.output(b.tanh(b.mul(t, t, name="sq"), name="y"), "y")
        b.output(b.softmax(t, -1, name="sm"), "sm")
        u = b.reshape(b.transpose(v, (2, 1, 0), name="u"), (5, 16, 6), name="ur")   # 8 x 10 regrouped as 5 x 16
        b.output(b.exp(b.neg(u, name="un"), name="z"), "z")
        w = b.reshape(b.transpose(v, (1, 2, 0), name="w"), (10, 48), name="wr")     # two dims of the source in one
        b.output(b.exp(b.neg(b.slice(w, (0, 3), (10, 48), name="ws"), name="wn"), name="wz"), "wz")

    got, _ = run_with_steps(build, {"x": x})
    check(got, run_ref(build, {"x": x}), 1e-5)


# candidates at the edges of a block, of the keys one thread holds, and of a power of two; ties; few and
# many results; boxes all overlapping (one chain per block) and hardly any
@pytest.mark.parametrize("n,boxes,classes,max_out,span", [(1, 1, 1, 1, 4), (2, 63, 2, 70, 4), (2, 64, 4, 64, 4), (3, 65, 5, 65, 6), (1, 129, 3, 128, 0.1),
                                                          (2, 1024, 2, 1024, 60), (2, 1025, 2, 1000, 60), (1, 2049, 1, 1, 30), (1, 8192, 1, 500, 90)])
def test_nms_block_edges(n, boxes, classes, max_out, span):
    announce("nms edges %s" % ((n, boxes, classes, max_out, span),))
    r = np.random.default_rng(boxes)
    cy, cx = r.random((n, boxes)) * span, r.random((n, boxes)) * span
    h, w = r.random((n, boxes)) * 2 + 0.1, r.random((n, boxes)) * 2 + 0.1
    bx = np.stack([cy - h / 2, cx - w / 2, cy + h / 2, cx + w / 2], axis=-1).astype(np.float32)
    bx[:, ::7, 2] = bx[:, ::7, 0]                     # empty boxes
    bx[:, 1::5] = bx[:, 1::5][..., [2, 3, 0, 1]]      # flipped corners
    sc = (r.integers(40, 100, (n, classes, boxes)) / 100).astype(np.float32)   # every box a candidate, many ties

    def build(b):
        bb, ss = b.arg("boxes", bx.shape), b.arg("scores", sc.shape)
        b.output(b.nms(bb, ss, max_out, 0.45, 0.3, name="y"), "y")
        b.output(b.nms(bb, ss, max_out, 0.0, 0.3, name="all"), "all")   # a threshold that every pair reaches

    got, want = run_both(build, {"boxes": bx, "scores": sc})
    assert np.array_equal(got["y"], want["y"])
    assert np.array_equal(got["all"], want["all"])


@pytest.mark.parametrize("mode", ["fp32", "fp16"])
def test_scores_that_fill_the_chip_share_the_launch_of_the_boxes(mode):
    """Groups of different programs in one launch (a workgroup per compute unit and more of class
    scores), with heads below and above that size."""
    sizes, classes, n = (9, 5000, 700), 80, 3
    announce("decode in one launch, %s" % mode)
    r = np.random.default_rng(5)
    feeds = {"h%d" % i: r.standard_normal((n, 3 * (5 + classes), g)).astype(np.float32) for i, g in enumerate(sizes)}
    build = lambda b: decode(b, n, sizes, classes)
    got, steps = run_with_steps(build, feeds, fp16=(mode == "fp16"))
    check(got, run_ref(build, feeds), 1e-5 if mode == "fp32" else 2e-2)
    if mode == "fp32":
        assert len(fused(steps)) <= 2, steps
