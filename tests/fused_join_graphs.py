"""Graphs in which an element-wise group reads a Concat that is filled by several launches: nothing
may run such a group beside, or in front of, the last of them."""
import numpy as np


def parts_of_two_groups(n, rows, same):
    """Two groups store a part each, a Softmax stands between them; with `same` the reader of the
    Concat repeats the program of the second one."""
    def build(b):
        h0, h1 = b.arg("h0", (n, rows, 64)), b.arg("h1", (n, 3 * rows, 64))
        p0 = b.sigmoid(b.mul(h0, h0, name="a0"), name="p0")
        q = b.softmax(h1, -1, name="q")
        p1 = b.tanh(b.mul(q, q, name="a1"), name="p1") if same else b.relu(b.tanh(b.add(q, q, name="a1"), name="t1"), name="p1")
        cc = b.concat([p0, p1], 1, name="cc")
        b.output(b.tanh(b.mul(cc, cc, name="a2"), name="y"), "y")

    return build, feeds(h0=(n, rows, 64), h1=(n, 3 * rows, 64)), ["fused:p0", "softmax:q", "fused:p1", "fused:y"]


def part_of_a_copy(n, rows):
    """One part is stored by its group, the other one copied by the Concat itself, behind an
    independent group that the reader could ride with."""
    def build(b):
        h0, h1, z = b.arg("h0", (n, rows, 64)), b.arg("h1", (n, 3 * rows, 64)), b.arg("z", (3, 5, 7))
        p0 = b.sigmoid(b.mul(h0, h0, name="a0"), name="p0")
        b.output(b.relu(b.tanh(b.add(z, z, name="b0"), name="b1"), name="w"), "w")
        p1 = b.softmax(h1, -1, name="p1")
        cc = b.concat([p0, p1], 1, name="cc")
        b.output(b.tanh(b.mul(cc, cc, name="a2"), name="y"), "y")

    return build, feeds(h0=(n, rows, 64), h1=(n, 3 * rows, 64), z=(3, 5, 7)), ["fused:p0", "fused:w", "softmax:p1", "concat:cc", "fused:y"]


def feeds(**shapes):
    r = np.random.default_rng(17)
    return {k: r.standard_normal(s).astype(np.float32) for k, s in shapes.items()}


# (a reader of one workgroup, of more than one per compute unit, and of many)
GRAPHS = {"%s_%d_%d" % (kind, n, rows): make(n, rows)
          for n, rows in ((1, 10), (64, 10), (16, 1000))
          for kind, make in (("groups", lambda n, r: parts_of_two_groups(n, r, False)), ("repeated", lambda n, r: parts_of_two_groups(n, r, True)),
                             ("copy", part_of_a_copy))}
