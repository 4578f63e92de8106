"""Graphs whose stem (7x7 convolution, ReLU, 3x3 maximum) ends in a channel Concat with other branches."""
import numpy as np

# channels of the parts ("stem": the stem's 64), and whether the stem is one launch there
CONCATS = [(("stem", 64), True), ((64, "stem"), True), ((16, "stem", 24), True), (("stem",), True),
           ((12, "stem"), False), (("stem", 12), False), ((8, "stem", 4), False)]


def concat_graph(n, h, w, parts):
    r = np.random.default_rng(h * 3 + w + len(parts))
    x = r.standard_normal((n, 3, h, w)).astype(np.float32)
    k, bias = (r.standard_normal((64, 3, 7, 7)) * 0.12).astype(np.float32), r.standard_normal(64).astype(np.float32) * 0.3
    ks = [None if c == "stem" else (r.standard_normal((c, 3, 3, 3)) * 0.2).astype(np.float32) for c in parts]

    def build(b):
        image = b.arg("x", x.shape)
        made = []
        for i, c in enumerate(parts):
            if c == "stem":
                t = b.relu(b.conv(image, b.const("w", k), b.const("b", bias), (2, 2), (3, 3, 3, 3), name="y"), name="t")
                made.append(b.maxpool(t, (3, 3), (2, 2), (1, 1, 1, 1), name="p"))
            else:
                t = b.relu(b.conv(image, b.const("w%d" % i, ks[i]), None, (2, 2), (1, 1, 1, 1), name="y%d" % i), name="t%d" % i)
                made.append(b.maxpool(t, (3, 3), (2, 2), (1, 1, 1, 1), name="q%d" % i))
        b.output(b.relu(b.concat(made, 1, name="cat"), name="out_relu"), "out")

    return build, {"x": x}
