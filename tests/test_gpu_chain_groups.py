"""Element-wise groups that walk one axis with a single value in hand, and the best class scores that
they leave for NonMaxSuppression: walks that no batch of points divides, few and many boxes, ties and
NaN among the scores."""
import numpy as np
import pytest

from test_plan_layernorm_cpu import steps_of
from util import run_hip, run_both

pytestmark = pytest.mark.gpu


def scores_graph(b, x, classes, op):
    """[n, boxes, 1 + classes] -> sigmoid(class) op sigmoid(object), stored as [n, classes, boxes]."""
    n, boxes, _ = x.shape
    t = b.arg("x", x.shape)
    obj = b.sigmoid(b.slice(t, (0, 0, 0), (n, boxes, 1), name="o"), name="so")
    cls = b.sigmoid(b.slice(t, (0, 0, 1), (n, boxes, 1 + classes), name="c"), name="sc")
    return b.transpose(op(b, cls, obj), (0, 2, 1), name="scores")


OPS = {"mul": lambda b, c, o: b.mul(c, o, name="v"), "sub": lambda b, c, o: b.sub(o, c, name="v"),
       "exp": lambda b, c, o: b.exp(b.add(c, o, name="s"), name="v")}


@pytest.mark.parametrize("mode", [{}, {"fp16": True}, {"bf16": "performance"}], ids=["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("n,boxes,classes", [(1, 128, 16), (2, 127, 17), (1, 200, 33), (3, 1000, 80), (2, 5000, 21)])
def test_walks(n, boxes, classes, op, mode):
    print("chain", n, boxes, classes, op, mode, flush=True)
    x = np.random.default_rng(classes).standard_normal((n, boxes, 1 + classes)).astype(np.float32) * 3
    got, want = run_both(lambda b: b.output(scores_graph(b, x, classes, OPS[op]), "y"), {"x": x}, **mode)
    # three roundings of a storage type behind values of at most e^2; fp32: the functions' own last places
    tol = 3e-6 if not mode else 8 * (2.0 ** -11 if "fp16" in mode else 2.0 ** -8)
    assert np.max(np.abs(got["y"] - want["y"])) <= tol * max(1.0, float(np.max(np.abs(want["y"]))))


@pytest.mark.parametrize("mode", [{}, {"fp16": True}], ids=["fp32", "fp16"])
@pytest.mark.parametrize("n,hw,classes", [(1, 224, 16), (3, 224, 19), (1, 320, 80), (2, 352, 33)])
def test_best_scores_as_the_scores_themselves(odla, n, hw, classes, mode):
    """The detections of the whole post-processing are those of a NonMaxSuppression that is given its
    boxes and scores as arguments and reduces the classes itself."""
    import __graft_entry__ as entry
    yolo = entry.load().models_yolo
    print("best scores", n, hw, classes, mode, flush=True)
    r = np.random.default_rng(hw + classes)
    feeds = {}
    for i, stride in enumerate((32, 16, 8)):
        g = hw // stride
        h = r.standard_normal((n, 3, 5 + classes, g, g)).astype(np.float32)
        h[:, :, 4:] -= 1.0
        h[:, :, 5:, 0, 0] = 1.5                  # equal scores: the first class
        h[:, 0, 5 + classes // 2, 1, 1] = np.nan  # never larger than another
        h[:, 1, 5, 1, 0] = np.nan                 # the first class: stays
        h[:, 2, 4, 0, 1] = np.inf
        feeds["head%d" % i] = h.reshape(n, -1, g, g)

    def post(b):
        heads = [b.arg("head%d" % i, f.shape) for i, f in enumerate(feeds.values())]
        b.output(yolo.yolo_postprocess(b, heads, n, hw, classes, 100, 0.45, 0.3), "detections")

    assert any(s.startswith("nms.best") for s in steps_of(odla, post, **mode))
    got = run_hip(post, feeds, **mode)
    boxes, scores = got["boxes"], got["scores"]

    def alone(b):
        b.output(b.nms(b.arg("boxes", boxes.shape), b.arg("scores", scores.shape), 100, 0.45, 0.3, name="d"), "detections")

    assert not any(s.startswith("nms.best") for s in steps_of(odla, alone, **mode))
    assert np.array_equal(got["detections"], run_hip(alone, {"boxes": boxes, "scores": scores}, **mode)["detections"])
