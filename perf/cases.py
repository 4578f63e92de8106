"""The work that users of this framework have it do, as cases that can be timed.

A user records a computation once, compiles it into a context and then executes it
on one input after the other: the classifier and detector images of the benchmark
configurations, the sequences of the encoder, on device buffers (a serving loop)
or on host arrays (the Python harness).  A program here is one computation with one
context, kept as such a user keeps it; a state is one set of inputs and results.

Families and the ranges that `draw` covers:
  mnist     softmax regression, 1 .. 4096 digits, host arrays or device buffers
  resnet50  int8 / fp16 / bf16 / fp32, 1 .. 256 images of 96 .. 320 pixels (every
            size in between, so odd maps too), host arrays or device buffers
  bert      encoder of base size, bf16 in both modes / fp16 / fp32, 1 .. 64 sequences
            of 8 .. 512 tokens with their own lengths in the mask
  yolov3    network to its three heads, fp16 / bf16, 1 .. 16 images of 320 .. 608 pixels
  yolo_post box decode and non-maximum suppression on given heads, fp32, 1 .. 16 images
  vision    operators between the convolutions, fp16 / fp32, odd channels and maps
"""
import importlib
import math
import random

import numpy as np
import torch
import torch.nn.functional as F

_pkg = importlib.import_module("heterogeneity-aware-lowering-and-optimization_amd")
_odla = _pkg.odla

_TORCH = {np.dtype(np.float32): torch.float32, np.dtype(np.int32): torch.int32}


def listed():
    return [
        # the smallest call: 64 digits as the Python harness hands them over, numpy in and out
        {"name": "mnist_fp32_b64_host", "family": "mnist", "batch": 64, "io": "host"},
        # throughput serving, the two plans that the headline metric names
        {"name": "resnet50_int8_b256", "family": "resnet50", "mode": "int8", "batch": 256, "hw": 224, "io": "device"},
        {"name": "resnet50_fp16_b256", "family": "resnet50", "mode": "fp16", "batch": 256, "hw": 224, "io": "device"},
        # one image at a time: latency
        {"name": "resnet50_fp16_b1", "family": "resnet50", "mode": "fp16", "batch": 1, "hw": 224, "io": "device"},
        # a small batch as it comes, of images that no tile size divides
        {"name": "resnet50_int8_b13_hw237", "family": "resnet50", "mode": "int8", "batch": 13, "hw": 237, "io": "device"},
        # the default precision, a few images from host arrays
        {"name": "resnet50_fp32_b4_host", "family": "resnet50", "mode": "fp32", "batch": 4, "hw": 224, "io": "host"},
        # encoder: the benchmark batch, long sequences in the other bf16 mode, one short query
        {"name": "bert_bf16_b64_s128", "family": "bert", "mode": "bf16", "batch": 64, "seq": 128},
        {"name": "bert_bf16acc_b8_s384", "family": "bert", "mode": "bf16acc", "batch": 8, "seq": 384},
        {"name": "bert_bf16_b1_s41", "family": "bert", "mode": "bf16", "batch": 1, "seq": 41},
        # detector: the benchmark batch; its post-processing on the heads of that batch
        {"name": "yolov3_fp16_b16_hw416", "family": "yolov3", "mode": "fp16", "batch": 16, "hw": 416},
        {"name": "yolo_post_fp32_b16_hw416", "family": "yolo_post", "batch": 16, "hw": 416},
        # what stands between the convolutions of a vision graph: normalisation, pooling, up-sampling, concatenation
        {"name": "vision_fp16_b64_c96_hw75", "family": "vision", "mode": "fp16", "batch": 64, "channels": 96, "hw": 75},
    ]


def _log(rng, lo, hi):
    """A whole number in lo..hi, spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    family = rng.choice(["resnet50"] * 4 + ["bert"] * 3 + ["yolov3", "yolov3", "mnist", "yolo_post", "vision"])
    if family == "mnist":
        return {"family": family, "batch": _log(rng, 1, 4096), "io": rng.choice(["host", "device"])}
    if family == "resnet50":
        mode = rng.choice(["int8", "fp16", "int8", "fp16", "bf16", "fp32"])
        io = rng.choice(["device", "device", "host"])
        hw = rng.choice([224, rng.randint(96, 320)])
        most = {"fp32": 16}.get(mode, 256) if io == "device" else 16
        batch = _log(rng, 1, max(1, min(most, 256 * 224 * 224 // (hw * hw))))
        return {"family": family, "mode": mode, "batch": batch, "hw": hw, "io": io}
    if family == "bert":
        mode = rng.choice(["bf16", "bf16acc", "bf16", "bf16acc", "fp16", "fp32"])
        seq = rng.choice([128, _log(rng, 8, 512)])
        batch = _log(rng, 1, max(1, min(64, (1024 if mode == "fp32" else 8192) // seq)))
        return {"family": family, "mode": mode, "batch": batch, "seq": seq}
    if family == "yolov3":
        hw = rng.choice([416, 32 * rng.randint(10, 19)])
        batch = _log(rng, 1, max(1, 16 * 416 * 416 // (hw * hw)))
        return {"family": family, "mode": rng.choice(["fp16", "fp16", "bf16"]), "batch": batch, "hw": hw}
    if family == "yolo_post":
        hw = 32 * rng.randint(10, 19)
        return {"family": family, "batch": _log(rng, 1, max(1, 16 * 416 * 416 // (hw * hw))), "hw": hw}
    channels, hw = _log(rng, 3, 512), _log(rng, 7, 150)
    batch = _log(rng, 1, max(1, min(256, (64 * 96 * 75 * 75) // (channels * hw * hw))))
    return {"family": family, "mode": rng.choice(["fp16", "fp32"]), "batch": batch, "channels": channels, "hw": hw}


# ---------------------------------------------------------------- programs --
_weights = {}   # the seeded synthetic weights of a family, made once per process


def _kept(key, make):
    if key not in _weights:
        _weights[key] = make()
    return _weights[key]


def _resnet_forward(w, x, taps):
    """The fp32 network on the CPU: ranges for the quantisation table, size of the logits."""
    def conv(x, name, stride, pad, relu):
        y = F.conv2d(x, torch.from_numpy(w[name + ".w"]), torch.from_numpy(w[name + ".b"]), stride, pad)
        taps[name] = y
        if relu:
            y = taps[name + ".relu"] = torch.relu(y)
        return y

    taps["input"] = x
    x = F.max_pool2d(conv(x, "stem", 2, 3, True), 3, 2, 1)
    for si, (mid, blocks, stride) in enumerate(_pkg.models.RESNET50_STAGES):
        for bi in range(blocks):
            s, p = stride if bi == 0 else 1, "l%db%d" % (si + 1, bi)
            identity = conv(x, p + "ds", s, 0, False) if bi == 0 else x
            y = conv(conv(conv(x, p + "c1", 1, 0, True), p + "c2", s, 1, True), p + "c3", 1, 0, False)
            x = taps[p + "out"] = torch.relu(y + identity)
    return x.mean((2, 3)) @ torch.from_numpy(w["fc.w"])


def _resnet_weights():
    """Weights with unit-size logits (as a trained classifier's are of the order of ten, not of thousands),
    and the quantisation table of a two-image calibration."""
    models = _pkg.models
    w = models.resnet50_weights()
    taps = {}
    with torch.no_grad():
        logits = _resnet_forward(w, torch.from_numpy(models.resnet50_input(2, seed=1000)["input"]), taps)
    w["fc.w"] = (w["fc.w"] / float("%.3g" % float(logits.std()))).astype(np.float32)
    # three digits: the last bits of a CPU's sums are not part of the table
    ranges = {n: tuple(float("%.3g" % float(f(taps[n]))) for f in (torch.min, torch.max)) for n in models.resnet50_quantized_values()}
    return w, models.resnet50_quant_entries(w, ranges)


def _build_vision(b, case):
    n, c, hw = case["batch"], case["channels"], case["hw"]
    rng = np.random.default_rng(5)
    per_channel = lambda f: f(c).astype(np.float32)
    x = b.arg("x", (n, c, hw, hw))
    y = b.batchnorm(x, b.const("mean", per_channel(rng.standard_normal)), b.const("var", per_channel(rng.random) + np.float32(0.5)),
                    1e-5, b.const("gamma", per_channel(rng.standard_normal)), b.const("beta", per_channel(rng.standard_normal)), name="bn")
    y = b.leaky_relu(y, 0.1, name="act")
    p = b.maxpool(y, (3, 3), (2, 2), (1, 1, 1, 1), name="maxpool")
    a = b.avgpool(y, (2, 2), (1, 1), (0, 0, 0, 0), name="avgpool")
    up = b.resize_nearest(p, (hw, hw), name="up")
    b.output(b.concat([up, b.add(y, x, name="res")], 1, name="cat"), "features")
    b.output(b.softmax(b.reshape(b.reduce_mean(a, (2, 3), True, name="gap"), (n, c), name="flat"), -1, name="prob"), "prob")


class _Program:
    """A recorded computation and the context that executes it."""

    def __init__(self, case):
        family, mode = case["family"], case.get("mode", "fp32")
        table = None
        if family == "resnet50":
            w, entries = _kept("resnet50", _resnet_weights)
            table = _odla.quant_table(entries) if mode == "int8" else None
        self.b = b = _odla.HipBuilder(fp16=mode == "fp16", bf16={"bf16": "performance", "bf16acc": "accuracy"}.get(mode, False),
                                      quant_table=table)
        self.session = None
        if family == "mnist":
            _pkg.models.build_mnist(b, _kept("mnist", _pkg.models.mnist_weights), case["batch"])
        elif family == "resnet50":
            _pkg.models.build_resnet50(b, w, case["batch"], case["hw"])
        elif family == "bert":
            _pkg.models_bert.build_bert(b, _kept("bert", _pkg.models_bert.bert_weights), case["batch"], case["seq"])
        elif family == "yolov3":
            # (detections of a half-precision network are in an order that its last bits decide: they are a case of their own)
            w = _kept("yolov3", lambda: _pkg.models_yolo.yolov3_weights(head_scale=(0.05, 0.05, 0.05)))
            _pkg.models_yolo.build_yolov3(b, w, case["batch"], case["hw"], postprocess=False)
        elif family == "yolo_post":
            _pkg.models_yolo.build_yolo_postprocess(b, case["batch"], case["hw"])
        elif family == "vision":
            _build_vision(b, case)
        else:
            raise ValueError("unknown family %r" % family)
        self.session = b.session()

    def __del__(self):
        if getattr(self, "session", None) is not None:
            self.session.close()
        self.b.destroy()


_last = {}   # the program of the case at hand: one at a time


def _program(case):
    key = repr(sorted((k, v) for k, v in case.items() if k != "name"))
    if key not in _last:
        _last.clear()
        _last[key] = _Program(case)
    return _last[key]


# ------------------------------------------------------------------ states --
class _State:
    def __init__(self, program, feeds, host):
        self.program, self.host = program, host
        b = program.b
        if host:
            self.feeds = {k: v.cpu().numpy() for k, v in feeds.items()}
            return
        self.feeds = feeds
        self.results = {n: torch.empty(shape, dtype=_TORCH[dt], device="cuda") for n, (h, shape, dt) in b.outs.items()}
        self.args = [(b.args[n][0], t.data_ptr()) for n, t in feeds.items()]
        self.outs = [(b.outs[n][0], t.data_ptr()) for n, t in self.results.items()]


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    normal = lambda *shape: torch.randn(shape, generator=gen, device="cuda")
    uniform = lambda *shape: torch.rand(shape, generator=gen, device="cuda")
    n, family = case["batch"], case["family"]
    if family == "mnist":
        feeds = {"x": uniform(n, 784)}
    elif family == "resnet50":
        feeds = {"input": normal(n, 3, case["hw"], case["hw"])}       # mean and deviation of the data set taken out
    elif family == "bert":
        seq = case["seq"]
        ids = torch.randint(0, _pkg.models_bert.BERT_BASE["vocab"], (n, seq), generator=gen, device="cuda", dtype=torch.int32)
        lengths = torch.randint((seq + 1) // 2, seq + 1, (n, 1), generator=gen, device="cuda")   # padded to the longest
        mask = (torch.arange(seq, device="cuda")[None, :] < lengths).float()
        feeds = {"input_ids": ids, "attention_mask": mask.reshape(n, 1, 1, seq)}
    elif family == "yolov3":
        feeds = {"input": uniform(n, 3, case["hw"], case["hw"])}
    elif family == "yolo_post":
        feeds = {}
        for i, stride in enumerate((32, 16, 8)):
            g = case["hw"] // stride
            h = normal(n, 3, 5 + _pkg.models_yolo.NUM_CLASSES, g, g)
            h[:, :, 4:] -= 2.0                                        # most boxes hold nothing: about one score in a hundred passes
            feeds["head%d" % i] = h.reshape(n, -1, g, g)
    else:
        feeds = {"x": normal(n, case["channels"], case["hw"], case["hw"])}
    return _State(_program(case), feeds, case.get("io") == "host")


def run(state):
    s = state.program.session
    if state.host:
        return s.run(state.feeds)
    L, ctx = s.L, s.ctx
    for h, p in state.args:
        L.odla_BindToArgument(h, p, ctx)
    for h, p in state.outs:
        L.odla_BindToOutput(h, p, ctx)
    s.execute()
    return state.results


# -------------------------------------------------------------------- work --
_BYTES = {"int8": 1, "fp16": 2, "bf16": 2, "bf16acc": 2, "fp32": 4}


def work(case):
    """Arguments, weights at their compute type and results once each; operations of the convolutions and products."""
    family, n, es = case["family"], case["batch"], _BYTES[case.get("mode", "fp32")]
    if family == "mnist":
        return {"bytes": 4 * (n * (784 + 10) + 7850), "flops": 2 * n * 7840}
    if family == "resnet50":
        hw = case["hw"]
        layers = _pkg.models.resnet50_conv_elements(n, hw)
        flops = sum(v[0] for v in layers.values()) + 2 * n * 2048 * 1000
        weights = sum(v[2] for v in layers.values()) + 2048 * 1000
        return {"bytes": 4 * n * (3 * hw * hw + 2000) + es * weights, "flops": flops}
    if family == "bert":
        seq, cfg = case["seq"], _pkg.models_bert.BERT_BASE
        H, FF = cfg["hidden"], cfg["ffn"]
        weights = cfg["layers"] * (4 * H * H + 2 * H * FF)
        rows = min(cfg["vocab"], n * seq) * H
        return {"bytes": n * seq * (4 + 4 + 4 * H) + es * (weights + rows), "flops": 1e9 * n * _pkg.models_bert.bert_gflop_per_sequence(seq)}
    if family == "yolov3":
        hw, macs, weights, size = case["hw"], 0, 0, case["hw"]
        heads = {"1": 32, "2": 16, "3": 8}
        for name, cout, cin, k, stride, _ in _pkg.models_yolo.yolov3_conv_specs():
            if name[0] == "d":
                size //= stride
                at = size
            else:
                at = hw // heads[name[1]] // (2 if name.endswith(".lat") else 1)
            macs += cout * cin * k * k * at * at
            weights += cout * cin * k * k
        out = 255 * sum((hw // s) ** 2 for s in (32, 16, 8))
        return {"bytes": 4 * n * (3 * hw * hw + out) + es * weights, "flops": 2 * n * macs}
    if family == "yolo_post":
        boxes = 3 * sum((case["hw"] // s) ** 2 for s in (32, 16, 8))
        return {"bytes": 4 * n * boxes * (85 + 4 + 80) + 4 * n * 300, "flops": 4 * n * boxes * 85}
    elements = n * case["channels"] * case["hw"] ** 2
    return {"bytes": 4 * (3 * elements + n * case["channels"]), "flops": 20 * elements}


def tolerance(case):
    """What the storage types give through each network; the sums themselves are 32-bit everywhere."""
    mode, family = case.get("mode", "fp32"), case["family"]
    if mode == "bf16acc":
        return {"rel": 1.2e-2}       # operands of twelve layers rounded to bf16
    if mode == "bf16":
        return {"rel": 2.5e-2}       # every tensor rounded to bf16
    if mode == "fp16":
        return {"rel": 2e-3 if family == "vision" else 5e-3}
    if mode == "int8":
        return {"rel": 1e-5}         # whole numbers up to the fp32 head
    return {"rel": 3e-5 if family in ("resnet50", "bert") else 1e-5, "differ": 0.01}


if __name__ == "__main__":
    for c in listed() + [draw(random.Random(s)) for s in range(12)]:
        w = work(c)
        print("%-90s %10.2f MB %10.3f GFLOP" % (c, w["bytes"] / 1e6, w["flops"] / 1e9))
