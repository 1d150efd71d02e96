"""The work that programs have this library do, as cases that can be timed.

Most cases are short sequences of calls of the C ABI on device tensors, the way a
network's layers make them; two run a whole text model through ``shadow_amd.Network``.
Sizes are those of the library's own benchmark and tests, and around them.  Device
memory comes from torch tensors, work goes to torch's current stream, and nothing is
waited for except where the entry point itself hands its result to the host.

    listed()          the cases
    draw(rng)         one more case of the same ranges
    prepare(case, s)  the inputs of seed s, output buffers and prepared arguments
    run(state)        one pass; returns the outputs
    work(case)        bytes and operations that the pass cannot do without
    tolerance(case)   how far another correct implementation's outputs may be off
"""
import ctypes
import math

import torch

import shadow_amd

# enums of include/shadow_hip.h
ABS, SQRT, EXP = 0, 2, 4
ADD, SUB, MUL, DIV, MAX = 0, 1, 2, 3, 5
R_SUM, R_MAX, R_AVG = 1, 2, 4
RELU, SIGMOID, TANH = 1, 3, 5


def listed():
    return [
        # One image's late feature map through the activations: seven calls that take no
        # time on the device to speak of, as every layer of an unbatched program makes them.
        {"name": "unary_one_map", "kind": "unary", "n": 1, "c": 256, "h": 14, "w": 14},
        # The benchmark's own step: a batch of early feature maps through the same seven.
        {"name": "unary_batch64", "kind": "unary", "n": 64, "c": 256, "h": 56, "w": 56},
        # Binary operators on pairs that broadcast against each other (attention biases,
        # per-row and per-column terms) and the channel bias, both at the benchmark's size.
        {"name": "broadcast", "kind": "broadcast", "n": 16, "c": 32, "h": 128, "w": 256},
        # Pooled features, channel maxima, batch statistics and a full sum of one feature
        # map tensor, at the benchmark's size.
        {"name": "reduce", "kind": "reduce", "n": 32, "c": 512, "h": 28, "w": 28},
        # A text model of gated residual blocks, one image per call, host arrays in and
        # class probabilities out: launches and host work, as an interactive program sees it.
        {"name": "network_one_image", "kind": "network", "n": 1, "c": 256, "h": 14, "w": 14, "blocks": 4, "device": False},
        # The same model on a batch that is already on the device: a served classifier.
        {"name": "network_batch32", "kind": "network", "n": 32, "c": 512, "h": 28, "w": 28, "blocks": 2, "device": True},
        # Stem pooling (3x3 maximum by two), a 3x3 average at stride 1 and the whole-plane
        # average that closes a classifier.
        {"name": "pooling", "kind": "pooling", "n": 32, "c": 64, "h": 112, "w": 112},
        # Class scores: per pixel of a segmentation head, per box, per image.
        {"name": "softmax", "kind": "softmax", "n": 16, "classes": 150, "h": 72, "w": 72, "boxes": 8732, "box_classes": 21},
        # A single-shot detection head: L2 normalisation of the feature map per position,
        # two score maps to box-major order, concatenated, softmax over the classes.
        {"name": "detection_head", "kind": "detection", "n": 16, "c": 512, "side": 38, "classes": 21},
        # Group, instance and layer normalisation of one tensor with scale and bias.
        {"name": "norms", "kind": "norms", "n": 16, "c": 256, "h": 56, "w": 56, "groups": 32},
        # Response normalisation across channels and the maximum by two behind it, on the
        # odd-sided maps such networks have.
        {"name": "lrn_pool", "kind": "lrn", "n": 44, "c": 96, "h": 55, "w": 55},
        # A decoder stage: bilinear upsampling, concatenation with the skip maps, channel
        # shuffle, and the skip maps resampled along a flow field.
        {"name": "decoder", "kind": "decoder", "n": 8, "c": 64, "h": 56, "w": 56, "out_h": 112, "out_w": 112},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """Batches from one to 64, channels from a few to a thousand, maps from 7 to 128 a
    side, odd sizes included, kept to the number of elements that the listed cases reach."""
    kind = rng.choice(["unary", "broadcast", "reduce", "network", "pooling", "softmax", "detection", "norms", "lrn", "decoder"])
    most = {"unary": 51380224, "broadcast": 16777216, "reduce": 12845056, "network": 12845056, "pooling": 25690112,
            "softmax": 12441600, "detection": 11829248, "norms": 12845056, "lrn": 12777600, "decoder": 6422528}[kind]
    while True:
        n, c = _log_int(rng, 1, 64), _log_int(rng, 8, 1024)
        h = _log_int(rng, 7, 128)
        w = h if rng.random() < 0.6 else _log_int(rng, 7, 128)
        if kind == "decoder":
            c = min(c, 256)
        if kind == "unary":
            case = {"kind": kind, "n": n, "c": c, "h": h, "w": w}
            size = n * c * h * w
        elif kind == "network":
            blocks = rng.randint(1, 4)
            case = {"kind": kind, "n": n, "c": c, "h": h, "w": w, "blocks": blocks, "device": n * c * h * w > 300000}
            size = n * c * h * w * max(1, blocks // 2)
        elif kind == "softmax":
            case = {"kind": kind, "n": n, "classes": _log_int(rng, 2, 320), "h": h, "w": w,
                    "boxes": _log_int(rng, 100, 9000), "box_classes": rng.randint(2, 91)}
            size = max(n * case["classes"] * h * w, n * case["boxes"] * case["box_classes"])
        elif kind == "detection":
            side = _log_int(rng, 10, 64)
            case = {"kind": kind, "n": n, "c": c, "side": side, "classes": rng.randint(2, 91)}
            size = n * side * side * max(c, 4 * case["classes"])
        elif kind == "norms":
            groups = rng.choice([1, 2, 4, 8, 16, 32])
            c = max(groups, c - c % groups)
            case = {"kind": kind, "n": n, "c": c, "h": h, "w": w, "groups": groups}
            size = n * c * h * w
        elif kind == "decoder":
            f = rng.choice([2.0, 2.0, 1.5, rng.uniform(1.1, 2.5)])
            case = {"kind": kind, "n": n, "c": c, "h": h, "w": w, "out_h": int(h * f), "out_w": int(w * f)}
            size = n * c * case["out_h"] * case["out_w"]
        else:
            case = {"kind": kind, "n": n, "c": c, "h": h, "w": w}
            size = n * c * h * w
        if 2000 <= size <= most:
            return case


# ---------------------------------------------------------------------------
# helpers
# ---------------------------------------------------------------------------
class _Inputs:
    """Device tensors of one seed."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def normal(self, *shape, std=1.0):
        t = torch.randn(shape, generator=self.gen, device="cuda", dtype=torch.float32)
        return t if std == 1.0 else t.mul_(std)

    def uniform(self, lo, hi, *shape):
        return torch.rand(shape, generator=self.gen, device="cuda", dtype=torch.float32).mul_(hi - lo).add_(lo)


def _out(*shape):
    return torch.empty(shape, device="cuda", dtype=torch.float32)


def _scratch(nbytes):
    return torch.empty(max(16, nbytes), device="cuda", dtype=torch.uint8)


class _Calls:
    """A sequence of C-ABI calls with their arguments in hand."""

    def __init__(self):
        self.lib = shadow_amd.hip()
        self.stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        self.calls, self.kept, self.outputs = [], [], {}

    def add(self, name, *args):
        """Tensors stand for their device pointers, lists for host arrays of ints."""
        given = []
        for a in args:
            if isinstance(a, torch.Tensor):
                self.kept.append(a)
                a = a.data_ptr()
            elif isinstance(a, list):
                a = shadow_amd.ints(a)
            given.append(a)
        self.calls.append((getattr(self.lib, "shdw_hip_" + name), tuple(given) + (self.stream,)))

    def run(self):
        for fn, args in self.calls:
            rc = fn(*args)
            if rc:
                shadow_amd.check(rc)
        return self.outputs


# ---------------------------------------------------------------------------
# sequences of C-ABI calls
# ---------------------------------------------------------------------------
def _unary(case, gen):
    n, c, h, w = case["n"], case["c"], case["h"], case["w"]
    x, count, s = gen.normal(n, c, h, w, std=2.0), n * c * h * w, _Calls()
    gamma, beta = gen.uniform(0.5, 1.5, c), gen.uniform(-0.1, 0.1, c)
    o = s.outputs = {k: _out(n, c, h, w) for k in ("relu", "sigmoid", "exp", "abs", "sqrt", "tanh", "scale_relu")}
    s.add("activate", RELU, 0.0, count, x, o["relu"])
    s.add("activate", SIGMOID, 0.0, count, x, o["sigmoid"])
    s.add("unary", EXP, count, x, o["exp"])
    s.add("unary", ABS, count, x, o["abs"])
    s.add("unary", SQRT, count, o["abs"], o["sqrt"])
    s.add("activate", TANH, 0.0, count, x, o["tanh"])
    s.add("scale_bias", count, c, h * w, x, gamma, beta, 1, o["scale_relu"])
    return s


def _broadcast(case, gen):
    n, c, h, w = case["n"], case["c"], case["h"], case["w"]
    a, b = gen.normal(n, 1, h, w), gen.uniform(0.5, 2.0, 1, c, h, 1)
    x, bias, s = gen.normal(n, c, h, w), gen.uniform(-1.0, 1.0, 1, c, 1, 1), _Calls()
    s.outputs = {k: _out(n, c, h, w) for k in ("mul", "sub", "div", "max", "bias")}
    for key, op in (("mul", MUL), ("sub", SUB), ("div", DIV), ("max", MAX)):
        s.add("broadcast_binary", op, 4, [n, 1, h, w], [1, c, h, 1], [n, c, h, w], a, b, s.outputs[key])
    s.add("broadcast_binary", ADD, 4, [n, c, h, w], [1, c, 1, 1], [n, c, h, w], x, bias, s.outputs["bias"])
    return s


def _reduce(case, gen):
    n, c, h, w = case["n"], case["c"], case["h"], case["w"]
    x, shape, s = gen.normal(n, c, h, w), [n, c, h, w], _Calls()
    s.outputs = {"sum_hw": _out(n, c), "avg_hw": _out(n, c), "max_c": _out(n, h, w), "sum_all": _out(1), "avg_nhw": _out(c)}
    for key, op, axes in (("sum_hw", R_SUM, [2, 3]), ("avg_hw", R_AVG, [2, 3]), ("max_c", R_MAX, [1]),
                          ("sum_all", R_SUM, [0, 1, 2, 3]), ("avg_nhw", R_AVG, [0, 2, 3])):
        need = s.lib.shdw_hip_reduce_workspace_bytes(4, shadow_amd.ints(shape), len(axes), shadow_amd.ints(axes))
        s.add("reduce", op, 4, shape, len(axes), axes, x, s.outputs[key], _scratch(need), need)
    return s


def _pool_out(size, kernel, stride, pad):
    return (size + 2 * pad - kernel) // stride + 1


def _pooling(case, gen):
    n, c, h, w = case["n"], case["c"], case["h"], case["w"]
    oh, ow, s = _pool_out(h, 3, 2, 1), _pool_out(w, 3, 2, 1), _Calls()
    x = gen.normal(n, c, h, w).relu_()
    o = s.outputs = {"max": _out(n, c, oh, ow), "avg": _out(n, c, oh, ow), "plane": _out(n, c, 1, 1)}
    s.add("pooling2d", [n, c, h, w], 0, 3, 3, 2, 2, 1, 1, [n, c, oh, ow], x, o["max"])
    s.add("pooling2d", [n, c, oh, ow], 1, 3, 3, 1, 1, 1, 1, [n, c, oh, ow], o["max"], o["avg"])
    s.add("pooling2d", [n, c, oh, ow], 1, oh, ow, 1, 1, 0, 0, [n, c, 1, 1], o["avg"], o["plane"])
    return s


def _softmax(case, gen):
    n, k, h, w, boxes, bk = (case[f] for f in ("n", "classes", "h", "w", "boxes", "box_classes"))
    s = _Calls()
    maps, rows, images = gen.normal(n, k, h, w, std=3.0), gen.normal(n, boxes, bk, std=3.0), gen.normal(n, 1000, std=3.0)
    s.outputs = {"maps": _out(n, k, h, w), "boxes": _out(n, boxes, bk), "images": _out(n, 1000)}
    s.add("softmax", n, k, h * w, maps, s.outputs["maps"])
    s.add("softmax", n * boxes, bk, 1, rows, s.outputs["boxes"])
    s.add("softmax", n, 1000, 1, images, s.outputs["images"])
    return s


def _detection_parts(case):
    """(priors per cell, side) of the two score maps."""
    return [(4, case["side"]), (6, (case["side"] + 1) // 2)]


def _detection(case, gen):
    n, c, side, k = case["n"], case["c"], case["side"], case["classes"]
    s, parts = _Calls(), _detection_parts(case)
    x, scale = gen.normal(n, c, side, side).relu_(), gen.uniform(10.0, 20.0, c)
    boxes = sum(p * e * e for p, e in parts)
    o = s.outputs = {"feature": _out(n, c, side, side), "scores": _out(n, boxes, k), "prob": _out(n, boxes, k)}
    need = s.lib.shdw_hip_ssd_normalize_workspace_bytes(n, c, side * side, 0)
    s.add("ssd_normalize", n, c, side * side, 0, 1e-10, x, scale, 0, o["feature"], _scratch(need))
    at = 0
    for p, e in parts:
        score, moved, length = gen.normal(n, p * k, e, e, std=2.0), _out(n, e, e, p * k), e * e * p * k
        s.add("permute", 4, [n, p * k, e, e], [0, 2, 3, 1], score, moved)
        s.add("copy_chunks", n, length, moved, length, 0, o["scores"], boxes * k, at)
        at += length
    s.add("softmax", n * boxes, k, 1, o["scores"], o["prob"])
    return s


def _norms(case, gen):
    n, c, h, w, g = case["n"], case["c"], case["h"], case["w"], case["groups"]
    x, s, plane = gen.normal(n, c, h, w, std=1.5), _Calls(), h * w
    x += gen.normal(1, c, 1, 1)
    scale, bias = gen.uniform(0.5, 1.5, c), gen.normal(c, std=0.1)
    s.outputs = {k: _out(n, c, h, w) for k in ("group", "instance", "layer")}
    for key, outer, inner, each in (("group", n * g, c // g * plane, plane), ("instance", n * c, plane, plane), ("layer", n * plane, c, 1)):
        need = s.lib.shdw_hip_group_norm_workspace_bytes(outer, inner)
        s.add("group_norm_ws", outer, inner, 1e-5, x, scale, bias, c, each, s.outputs[key], _scratch(need), need)
    return s


def _lrn(case, gen):
    n, c, h, w = case["n"], case["c"], case["h"], case["w"]
    oh, ow, s = _pool_out(h, 3, 2, 0), _pool_out(w, 3, 2, 0), _Calls()
    x = gen.normal(n, c, h, w, std=4.0).relu_()
    s.outputs = {"lrn": _out(n, c, h, w), "max": _out(n, c, oh, ow)}
    s.add("lrn", [n, c, h, w], 5, 1e-4, 0.75, 1.0, x, s.outputs["lrn"])
    s.add("pooling2d", [n, c, h, w], 0, 3, 3, 2, 2, 0, 0, [n, c, oh, ow], s.outputs["lrn"], s.outputs["max"])
    return s


def _decoder(case, gen):
    n, c, h, w, oh, ow = (case[f] for f in ("n", "c", "h", "w", "out_h", "out_w"))
    s, plane = _Calls(), oh * ow
    x, skip = gen.normal(n, c, h, w), gen.normal(n, c, oh, ow)
    # the identity grid displaced by a smooth field of a few cells
    ys = torch.linspace(-1.0, 1.0, oh, device="cuda").view(1, oh, 1).expand(n, oh, ow)
    xs = torch.linspace(-1.0, 1.0, ow, device="cuda").view(1, 1, ow).expand(n, oh, ow)
    flow = torch.nn.functional.interpolate(gen.normal(n, 2, 8, 8, std=0.04), size=(oh, ow), mode="bilinear")
    grid = (torch.stack((xs, ys), 1) + flow).permute(0, 2, 3, 1).contiguous()
    both = _out(n, 2 * c, oh, ow)
    o = s.outputs = {"up": _out(n, c, oh, ow), "shuffled": _out(n, 2 * c, oh, ow), "warped": _out(n, c, oh, ow)}
    s.add("resize", [n, c, h, w], [n, c, oh, ow], 1, 0, x, o["up"])
    s.add("copy_chunks", n, c * plane, o["up"], c * plane, 0, both, 2 * c * plane, 0)
    s.add("copy_chunks", n, c * plane, skip, c * plane, 0, both, 2 * c * plane, c * plane)
    s.add("shuffle_channel", n, 2 * c, plane, 2, both, o["shuffled"])
    s.add("grid_sample", [n, c, oh, ow], [n, c, oh, ow], 1, 0, skip, grid, o["warped"])
    return s


# ---------------------------------------------------------------------------
# a text model through Network
# ---------------------------------------------------------------------------
def _network_text(case):
    """Residual blocks x + scale(gate(relu(scale(norm(x))))), the gate a sigmoid of the
    plane averages; then the plane averages of the last block and their softmax."""
    n, c, h, w = case["n"], case["c"], case["h"], case["w"]
    both = "[{axis, s_i, [1]}; {has_scale, s_i, [1]}; {has_bias, s_i, [1]}]"
    blobs, ops, x = [], [], "x"
    for b in range(case["blocks"]):
        blobs += ["%s%d" % (name, b) for name in ("mean", "variance", "gamma", "beta", "last_gamma", "last_beta")]
        ops += ["[BatchNorm] | [norm%d] | [3 1 1] | [%s; mean%d; variance%d] | [norm%d] | [{eps, s_f, [0.001]}]" % (b, x, b, b, b),
                "[Scale] | [scale%d] | [3 1 3] | [norm%d; gamma%d; beta%d] | [scale%d] | %s" % (b, b, b, b, b, both),
                "[Activate] | [relu%d] | [1 1 1] | [scale%d] | [scale%d] | [{type, s_i, [1]}]" % (b, b, b),
                "[Pooling] | [squeeze%d] | [1 1 2] | [scale%d] | [squeeze%d] | [{pool, s_i, [1]}; {global_pooling, s_i, [1]}]" % (b, b, b),
                "[Activate] | [gate%d] | [1 1 1] | [squeeze%d] | [gate%d] | [{type, s_i, [3]}]" % (b, b, b),
                "[Binary] | [gated%d] | [2 1 1] | [scale%d; gate%d] | [gated%d] | [{operation, s_i, [2]}]" % (b, b, b, b),
                "[Scale] | [last%d] | [3 1 3] | [gated%d; last_gamma%d; last_beta%d] | [last%d] | %s" % (b, b, b, b, b, both),
                "[Eltwise] | [sum%d] | [2 1 1] | [last%d; %s] | [block%d] | [{operation, s_i, [1]}]" % (b, b, x, b),
                "[Activate] | [out%d] | [1 1 1] | [block%d] | [block%d] | [{type, s_i, [1]}]" % (b, b, b)]
        x = "block%d" % b
    ops += ["[Reduce] | [pool] | [1 1 2] | [%s] | [pool] | [{operation, s_i, [4]}; {axes, v_i, [2 # 3]}]" % x,
            "[Flatten] | [flat] | [1 1 0] | [pool] | [flat] | []",
            "[Softmax] | [prob] | [1 1 1] | [flat] | [prob] | [{axis, s_i, [1]}]"]
    head = ["[gated_blocks]", "[{out_blob, v_s, [prob # pool]}]", "[%s]" % "; ".join("{%s, float, [%d]}" % (b, c) for b in blobs),
            "[Input] | [in] | [0 1 1] | [] | [x] | [{x, v_i, [%d # %d # %d # %d]}]" % (n, c, h, w)]
    return "\n".join(head + ops) + "\n"


class _DeviceArray:
    """A tensor's memory as Network.forward takes a device input."""

    def __init__(self, tensor):
        self.tensor, self.ptr = tensor, tensor.data_ptr()


class _Model(shadow_amd.Network):
    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


class _NetworkState:
    def __init__(self, case, gen):
        c, weights = case["c"], []
        for _ in range(case["blocks"]):
            weights += [gen.normal(c, std=0.2), gen.uniform(0.5, 1.5, c), gen.uniform(0.5, 1.5, c), gen.normal(c, std=0.1),
                        gen.uniform(0.5, 1.5, c), gen.normal(c, std=0.1)]
        x = gen.normal(case["n"], c, case["h"], case["w"])
        self.net = _Model(_network_text(case), [v.cpu().numpy() for v in weights], device_input=case["device"])
        self.feed = {"x": _DeviceArray(x) if case["device"] else x.cpu().numpy()}

    def run(self):
        self.net.forward(self.feed)
        return {"prob": self.net.blob("prob"), "pool": self.net.blob("pool")}


_KINDS = {"unary": _unary, "broadcast": _broadcast, "reduce": _reduce, "pooling": _pooling, "softmax": _softmax,
          "detection": _detection, "norms": _norms, "lrn": _lrn, "decoder": _decoder, "network": _NetworkState}


def prepare(case, seed):
    return _KINDS[case["kind"]](case, _Inputs(seed))


def run(state):
    return state.run()


# ---------------------------------------------------------------------------
# what a pass cannot do without, and what its results may be off by
# ---------------------------------------------------------------------------
def work(case):
    """Floats read and written with every input read once and every output written once,
    and roughly an operation per value that a step works on."""
    kind, n = case["kind"], case["n"]
    if kind == "softmax":
        maps, boxes, images = n * case["classes"] * case["h"] * case["w"], n * case["boxes"] * case["box_classes"], n * 1000
        return {"bytes": 8.0 * (maps + boxes + images), "flops": 4.0 * (maps + boxes + images)}
    if kind == "detection":
        feature = n * case["c"] * case["side"] ** 2
        scores = n * sum(p * e * e for p, e in _detection_parts(case)) * case["classes"]
        return {"bytes": 8.0 * feature + 12.0 * scores, "flops": 4.0 * (feature + scores)}
    t = n * case["c"] * case["h"] * case["w"]
    if kind == "unary":
        return {"bytes": 4.0 * 8 * t, "flops": 7.0 * t}
    if kind == "broadcast":
        small = n * case["h"] * case["w"] + case["c"] * case["h"]
        return {"bytes": 4.0 * (small + 6 * t), "flops": 5.0 * t}
    if kind == "reduce":
        return {"bytes": 4.0 * (t + 2 * n * case["c"] + n * case["h"] * case["w"] + case["c"]), "flops": 5.0 * t}
    if kind == "network":
        return {"bytes": 4.0 * (t + 2 * n * case["c"]), "flops": 10.0 * case["blocks"] * t}
    if kind == "pooling":
        pooled = n * case["c"] * _pool_out(case["h"], 3, 2, 1) * _pool_out(case["w"], 3, 2, 1)
        return {"bytes": 4.0 * (t + 2 * pooled + n * case["c"]), "flops": 19.0 * pooled}
    if kind == "norms":
        return {"bytes": 16.0 * t, "flops": 3 * 7.0 * t}
    if kind == "lrn":
        pooled = n * case["c"] * _pool_out(case["h"], 3, 2, 0) * _pool_out(case["w"], 3, 2, 0)
        return {"bytes": 8.0 * t + 4.0 * pooled, "flops": 6.0 * t + 9.0 * pooled}
    up = n * case["c"] * case["out_h"] * case["out_w"]
    return {"bytes": 4.0 * (t + 5 * up) + 8.0 * n * case["out_h"] * case["out_w"], "flops": 14.0 * up}


def tolerance(case):
    """Elementwise, selecting and moving operators and the sums that are kept in the
    reference's order have one right answer to the bit.  Sums and means are kept in 64
    bits and rounded once, so another order changes a last place here and there; the
    figures are four times the distance from an evaluation in 64 bits throughout
    (sums 4.5e-8 and 6e-8 at most, norms 6e-8 and 2.9e-7, networks 2.3e-6 and 3.3e-6)."""
    kind = case["kind"]
    if kind == "reduce":
        return {"rel": 2e-7, "max": 2.5e-7}
    if kind == "norms":
        return {"rel": 2.5e-7, "max": 1.2e-6}
    if kind == "network":
        return {"rel": 1e-5, "max": 1.3e-5}
    return "exact"
