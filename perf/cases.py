"""The work this framework is used for, as cases that can be timed and compared: whole models through
`smallframework_amd.models.HipExecutor`, single layers and the layout conversion through the C ABI.

A model case runs one forward pass of a benchmark topology with random weights of that architecture, the way a serving
program does: the executor (buffers, weights, plan, whole-model handle) is built once, the pass is repeated.  A layer
case is one call of an entry point of include/small_hip.h on tensors in the packed channel-blocked layout.
"""
import ctypes as C
import math

import torch

from smallframework_amd import capi, models
from smallframework_amd.layout import in_block

CB = capi.CB

MODELS = {"dscnn": models.dscnn, "mobilenet_v1": models.mobilenet_v1, "tiny_yolo_v2": models.tiny_yolo_v2,
          "resnet8_u8": lambda: models.resnet8_u8(discriminating=True)}
# models whose tensors fit one compute unit's LDS run as one launch, the others layer by layer
ONE_LAUNCH = ("dscnn", "resnet8_u8")


def _model(name, model, batch):
    return {"name": name, "op": "model", "model": model, "batch": batch}


def _conv(name, dtype, batch, co, ci, h, w, k, stride):
    return {"name": name, "op": "conv", "dtype": dtype, "batch": batch, "co": co, "ci": ci, "h": h, "w": w, "k": k, "stride": stride}


def _window(name, op, batch, c, h, w, k, stride):
    return {"name": name, "op": op, "batch": batch, "c": c, "h": h, "w": w, "k": k, "stride": stride}


def listed():
    return [
        # one keyword-spotting clip at a time: the smallest call there is, latency is everything
        _model("dscnn_b1", "dscnn", 1),
        # quantised image classification of small images in bulk
        _model("resnet8_u8_b256", "resnet8_u8", 256),
        # classification of one photograph (interactive use), and of a full batch (the headline workload)
        _model("mobilenet_v1_b1", "mobilenet_v1", 1),
        _model("mobilenet_v1_b64", "mobilenet_v1", 64),
        # detection on one video frame, and on the frames of sixteen streams
        _model("tiny_yolo_v2_b1", "tiny_yolo_v2", 1),
        _model("tiny_yolo_v2_b16", "tiny_yolo_v2", 16),
        # the layer-sweep convolution at its large batch: the largest single call
        _conv("conv3x3_256_b64", "f32", 64, 256, 256, 56, 56, 3, 1),
        # a mid-sized convolution on a map and a batch that no tile divides (the regression fixtures' 96 channels, 30x30)
        _conv("conv3x3_96_30x30_b7", "f32", 7, 96, 96, 30, 30, 3, 1),
        # a quantised convolution too large for the whole-model launch
        _conv("conv3x3_u8_96_30x30_b64", "u8", 64, 96, 96, 30, 30, 3, 1),
        # the bandwidth-bound layers of the sweep: depthwise, pooling
        _window("dw3x3_256_b64", "dw", 64, 256, 56, 56, 3, 1),
        _window("maxpool3x3s2_256_b8", "maxpool", 8, 256, 56, 56, 3, 2),
        # NCHW camera images into the layout the first layer reads
        {"name": "pack_3x224x224_b64", "op": "pack", "batch": 64, "c": 3, "h": 224, "w": 224},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(("model", "model", "model", "conv", "conv", "conv_u8", "window", "pack"))
    if op == "model":
        m = rng.choice(sorted(MODELS))
        top = {"dscnn": 256, "resnet8_u8": 1024, "mobilenet_v1": 64, "tiny_yolo_v2": 16}[m]
        return {"op": "model", "model": m, "batch": _log_int(rng, 1, top)}
    if op in ("conv", "conv_u8"):
        while True:
            case = {"op": "conv", "dtype": "f32" if op == "conv" else "u8", "batch": _log_int(rng, 1, 64),
                    "co": CB * _log_int(rng, 1, 64), "ci": CB * _log_int(rng, 1, 64), "h": _log_int(rng, 5, 112),
                    "w": 0, "k": rng.choice((1, 3, 3, 5)), "stride": rng.choice((1, 1, 2))}
            case["w"] = max(5, case["h"] + rng.choice((0, 0, -3, 1, 6)))
            if 2e7 <= work(case)["flops"] <= 1e11 and work(case)["bytes"] <= 4e8:
                return case
    if op == "window":
        while True:
            case = {"op": rng.choice(("dw", "dw", "maxpool")), "batch": _log_int(rng, 1, 64), "c": CB * _log_int(rng, 1, 64),
                    "h": _log_int(rng, 7, 112), "w": 0, "k": 3, "stride": rng.choice((1, 2))}
            if case["op"] == "maxpool":
                case["k"] = rng.choice((2, 3))
            case["w"] = max(5, case["h"] + rng.choice((0, 0, -2, 1, 5)))
            if 1e6 <= work(case)["bytes"] <= 4e8:
                return case
    c = rng.choice((1, 3, 3, CB * _log_int(rng, 1, 16)))
    while True:
        case = {"op": "pack", "batch": _log_int(rng, 1, 64), "c": c, "h": _log_int(rng, 16, 416), "w": 0}
        case["w"] = max(16, case["h"] + rng.choice((0, 0, -5, 3)))
        if 1e6 <= work(case)["bytes"] <= 4e8:
            return case


# ---- shapes -----------------------------------------------------------------------------------------------------------
def _pads(case):
    """Same-style padding for convolutions, none for pooling: t, b, l, r."""
    if case["op"] == "maxpool":
        return (0, 0, 0, 0)
    return models.same_pads(case["h"], case["w"], case["k"], case["k"], case["stride"])


def _out_hw(case):
    t, b, l, r = _pads(case)
    return capi.out_dim(case["h"], t, b, case["k"], case["stride"]), capi.out_dim(case["w"], l, r, case["k"], case["stride"])


# ---- inputs -----------------------------------------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, n, std=1.0):
    return torch.randn(n, generator=g, device="cuda", dtype=torch.float32) * std


def _bytes(g, n):
    return torch.randint(0, 256, (n,), generator=g, device="cuda", dtype=torch.uint8)


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def _stream():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


def _model_weights(model, g):
    """He-normal (float32) or uniform (uint8) weights, drawn in the packed order; padding output channels are zero."""
    w = {}
    for op in model.ops:
        if not op.weight:
            continue
        dense = op.kind != "dw"
        fan_in = op.kh * op.kw * (op.C if dense else 1)
        n = op.weight_elems()
        t = _normal(g, n, math.sqrt(2.0 / fan_in)) if model.dtype == "f32" else _bytes(g, n)
        if dense and op.Co_eff and op.Co_eff < op.Co:
            ib = in_block(op.C)
            v = t.view(op.Co // CB, op.C // ib, op.kh, op.kw, ib, CB)
            v[op.Co_eff // CB, ..., op.Co_eff % CB:] = 0
        w[op.weight] = t.cpu().numpy()
    return w


def _model_input(model, batch, g):
    c, h, wd = model.in_shape
    n = batch * c * h * wd
    if model.input_kind == "u8":
        return _bytes(g, n).cpu().numpy()
    if model.input_kind == "uniform01":
        return torch.rand(n, generator=g, device="cuda", dtype=torch.float32).cpu().numpy()
    return _normal(g, n).cpu().numpy()


def prepare(case, seed):
    g = _gen(seed)
    lib = capi.load()
    if case["op"] == "model":
        m = MODELS[case["model"]]()
        ex = models.HipExecutor(m, case["batch"], weights=_model_weights(m, g), x=_model_input(m, case["batch"], g))
        if case["model"] in ONE_LAUNCH:
            ex.build_one_launch()
            return {"step": ex.forward_one_launch, "out": ex.one_out}
        c, h, w = m.ops[-1].out_shape()
        return {"step": ex.forward, "out": ex.buf[ex.out_name][: case["batch"] * c * h * w]}
    n = case["batch"]
    if case["op"] == "pack":
        x = torch.rand(n * case["c"] * case["h"] * case["w"], generator=g, device="cuda", dtype=torch.float32)
        y = torch.empty_like(x)
        # the image block is 1 x C x H x W; fewer channels than a block form a block of their own
        args = (0, n, 1, case["c"], case["h"], case["w"], CB, CB, _ptr(x), _ptr(y), 4)
        return {"call": lib.small_hip_pack, "args": args, "hold": (x,), "out": y}
    t, b, l, r = _pads(case)
    h, w, k, s = case["h"], case["w"], case["k"], case["stride"]
    ho, wo = _out_hw(case)
    if case["op"] == "maxpool":
        c = case["c"]
        x = _normal(g, n * c * h * w)
        y = torch.empty(n * c * ho * wo, dtype=torch.float32, device="cuda")
        return {"call": lib.small_hip_maxpool2d_f32, "args": (n, k, k, s, t, b, l, r, c, h, w, _ptr(x), _ptr(y)), "hold": (x,), "out": y}
    if case["op"] == "dw":
        c = case["c"]
        x, f, bias = _normal(g, n * c * h * w), _normal(g, c * k * k, math.sqrt(2.0) / k), _normal(g, c, 0.1)
        y = torch.empty(n * c * ho * wo, dtype=torch.float32, device="cuda")
        args = (n, k, k, s, t, b, l, r, c, h, w, _ptr(x), _ptr(f), _ptr(bias), capi.ACT_RELU, 0.0, _ptr(y))
        return {"call": lib.small_hip_depthwise_conv2d_bias_act_f32, "args": args, "hold": (x, f, bias), "out": y}
    co, ci = case["co"], case["ci"]
    shape = (n, k, k, s, t, b, l, r, co, ci, h, w)
    if case["dtype"] == "f32":
        x, f, bias = _normal(g, n * ci * h * w), _normal(g, co * ci * k * k, math.sqrt(2.0 / (ci * k * k))), _normal(g, co, 0.1)
        y = torch.empty(n * co * ho * wo, dtype=torch.float32, device="cuda")
        args = shape + (_ptr(x), _ptr(f), _ptr(bias), capi.ACT_RELU, 0.0, _ptr(y))
        return {"call": lib.small_hip_conv2d_bias_act_f32, "args": args, "hold": (x, f, bias), "out": y}
    # quantised: image and filter centred (the library ADDS the zero points), the output scaled so that about half of its
    # values lie strictly between 0 and 255
    x, f = _bytes(g, n * ci * h * w), _bytes(g, co * ci * k * k)
    y = torch.empty(n * co * ho * wo, dtype=torch.uint8, device="cuda")
    prep = torch.empty(lib.small_hip_conv2d_u8_prepared_filter_bytes(k, k, co, ci), dtype=torch.uint8, device="cuda")
    capi.check(lib.small_hip_conv2d_u8_prepare_filter(k, k, co, ci, _ptr(f), _ptr(prep), _stream()))
    spread = 74.0 * 74.0 * math.sqrt(ci * k * k)
    shift = min(15, max(0, int(math.log2(0.7 * spread / 100.0))))
    quants = (capi.Quant(-128), capi.Quant(-128), capi.Quant(0, 1518500250, 0, shift))
    iq, fq, oq = (C.byref(q) for q in quants)
    args = shape + (_ptr(x), iq, _ptr(prep), fq, _ptr(y), oq)
    return {"call": lib.small_hip_conv2d_u8_prepared, "args": args, "hold": (x, f, prep, quants), "out": y}


def run(state):
    if "step" in state:
        state["step"]()
    else:
        capi.check(state["call"](*state["args"], _stream()))
    return state["out"]


def work(case):
    """Operations (a multiply and an add each) and the bytes of the inputs, weights and outputs, each once.  A model's
    intermediate tensors are not counted: nothing but the present code makes them pass through memory."""
    n = case["batch"]
    if case["op"] == "model":
        m = MODELS[case["model"]]()
        c, h, w = m.in_shape
        co, ho, wo = m.ops[-1].out_shape()
        elems = n * (c * h * w + co * ho * wo) + sum(o.weight_elems() for o in m.ops)
        return {"bytes": m.esize() * elems, "flops": n * m.flops_per_image()}
    if case["op"] == "pack":
        return {"bytes": 8 * n * case["c"] * case["h"] * case["w"], "flops": 0}
    ho, wo = _out_hw(case)
    taps = case["k"] * case["k"]
    if case["op"] in ("dw", "maxpool"):
        c = case["c"]
        weights = c * (taps + 1) if case["op"] == "dw" else 0
        return {"bytes": 4 * (n * c * (case["h"] * case["w"] + ho * wo) + weights),
                "flops": 2 * n * c * ho * wo * taps if case["op"] == "dw" else 0}
    co, ci = case["co"], case["ci"]
    esize = 4 if case["dtype"] == "f32" else 1
    return {"bytes": esize * (n * (ci * case["h"] * case["w"] + co * ho * wo) + co * ci * taps),
            "flops": 2 * n * co * ho * wo * ci * taps}


def tolerance(case):
    """Whole numbers, maxima and moved values are exact.  Float32 sums: about four times the distance of the results from
    the same network or layer computed in float64 (relative 2-norm, measured on an MI355X): DS-CNN 2.4e-7, MobileNetV1
    2.8e-7, Tiny-YOLOv2 1.2e-6, a depthwise 3x3 layer 5.6e-8, a convolution of K = taps x input channels products
    1.05e-7 (K = 32), 3.7e-7 (432), 8.5e-7 (2304), 1.6e-6 (8400), i.e. 1.8e-8 sqrt(K).  The largest single difference was
    6 to 14 times the 2-norm figure."""
    if case["op"] in ("pack", "maxpool") or case.get("dtype") == "u8" or case.get("model") == "resnet8_u8":
        return "exact"
    if case["op"] == "model":
        rel = {"dscnn": 1e-6, "mobilenet_v1": 1.2e-6, "tiny_yolo_v2": 5e-6}[case["model"]]
    elif case["op"] == "dw":
        rel = 2.5e-7
    else:
        rel = max(2.5e-7, 7.2e-8 * math.sqrt(case["ci"] * case["k"] * case["k"]))
    return {"rel": rel, "max": 20 * rel}
