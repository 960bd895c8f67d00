"""The work that users of this library have it do, as cases to time: the layers of quantized networks one by one
(int8 GEMM and convolution), the fp32 operators, and whole networks, through the public entry points of
tennis_amd.capi, tennis_amd.resnet50 and tennis_amd.yolov4.

listed() and draw() describe cases as plain dicts; prepare() makes what a program holds before the call (inputs on the
GPU, layer objects with their weights, a captured graph where the program serves from one), run() is one pass, work()
the bytes and operations that pass cannot do without, tolerance() how far another correct implementation may be off.
"""
import math

import torch

from tennis_amd import capi, resnet50, yolov4


# ---------------------------------------------------------------------------------------------- cases

def listed():
    return [
        # The classifier of an int8 network answering one request: one row against a weight matrix, where the call
        # itself is most of the time (the smallest call a user makes; shapes of the GEMM sweep, config 3).
        {"name": "gemm_i8 1 row", "kind": "gemm_i8", "m": 1, "k": 1024, "n": 1024, "out": "f32", "act": "none", "row_scale": True},
        # A hidden quantized inner product in mid network: sizes that are no multiple of any tile, int8 to int8.
        {"name": "gemm_i8 ragged int8 out", "kind": "gemm_i8", "m": 197, "k": 1500, "n": 777, "out": "i8", "act": "relu", "row_scale": False},
        # The largest GEMM of the sweep: a large batch through a large layer.
        {"name": "gemm_i8 4096", "kind": "gemm_i8", "m": 4096, "k": 4096, "n": 4096, "out": "f32", "act": "none", "row_scale": True},
        # A late layer of a small detection network on one image: odd map, odd channels, stride 2, int8 handed on.
        {"name": "conv_i8 13x13 one image", "kind": "conv_i8", "batch": 1, "c": 100, "h": 13, "w": 13, "cout": 150, "k": 3, "stride": 2,
         "src": "i8", "out": "i8", "act": "leaky_relu"},
        # The quantized chain on fp32 activations (config 2): quantize, 3x3 convolution, bias, ReLU, batch of 32.
        {"name": "conv_i8 config 2", "kind": "conv_i8", "batch": 32, "c": 256, "h": 28, "w": 28, "cout": 256, "k": 3, "stride": 1,
         "src": "f32", "out": "f32", "act": "relu"},
        # One small fp32 layer on one image (config 1).
        {"name": "conv_f32 config 1", "kind": "conv_f32", "batch": 1, "c": 64, "h": 56, "w": 56, "cout": 64, "k": 3, "stride": 1, "act": "relu"},
        # A middle fp32 layer on a small batch, by the direct convolution ...
        {"name": "conv_f32 8 images", "kind": "conv_f32", "batch": 8, "c": 256, "h": 28, "w": 28, "cout": 256, "k": 3, "stride": 1, "act": "relu"},
        # ... and by Winograd F(6,3), the mode the reference's selector gives this shape.
        {"name": "winograd 8 images", "kind": "winograd", "mode": "f63", "fast": False, "batch": 8, "c": 256, "h": 28, "w": 28, "cout": 256,
         "act": "relu"},
        # An fp32 graph kept as separate operators: depthwise block with batch norm, pointwise convolution, residual
        # join, pooling and classifier.
        {"name": "fp32 graph 32 images", "kind": "fp32_graph", "batch": 32, "c": 256, "h": 56, "w": 56, "classes": 1000},
        # A whole int8 network on one image, called layer by layer from the host: the latency of a request.
        {"name": "resnet50 one image", "kind": "resnet50", "batch": 1, "size": 224, "captured": False},
        # The same at the serving batch (config 4), replayed from a captured graph as a server with fixed shapes does.
        {"name": "resnet50 batch 32", "kind": "resnet50", "batch": 32, "size": 224, "captured": True},
        # The detection network (config 5), exact Mish: the largest pass.
        {"name": "yolov4 batch 8", "kind": "yolov4", "batch": 8, "size": 608, "mish": "exact", "captured": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemm_i8", "gemm_i8", "conv_i8", "conv_i8", "conv_i8", "conv_f32", "conv_f32", "winograd", "fp32_graph", "resnet50",
                       "yolov4"])
    if kind == "gemm_i8":
        return {"kind": kind, "m": _log_int(rng, 1, 4096), "k": _log_int(rng, 128, 4096), "n": _log_int(rng, 64, 4096),
                "out": rng.choice(["f32", "f32", "i8"]), "act": rng.choice(["none", "relu"]), "row_scale": rng.random() < 0.5}
    if kind in ("conv_i8", "conv_f32", "winograd"):
        fp32 = kind != "conv_i8"
        while True:     # a layer no larger than the networks' own
            case = {"kind": kind, "batch": _log_int(rng, 1, 32), "c": _log_int(rng, 3, 512), "h": _log_int(rng, 7, 304), "cout": _log_int(rng, 16, 512)}
            case["w"] = case["h"] if rng.random() < 0.5 else _log_int(rng, 7, 304)
            if kind == "winograd":
                case.update(mode=rng.choice(["f63", "f23"]), act=rng.choice(["none", "relu"]))
                case["fast"] = case["mode"] == "f63" and rng.random() < 0.5
            else:
                case.update(k=rng.choice([1, 3, 3, 3, 5]), stride=rng.choice([1, 1, 2]), act=rng.choice(["relu", "leaky_relu"]))
                if not fp32:
                    case.update(src=rng.choice(["f32", "i8"]), out=rng.choice(["f32", "i8"]))
            w = work(case)
            if w["flops"] <= (20e9 if fp32 else 60e9) and w["bytes"] <= 3e8:
                return case
    if kind == "fp32_graph":
        while True:
            case = {"kind": kind, "batch": _log_int(rng, 1, 32), "c": 4 * _log_int(rng, 8, 64), "h": _log_int(rng, 7, 112), "classes": _log_int(rng, 10, 1000)}
            case["w"] = case["h"] + rng.choice([0, 0, 1, 3])
            if case["batch"] * case["c"] * case["h"] * case["w"] <= 32 * 256 * 56 * 56:
                return case
    if kind == "resnet50":
        return {"kind": kind, "batch": _log_int(rng, 1, 32), "size": rng.choice([128, 160, 192, 224]), "captured": rng.random() < 0.5}
    return {"kind": kind, "batch": rng.randint(1, 8), "size": 32 * rng.randint(7, 18), "mish": rng.choice(["exact", "fast"]),
            "captured": rng.random() < 0.5}


# ---------------------------------------------------------------------------------------------- inputs

class _State:
    pass


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, *shape):
    return torch.randn(shape, device="cuda", generator=g)


def _quantize_weights(w):
    """Symmetric int8 per output channel (first axis), half away from zero: the weights and their multipliers."""
    s = 127.0 / w.reshape(w.shape[0], -1).abs().amax(1).clamp_min(1e-12)
    q = w * s.reshape((-1,) + (1,) * (w.dim() - 1))
    return (torch.sign(q) * torch.floor(q.abs() + 0.5)).clamp(-127, 127).to(torch.int8), s


def _network_weights(g, cout, cin, k):
    """One convolution of a network: random-init weights (the He scale) and a small bias, as host arrays."""
    wq, sw = _quantize_weights(_normal(g, cout, cin, k, k) * math.sqrt(2.0 / (cin * k * k)))
    return {"wq": wq.cpu().numpy(), "sw": sw.cpu().numpy(), "bias": (_normal(g, cout) * 0.05).cpu().numpy()}


def _capture(forward, x):
    """A captured graph of forward(x) and its static outputs, as a server with fixed shapes keeps it."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        forward(x)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = forward(x)
    return graph, out


def prepare(case, seed):
    g, s, kind = _generator(seed), _State(), case["kind"]
    s.kind, s.case = kind, case
    if kind == "gemm_i8":
        m, k, n = case["m"], case["k"], case["n"]
        wq, sw = _quantize_weights(_normal(g, n, k) / math.sqrt(k))
        s.layer = capi.GemmI8(wq.t().contiguous())
        s.x = (_normal(g, m, k) * 32).round().clamp(-127, 127).to(torch.int8)
        rows = torch.rand(m, device="cuda", generator=g) + 0.5 if case["row_scale"] else None
        s.kw = {"dq": 1.0 / (32.0 * sw), "row_scale": rows, "bias": _normal(g, n) * 0.1, "act": case["act"]}
        if case["out"] == "i8":
            s.kw.update(q_scales=torch.full((m,), 32.0, device="cuda"), want_f32=False)
    elif kind == "conv_i8":
        b, c, k, p = case["batch"], case["c"], case["k"], case["k"] // 2
        wq, sw = _quantize_weights(_normal(g, case["cout"], c, k, k) / math.sqrt(c * k * k))
        s.layer = capi.Conv2dI8(wq, (p, p, p, p), (case["stride"],) * 2)
        s.x = _normal(g, b, c, case["h"], case["w"])
        x_scale = 127.0 / s.x.abs().max()
        s.kw = {"dq": 1.0 / (x_scale * sw), "bias": _normal(g, case["cout"]) * 0.1, "act": case["act"], "slope": 0.1}
        if case["src"] == "i8":     # what a rectified layer hands on
            s.x = (s.x.clamp_min(0) * x_scale).round().to(torch.int8)
        else:
            s.kw["x_scales"] = x_scale.repeat(b)
        if case["out"] == "i8":
            s.kw.update(q_scales=torch.full((b,), 32.0, device="cuda"), want_f32=False)
    elif kind in ("conv_f32", "winograd"):
        c, k = case["c"], case.get("k", 3)
        s.pads = (k // 2,) * 4
        s.x = _normal(g, case["batch"], c, case["h"], case["w"])
        s.w = _normal(g, case["cout"], c, k, k) * math.sqrt(2.0 / (c * k * k))
        s.bias = _normal(g, case["cout"]) * 0.1
        if kind == "winograd":
            s.layer = capi.Winograd(s.w, s.pads, mode=case["mode"])
    elif kind == "fp32_graph":
        c = case["c"]
        s.x = _normal(g, case["batch"], c, case["h"], case["w"])
        s.dw, s.pw = _normal(g, 1, c, 3, 3) / 3, _normal(g, c, c, 1, 1) * math.sqrt(2.0 / c)
        s.mean, s.var = _normal(g, c) * 0.1, torch.rand(c, device="cuda", generator=g) + 0.5
        s.scale, s.shift, s.bias = torch.rand(c, device="cuda", generator=g) + 0.5, _normal(g, c) * 0.1, _normal(g, c) * 0.1
        s.fc, s.fc_bias = _normal(g, c, case["classes"]) / math.sqrt(c), _normal(g, case["classes"]) * 0.1
    elif kind == "resnet50":
        desc = resnet50.layers()
        stem, blocks, fc = desc
        params = {spec.name: _network_weights(g, spec.cout, spec.cin, spec.k) for spec in [stem] + [c for blk in blocks for c in blk if c is not None]}
        head = _network_weights(g, fc[1], fc[0], 1)
        params["fc"] = dict(head, wq=head["wq"].reshape(fc[1], fc[0]).T.copy())
        s.net = resnet50.ResNet50Int8(desc, params)
        s.x = torch.rand((case["batch"], 3, case["size"], case["size"]), device="cuda", generator=g)
        s.net.set_scales(s.net.calibrate(s.x), case["batch"])
    elif kind == "yolov4":
        L, heads = yolov4.layers()
        srcs, chans = yolov4.resolve(L)
        params = {i: _network_weights(g, l["filters"], 3 if srcs[i][0] < 0 else chans[srcs[i][0]], l["size"])
                  for i, l in enumerate(L) if l["type"] == "conv"}
        s.net = yolov4.YoloV4Int8(L, heads, params, mish=case["mish"])
        s.x = torch.rand((case["batch"], 3, case["size"], case["size"]), device="cuda", generator=g)
        s.net.calibrate(s.x)
    else:
        raise ValueError(kind)
    s.graph = None
    if case.get("captured"):
        s.graph, s.out = _capture(s.net.forward, s.x)
    return s


# ---------------------------------------------------------------------------------------------- one pass

def run(s):
    kind = s.kind
    if kind in ("gemm_i8", "conv_i8"):
        return [o for o in s.layer(s.x, **s.kw) if o is not None]
    if kind == "conv_f32":
        return capi.conv2d_f32(s.x, s.w, s.pads, (s.case["stride"],) * 2, bias=s.bias, act=s.case["act"], slope=0.1)
    if kind == "winograd":
        return s.layer(s.x, bias=s.bias, act=s.case["act"], fast=s.case["fast"])
    if kind == "fp32_graph":
        y = capi.relu(capi.fused_batch_norm(capi.depthwise_conv2d(s.x, s.dw, (1, 1, 1, 1)), s.mean, s.var, s.scale, s.shift))
        joined = capi.add(capi.conv2d_f32(y, s.pw, bias=s.bias), s.x, act="relu")
        pooled = capi.pooling2d(joined, "max", (3, 3), (2, 2), (1, 1, 1, 1))
        features = capi.global_pooling2d(pooled, "avg").reshape(s.x.shape[0], -1)
        return [joined, pooled, capi.add_bias(capi.inner_prod_f32(features, s.fc), s.fc_bias)]
    if s.graph is not None:
        s.graph.replay()
        return s.out
    return s.net.forward(s.x)


# ---------------------------------------------------------------------------------------------- what a pass needs

def _out_size(case):
    k, st = case.get("k", 3), case.get("stride", 1)
    return [(case[d] + 2 * (k // 2) - k) // st + 1 for d in ("h", "w")]


def work(case):
    kind = case["kind"]
    if kind == "gemm_i8":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": m * k + k * n + m * n * (4 if case["out"] == "f32" else 1) + 8 * n, "flops": 2.0 * m * k * n}
    if kind in ("conv_i8", "conv_f32", "winograd"):
        b, c, cout, k = case["batch"], case["c"], case["cout"], case.get("k", 3)
        ho, wo = _out_size(case)
        size_w = 1 if kind == "conv_i8" else 4
        size_in, size_out = 4 if case.get("src", "f32") == "f32" else 1, 4 if case.get("out", "f32") == "f32" else 1
        # Winograd stands for the direct convolution: its operations are counted as that one's
        return {"bytes": b * c * case["h"] * case["w"] * size_in + cout * c * k * k * size_w + b * cout * ho * wo * size_out,
                "flops": 2.0 * b * cout * ho * wo * c * k * k}
    if kind == "fp32_graph":
        b, c, h, w, classes = (case[q] for q in ("batch", "c", "h", "w", "classes"))
        one = 4.0 * b * c * h * w
        pooled = one / 4
        # separate operators, each reading its inputs and writing its output: depthwise, batch norm, relu, pointwise
        # (2 each), join (3), max pooling and global pooling of its output
        return {"bytes": 11 * one + one + 2 * pooled + 4.0 * (c * c + c * classes + b * (c + 3 * classes)),
                "flops": 2.0 * b * c * h * w * (9 + c) + 2.0 * b * c * classes}
    # whole networks: the image, every weight and the outputs once; activations can stay on the chip
    b, size = case["batch"], case["size"]
    if kind == "resnet50":
        desc = resnet50.layers()
        weights = sum(p.cin * p.cout * p.k * p.k for p in [desc[0]] + [c for blk in desc[1] for c in blk if c is not None]) + desc[2][0] * desc[2][1]
        return {"bytes": 12.0 * b * size * size + weights + 4.0 * b * desc[2][1], "flops": 2.0 * resnet50.total_macs(desc, b, size)}
    L, heads = yolov4.layers()
    srcs, chans = yolov4.resolve(L)
    weights = sum(l["filters"] * (3 if srcs[i][0] < 0 else chans[srcs[i][0]]) * l["size"] ** 2 for i, l in enumerate(L) if l["type"] == "conv")
    outs = sum(L[h]["filters"] * (size // d) ** 2 for h, d in zip(heads, (8, 16, 32)))
    return {"bytes": 12.0 * b * size * size + weights + 4.0 * b * outs, "flops": 2.0 * yolov4.total_macs(L, b, size)}


def tolerance(case):
    # The int8 path and the reference-order Winograd promise every rounding of the operator chain they stand for.
    if case["kind"] in ("gemm_i8", "conv_i8", "resnet50"):
        return "exact"
    if case["kind"] == "yolov4":
        # the exact Mish is the chain's values; the short form may requantize a value in a million one step off
        return "exact" if case["mish"] == "exact" else {"rel": 1e-3}
    if case["kind"] == "winograd" and not case["fast"]:
        return "exact"
    return {"rel": 1e-5}      # fp32 sums in another order
