"""The convolution calls whose speed this library is held to, over the range of layers that an image network has it
run: batch 1 and batches of tens, 3x3, 1x1 and 7x7 filters and irregular ones, stride 1 and 2, 16-bit and 32-bit
storage, single layers through Conv2D::forward (the dispatcher's own choice of kernel, nothing tuned beforehand) and
bottleneck blocks as chains of calls or as one captured graph. Sizes are those of the benchmark's five
configurations and of examples/workloads.json, or generic ones.

A case is a dict of plain values. `kind` "layer" is one call; "block" is a bottleneck block (1x1 reduce, 3x3, 1x1
expand and, with `project`, the 1x1 projection of the block's input), every layer's output returned.
"""
import ctypes
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cuda-inference_amd"))
import gie  # noqa: E402

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32, "tf32": torch.float32}


def _layer(n, c, h, w, o, kh, kw, stride, ph, pw, precision, bias=True, relu=True):
    return {"kind": "layer", "n": n, "c": c, "h": h, "w": w, "o": o, "kh": kh, "kw": kw, "stride": stride, "ph": ph,
            "pw": pw, "precision": precision, "bias": bias, "relu": relu}


def _block(n, h, w, c, mid, o, stride, project, graph, precision):
    return {"kind": "block", "n": n, "h": h, "w": w, "c": c, "mid": mid, "o": o, "stride": stride, "project": project,
            "graph": graph, "precision": precision}


def listed():
    cases = {
        # one image through a residual block deep in a network: three small dependent calls, where latency counts
        "block_n1_14": _block(1, 14, 14, 1024, 256, 1024, 1, False, False, "fp16"),
        # one image, strict FP32 (the library's FP32 path and the benchmark's first configuration)
        "fp32_3x3_n1": _layer(1, 64, 56, 56, 64, 3, 3, 1, 1, 1, "fp32"),
        # a 3x3 layer in the middle of a network, batch 32
        "fp16_3x3_14": _layer(32, 256, 14, 14, 256, 3, 3, 1, 1, 1, "fp16"),
        # a wide pointwise layer, batch 64: the largest output
        "fp16_1x1_28": _layer(64, 256, 28, 28, 1024, 1, 1, 1, 0, 0, "fp16"),
        # a network's first layer, batch 64: three input channels, the most output pixels
        "fp16_7x7s2_stem": _layer(64, 3, 224, 224, 64, 7, 7, 2, 3, 3, "fp16"),
        # a long reduction over few pixels, small batch
        "bf16_3x3_7": _layer(8, 512, 7, 7, 512, 3, 3, 1, 1, 1, "bf16"),
        # an early 3x3 layer, batch 32: few channels, many pixels
        "bf16_3x3_56": _layer(32, 64, 56, 56, 64, 3, 3, 1, 1, 1, "bf16"),
        # a strided projection shortcut
        "bf16_1x1s2_56": _layer(16, 256, 56, 56, 512, 1, 1, 2, 0, 0, "bf16"),
        # an irregular layer: odd image sides, channels that fill no tile, no ReLU
        "fp16_3x3_ragged": _layer(3, 130, 9, 11, 70, 3, 3, 1, 1, 1, "fp16", relu=False),
        # a whole downsampling block with its projection, batch 32, replayed as one captured graph
        "block_down_graph": _block(32, 56, 56, 256, 128, 512, 2, True, True, "fp16"),
        # the most arithmetic: a 3x3 layer of a plain (not residual) network
        "bf16_3x3_big": _layer(16, 256, 56, 56, 256, 3, 3, 1, 1, 1, "bf16"),
        # a 3x3 layer in strict FP32, batch 32
        "fp32_3x3_28": _layer(32, 128, 28, 28, 128, 3, 3, 1, 1, 1, "fp32"),
    }
    return [dict(case, name=name) for name, case in cases.items()]


# No drawn case has more arithmetic or traffic than the largest listed one of its storage.
_MOST_BYTES = 120e6
_MOST_FLOPS = {"fp16": 59e9, "bf16": 59e9, "fp32": 7.3e9, "tf32": 7.3e9}


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def _channels(rng, lo, hi):
    """Mostly multiples of 32, some of 8, some of nothing."""
    v, r = _log_int(rng, lo, hi), rng.random()
    return v if r < 0.2 else max(8, v // 8 * 8) if r < 0.4 else max(32, v // 32 * 32)


def _draw(rng):
    precision = rng.choice(("fp16", "fp16", "fp16", "bf16", "bf16", "bf16", "fp32", "tf32"))
    n, side = _log_int(rng, 1, 64), _log_int(rng, 7, 56)
    other = side if rng.random() < 0.7 else _log_int(rng, 7, 56)
    kind = rng.choice(("3x3", "3x3", "3x3", "1x1", "1x1", "1x1", "stem", "other", "block"))
    bias, relu = rng.random() < 0.9, rng.random() < 0.8
    if kind == "stem":
        side = rng.choice((96, 128, 160, 192, 224, 224, 224, 225))
        return _layer(n, 3, side, side, rng.choice((32, 64, 64, 96)), 7, 7, 2, 3, 3, precision, bias, relu)
    if kind == "block":
        mid = _channels(rng, 64, 512)
        return _block(n, side, side, mid * rng.choice((2, 4)), mid, mid * 4, rng.choice((1, 1, 2)),
                      rng.random() < 0.5, rng.random() < 0.5, rng.choice(("fp16", "bf16")))
    c, o = _channels(rng, 16, 1024 if kind == "1x1" else 512), _channels(rng, 16, 1024 if kind == "1x1" else 512)
    stride = 2 if rng.random() < 0.25 else 1
    if kind == "3x3":
        return _layer(n, c, side, other, o, 3, 3, stride, 1, 1, precision, bias, relu)
    if kind == "1x1":
        return _layer(n, c, side, other, o, 1, 1, stride, 0, 0, precision, bias, relu)
    kh, kw = rng.choice(((5, 5), (1, 7), (7, 1), (1, 3), (3, 1)))
    return _layer(n, c, side, other, o, kh, kw, 1, kh // 2, kw // 2, precision, bias, relu)


def draw(rng):
    while True:
        case = _draw(rng)
        w = work(case)
        if w["bytes"] <= _MOST_BYTES and w["flops"] <= _MOST_FLOPS[case["precision"]]:
            return case


def _problems(case):
    """The case's layers in call order, and for each the layer whose output it reads (-1: the case's input)."""
    if case["kind"] == "layer":
        return [(gie.Problem(case["n"], case["c"], case["h"], case["w"], case["o"], case["kh"], case["kw"],
                             case["stride"], case["stride"], case["ph"], case["pw"], precision=case["precision"],
                             has_bias=case["bias"], relu=case["relu"]), -1)]
    n, h, w, s, prec = case["n"], case["h"], case["w"], case["stride"], case["precision"]
    reduce = gie.Problem(n, case["c"], h, w, case["mid"], 1, 1, precision=prec)
    conv = gie.Problem(n, case["mid"], h, w, case["mid"], 3, 3, s, s, 1, 1, precision=prec)
    expand = gie.Problem(n, case["mid"], conv.out_h, conv.out_w, case["o"], 1, 1, precision=prec, relu=False)
    layers = [(reduce, -1), (conv, 0), (expand, 1)]
    if case["project"]:
        layers.append((gie.Problem(n, case["c"], h, w, case["o"], 1, 1, s, s, precision=prec, relu=False), -1))
    return layers


def _numel(shape):
    return shape[0] * shape[1] * shape[2] * shape[3]


def _inputs(case, seed):
    """x uniform in [-1, 1], weights uniform in [-1, 1] / sqrt(fan-in), bias uniform in [-0.1, 0.1], in storage type."""
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def uniform(shape, scale):
        return ((torch.rand(shape, generator=gen, device="cuda") * 2 - 1) * scale).to(DTYPES[case["precision"]])

    layers = _problems(case)
    x = uniform(layers[0][0].x_shape(), 1.0)
    weights = [uniform(p.w_shape(), p.gemm_k ** -0.5) for p, _ in layers]
    biases = [uniform((p.out_channels,), 0.1) if p.has_bias else None for p, _ in layers]
    return layers, x, weights, biases


def prepare(case, seed):
    layers, x, weights, biases = _inputs(case, seed)
    outputs = [torch.empty(p.y_shape(), dtype=x.dtype, device="cuda") for p, _ in layers]
    sources = [x if src < 0 else outputs[src] for _, src in layers]
    sizes = [gie.workspace_size(p) for p, _ in layers]
    workspace = torch.empty(max(max(sizes), 1), dtype=torch.uint8, device="cuda")
    state = {"outputs": outputs, "keep": [x, weights, biases, workspace], "graph": None, "calls": []}
    if case.get("graph"):
        steps = []
        for (p, _), src, w, b, y in zip(layers, sources, weights, biases, outputs):
            plan = gie.Plan(p, gie.select(p)[0])
            steps.append((plan, src.data_ptr(), w.data_ptr(), b.data_ptr(), y.data_ptr(), workspace.data_ptr(),
                          workspace.numel()))
        torch.cuda.synchronize()  # the capture runs the chain once, on a stream of its own
        state["graph"] = gie.Graph()
        state["graph"].capture(steps)
        state["keep"].append(steps)
        return state
    stream = torch.cuda.current_stream().cuda_stream or None
    for (p, _), src, w, b, y in zip(layers, sources, weights, biases, outputs):
        tensors = [ctypes.byref(gie.tensor(t.data_ptr(), p, which)) if t is not None else None
                   for t, which in ((src, "x"), (w, "w"), (b, "b"), (y, "y"))]
        state["calls"].append((ctypes.byref(p.c()), *tensors, workspace.data_ptr(), workspace.numel(), stream, None))
    return state


def run(state):
    if state["graph"] is not None:
        state["graph"].launch()
        return state["outputs"]
    forward = gie.capi().gie_conv2d_forward
    for args in state["calls"]:
        gie.check(forward(*args), "Conv2D::forward")
    return state["outputs"]


def work(case):
    layers = _problems(case)
    values = _numel(layers[0][0].x_shape()) + sum(_numel(p.w_shape()) + _numel(p.y_shape()) for p, _ in layers)
    values += sum(p.out_channels for p, _ in layers if p.has_bias)
    return {"bytes": float(values * layers[0][0].esize), "flops": float(sum(p.flops() for p, _ in layers))}


def tolerance(case):
    # Every layer sums in FP32 and rounds once to the storage type, so another order of the sums moves a value by an
    # FP32 rounding (FP32, TF32) or, now and then, across a rounding boundary of its 16-bit type by one step; in a
    # block such steps pass through the layers that follow. About four times what the library's own kernels (other
    # tiles, split reductions) differ by from each other over these ranges: 1.4e-5 (fp16) and 3.7e-5 (bf16) in a
    # layer, 8.6e-5 and 2.7e-4 at a block's end, 6.3e-7 in FP32; the largest difference is one rounding step.
    rel = {"fp16": (6e-5, 3.5e-4), "bf16": (1.6e-4, 1.1e-3), "fp32": (2.5e-6, 2.5e-6), "tf32": (2.5e-6, 2.5e-6)}
    most = {"fp16": 4e-3, "bf16": 3e-2, "fp32": 2.5e-5, "tf32": 2.5e-5}
    return {"rel": rel[case["precision"]][case["kind"] == "block"], "max": most[case["precision"]]}


def _conv64(p, x, w, b):
    """The fused layer in 64 bits: one matrix product for each filter tap, over the padded input."""
    x = torch.nn.functional.pad(x, (p.pad_w, p.pad_w, p.pad_h, p.pad_h)).permute(1, 0, 2, 3)
    y = torch.zeros((p.out_channels, p.batch * p.out_h * p.out_w), dtype=torch.float64, device=x.device)
    for r in range(p.kernel_h):
        for s in range(p.kernel_w):
            tap = x[:, :, r:r + (p.out_h - 1) * p.stride_h + 1:p.stride_h, s:s + (p.out_w - 1) * p.stride_w + 1:p.stride_w]
            y += w[:, :, r, s].contiguous() @ tap.reshape(p.in_channels, -1)
    if b is not None:
        y += b[:, None]
    if p.relu:
        y.clamp_(min=0)
    return y.reshape(p.out_channels, p.batch, p.out_h, p.out_w).permute(1, 0, 2, 3).contiguous()


def exact(case, seed):
    layers, x, weights, biases = _inputs(case, seed)
    x, outputs = x.double(), []
    for (p, src), w, b in zip(layers, weights, biases):
        source = x if src < 0 else outputs[src]
        outputs.append(_conv64(p, source, w.double(), b.double() if b is not None else None))
    return outputs
