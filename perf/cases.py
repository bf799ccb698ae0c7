"""The work a program built on this package has it do: quantizing tensors, binary affine and convolution layers in
inference and training, and a whole quantized multi-layer perceptron built with the ``F.*`` front end.

``listed()`` names fixed cases, ``draw(rng)`` gives one more of the same ranges, ``prepare`` makes what a program holds
before the call, ``run`` is one pass through the public entry points, ``work`` what a pass cannot do without and
``tolerance`` how far another correct implementation may be off.
"""
import math

import numpy as np
import torch

import nnabla_amd as nn
import nnabla_amd.functions as F
from nnabla_amd import kernels
from nnabla_amd.ext_utils import get_extension_context


def listed():
    return [
        # The output of a small network's last layer put on the fixed-point grid: the smallest call there is.
        quantize("quantize-scores", "fixed", 64, 1000, 1, 1),
        # The weights of one 3 x 3 convolution rounded to powers of two, and the gradient through the rounding, as
        # every training step of a power-of-two network does for each of its layers.
        quantize("quantize-weights", "pow2", 512, 512, 3, 3, backward=True),
        # Activations of a large map quantized with a running range for the whole tensor: one training step.
        quantize("quantize-map", "minmax", 64, 256, 56, 56, backward=True, ranges="running"),
        # The same with a learnt range per channel, over maps of odd extent.
        quantize("quantize-odd-map", "minmax", 64, 256, 27, 27, backward=True, ranges="learnt"),
        # One row through a wide binary layer: answering a single request.
        affine("affine-row", "weight", 1, 4096, 11008),
        # A batch of rows through the same layer, its extents no multiples of anything.
        affine("affine-ragged", "connect", 300, 4095, 11007, bias=True),
        # A training step of the layer at the largest batch.
        affine("affine-train", "weight", 4096, 4096, 11008, bias=True, backward=True),
        # Inference of a binary convolution in the middle of an image network.
        convolution("conv-inference", "weight", 32, 256, 14, 14, 256, 3),
        # A training step of an early binary convolution: few channels, a large map.
        convolution("conv-train-early", "connect", 32, 64, 56, 56, 64, 3, backward=True),
        # A training step of a strided convolution under incremental quantization, half of its weights fixed.
        convolution("conv-train-inq", "inq", 16, 128, 28, 28, 256, 3, stride=2, bias=True, backward=True),
        # A small perceptron on a small batch, run as a graph: many launches with little work in each.
        mlp("mlp-small", 20, 250, 4),
        # The perceptron at the sizes of a wide layer stack.
        mlp("mlp-wide", 1024, 4096, 4),
    ]


def quantize(name, op, batch, channels, height, width, backward=False, ranges="none"):
    return dict(name=name, kind="quantize", op=op, batch=batch, channels=channels, height=height, width=width,
                backward=backward, ranges=ranges)


def affine(name, op, rows, inputs, outputs, bias=False, backward=False):
    return dict(name=name, kind="affine", op=op, rows=rows, inputs=inputs, outputs=outputs, bias=bias,
                backward=backward)


def convolution(name, op, batch, channels, height, width, maps, kernel, stride=1, bias=False, backward=False):
    return dict(name=name, kind="convolution", op=op, batch=batch, channels=channels, height=height, width=width,
                maps=maps, kernel=kernel, stride=stride, bias=bias, backward=backward)


def mlp(name, batch, width, layers):
    return dict(name=name, kind="mlp", batch=batch, width=width, layers=layers)


def _log(rng, low, high):
    """A whole number between low and high, spread over its logarithm; every second one a multiple of eight where
    it is large enough to be one."""
    v = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    if v >= 16 and rng.random() < 0.5:
        v -= v % 8
    return max(low, min(high, v))


def draw(rng):
    kind = rng.choice(("quantize", "affine", "convolution", "mlp"))
    if kind == "quantize":
        op = rng.choice(("fixed", "pow2", "minmax"))
        c = quantize("", op, _log(rng, 1, 64), _log(rng, 16, 512), *([rng.choice((1, 3, 7, 13, 14, 27, 28, 55, 56))] * 2),
                     backward=rng.random() < 0.5,
                     ranges=rng.choice(("running", "learnt")) if op == "minmax" else "none")
        while c["batch"] * c["channels"] * c["height"] * c["width"] > 64 * 256 * 56 * 56:
            c["batch"] = max(1, c["batch"] // 2)
    elif kind == "affine":
        c = affine("", rng.choice(("weight", "connect")), _log(rng, 1, 4096), _log(rng, 64, 4096),
                   _log(rng, 64, 11008), bias=rng.random() < 0.5)
        c["backward"] = c["rows"] >= 16 and rng.random() < 0.5
    elif kind == "convolution":
        size = rng.choice((7, 13, 14, 27, 28, 55, 56))
        c = convolution("", rng.choice(("weight", "connect", "inq")), _log(rng, 1, 64), _log(rng, 16, 512), size, size,
                        _log(rng, 16, 512), rng.choice((1, 3, 3, 5)), stride=rng.choice((1, 1, 2)),
                        bias=rng.random() < 0.5, backward=rng.random() < 0.5)
        # at most the products of the early layer's training step
        most = 3 * 2.0 * 32 * 56 * 56 * 64 * 576
        while c["batch"] > 1 and work(c)["flops"] > most:
            c["batch"] //= 2
        while work(c)["flops"] > most:
            c["maps"] = max(16, c["maps"] // 2)
            c["channels"] = max(16, c["channels"] // 2)
    else:
        c = mlp("", _log(rng, 1, 1024), _log(rng, 64, 4096), rng.randint(2, 4))
    del c["name"]
    return c


# ---------------------------------------------------------------------------------------------- quantizers

def _normal(gen, shape, scale):
    return torch.randn(shape, generator=gen, device="cuda") * scale


def _prepare_quantize(c, gen):
    shape = (c["batch"], c["channels"], c["height"], c["width"])
    s = {"x": _normal(gen, shape, 0.5 if c["op"] == "pow2" else 2.0)}
    if c["backward"]:
        s["dy"] = _normal(gen, shape, 1e-2)
    if c["op"] == "minmax":
        per = (1, c["channels"], 1, 1) if c["ranges"] == "learnt" else (1, 1, 1, 1)
        s["qr_min"] = -4.0 + 0.1 * torch.rand(per, generator=gen, device="cuda")
        s["qr_max"] = 4.0 + 0.1 * torch.rand(per, generator=gen, device="cuda")
        s["ql_min"] = torch.full(per, 0.0, device="cuda")
        s["ql_max"] = torch.full(per, 255.0, device="cuda")
    return s


def _run_quantize(c, s):
    x = s["x"]
    if c["op"] == "fixed":
        out = [kernels.fixed_point_quantize(x, True, 8, 2.0 ** -4)]
        if c["backward"]:
            out.append(kernels.fixed_point_quantize_backward(s["dy"], x, True, 8, 2.0 ** -4, True))
    elif c["op"] == "pow2":
        out = [kernels.pow2_quantize(x, True, True, 4, 1)]
        if c["backward"]:
            out.append(kernels.pow2_quantize_backward(s["dy"], x, True, True, 4, 1, True))
    else:
        running = c["ranges"] == "running"
        r = (s["qr_min"], s["qr_max"], s["ql_min"], s["ql_max"])
        y, scale = kernels.min_max_quantize(x, *r, decay=0.999, x_min_max=running, ema=running)
        out = [y, scale, s["qr_min"], s["qr_max"]]
        if c["backward"]:
            out += kernels.min_max_quantize_backward(s["dy"], x, *r, scale, True, x_min_max=running, ema=running,
                                                     want_min=not running, want_max=not running)
    return out


# ------------------------------------------------------------------------------------- binary affine layers

def _prepare_affine(c, gen):
    M, K, N = c["rows"], c["inputs"], c["outputs"]
    s = {"x": _normal(gen, (M, K), 1.0), "W": _normal(gen, (K, N), 0.02),
         "b": _normal(gen, (N,), 0.1) if c["bias"] else None}
    if c["backward"]:
        s["dy"] = _normal(gen, (M, N), 1e-2)
    return s


def _run_affine(c, s):
    if c["op"] == "weight":
        y, Wb, alpha = kernels.binary_weight_affine(s["x"], s["W"], s["b"])
        out = [y, Wb, alpha]
    else:
        (y, Wb), alpha = kernels.binary_connect_affine(s["x"], s["W"], s["b"]), None
        out = [y, Wb]
    if c["backward"]:
        out += kernels.binary_affine_backward(s["dy"], s["x"], s["W"], Wb, alpha, want=(True, True, c["bias"]))
    return out


# -------------------------------------------------------------------------------------------- convolutions

def _out_extent(c, n):
    return (n + 2 * (c["kernel"] // 2) - c["kernel"]) // c["stride"] + 1


def _prepare_convolution(c, gen):
    B, C, H, W, O, k = c["batch"], c["channels"], c["height"], c["width"], c["maps"], c["kernel"]
    s = {"x": _normal(gen, (B, C, H, W), 1.0).clamp_(min=0.0),
         "W": _normal(gen, (O, C, k, k), math.sqrt(2.0 / (C * k * k))),
         "b": _normal(gen, (O,), 0.1) if c["bias"] else None}
    if c["backward"]:
        s["dy"] = _normal(gen, (B, O, _out_extent(c, H), _out_extent(c, W)), 1e-2)
    if c["op"] == "inq":
        # the layer as it stands half way through its schedule: the larger half of its weights fixed
        s["I"] = torch.zeros(O, C, k, k, dtype=torch.int32, device="cuda")
        s["old_W"], s["old_I"] = s["W"].clone(), s["I"].clone()
        kernels.inq_convolution(s["x"][:1], s["W"], s["I"], s["old_W"], s["old_I"], s["b"], *_geometry(c), 1, 4,
                                kernels.INQ_LARGEST_ABS)
    return s


def _geometry(c):
    return (c["kernel"] // 2,) * 2, (c["stride"],) * 2, (1, 1)


def _run_convolution(c, s):
    x, W, b = s["x"], s["W"], s["b"]
    want = (True, True, c["bias"])
    if c["op"] == "inq":
        y = kernels.inq_convolution(x, W, s["I"], s["old_W"], s["old_I"], b, *_geometry(c), 1, 4,
                                    kernels.INQ_NO_SELECTION)
        out = [y, W, s["I"]]
        if c["backward"]:
            out += kernels.convolution_backward(s["dy"], x, W, *_geometry(c), 1, want=want)
        return out
    if c["op"] == "weight":
        y, Wb, alpha = kernels.binary_weight_convolution(x, W, b, *_geometry(c), 1)
        out = [y, Wb, alpha]
    else:
        (y, Wb), alpha = kernels.binary_connect_convolution(x, W, b, *_geometry(c), 1), None
        out = [y, Wb]
    if c["backward"]:
        out += kernels.binary_convolution_backward(s["dy"], x, W, Wb, alpha, *_geometry(c), 1, want=want)
    return out


# ------------------------------------------------------------------- a quantized perceptron as an F.* graph

class _OnDevice(object):
    """A variable's data where it lies on the device, for torch to look at."""

    def __init__(self, v, dtype=np.float32):
        self.__cuda_array_interface__ = {"shape": v.shape, "typestr": np.dtype(dtype).str, "version": 2,
                                         "data": (v.device_pointer(dtype), False)}


def _variable(tensor):
    v = nn.Variable(tuple(tensor.shape))
    v.set_data(tensor.cpu().numpy())
    return v


def _prepare_mlp(c, gen):
    B, D = c["batch"], c["width"]
    with nn.context_scope(get_extension_context("hip")):
        x = _variable(_normal(gen, (B, D), 1.0))
        h = F.fixed_point_quantize(x, True, 8, 2 ** -4)
        W = _variable(_normal(gen, (D, D), 0.02))
        indicators = _variable(torch.zeros(D, D, dtype=torch.int32))
        h = F.inq_affine(h, W, indicators, None, 1, 4, (0,), "largest_abs")
        for _ in range(1, c["layers"]):
            h = F.relu(h)
            h = F.fixed_point_quantize(h, True, 8, 2 ** -4)
            h = F.binary_weight_affine(h, _variable(_normal(gen, (D, D), 0.02)), nn.Variable((D, D)),
                                       nn.Variable((D,)))
        # the inputs' first trip to the device
        for v in [x, W] + [node.inputs[1] for node in h._function_order() if len(node.inputs) == 4]:
            v.device_pointer()
        indicators.device_pointer(np.int32)
    return {"y": h, "W": W, "I": indicators}


def _run_mlp(c, s):
    s["y"].forward()
    return [torch.as_tensor(_OnDevice(s["y"]), device="cuda"), torch.as_tensor(_OnDevice(s["W"]), device="cuda"),
            torch.as_tensor(_OnDevice(s["I"], np.int32), device="cuda")]


_PREPARE = {"quantize": _prepare_quantize, "affine": _prepare_affine, "convolution": _prepare_convolution,
            "mlp": _prepare_mlp}
_RUN = {"quantize": _run_quantize, "affine": _run_affine, "convolution": _run_convolution, "mlp": _run_mlp}


def prepare(case, seed):
    kernels.init(0)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    return {"case": case, "hold": _PREPARE[case["kind"]](case, gen)}


def run(state):
    return _RUN[state["case"]["kind"]](state["case"], state["hold"])


def work(case):
    """Every input read once and every output written once; two operations per product and sum."""
    c = case
    if c["kind"] == "quantize":
        n = c["batch"] * c["channels"] * c["height"] * c["width"]
        per = {"fixed": 3, "pow2": 6, "minmax": 9}[c["op"]] + (3 if c["backward"] else 0)
        return {"bytes": 4.0 * n * (4 if c["backward"] else 2), "flops": float(per * n)}
    if c["kind"] == "affine":
        M, K, N = c["rows"], c["inputs"], c["outputs"]
        back = M * N + M * K + K * N if c["backward"] else 0   # dy, dx and dW
        return {"bytes": 4.0 * (M * K + 2 * K * N + M * N + N + back),
                "flops": 2.0 * M * K * N * (3 if c["backward"] else 1)}
    if c["kind"] == "convolution":
        windows = c["batch"] * _out_extent(c, c["height"]) * _out_extent(c, c["width"])
        x = c["batch"] * c["channels"] * c["height"] * c["width"]
        w = c["maps"] * c["channels"] * c["kernel"] ** 2
        weights = 4 * w if c["op"] == "inq" else 2 * w   # weights, indicators and their snapshots / weights and signs
        back = x + w + windows * c["maps"] if c["backward"] else 0
        return {"bytes": 4.0 * (x + weights + windows * c["maps"] + back),
                "flops": 2.0 * windows * w * (3 if c["backward"] else 1)}
    B, D, L = c["batch"], c["width"], c["layers"]
    # the first layer's weights, indicators and snapshots; per further layer the weights and their signs; x and y
    return {"bytes": 4.0 * (4 * D * D + (L - 1) * 2 * D * D + 2 * B * D), "flops": 2.0 * B * D * D * L}


def tolerance(case):
    """Four times what was seen at the listed sizes against the same path in 64 bits, with the sums of 32-bit products
    taken in another order beside it: 1e-6 and 1.4e-6 for the weight gradients (largest element 7.6e-6 of the root mean
    square), 8e-8 for the gradients of a range."""
    if case["kind"] == "quantize":
        return {"rel": 1e-6, "max": 1e-5} if case["ranges"] == "learnt" and case["backward"] else "exact"
    if case["kind"] == "mlp":
        # 2.5e-8 where no activation lies at a tie of the grid; one bit of alpha moves about 2e-6 of the activations
        # of a layer by a step of 1/16, 7e-5 of its norm
        return {"rel": 5e-4}
    return {"rel": 5e-6, "max": 4e-5}
