"""Timed cases of the quantized-linear path and of the full-precision Linear beside it.

Two kinds of program use this package.  One keeps its tensors on the host, as VTL does, and
goes through the layers (`Sequential.forward`, `QuantLinearLayer.forward`, the hooks of the
Linear gate's backward, `la.matmul`): numpy in, numpy out.  The other keeps its tensors on
the device (`HipTensor`) and calls the operations on them.  Both are covered: inference and
training, one token and many, int8, f32 and f64, whole and ragged sizes.
"""
from __future__ import annotations

import math
import os

import numpy as np
import torch

from vtl_amd import (PER_CHANNEL, PER_TENSOR, HipSession, HipTensor, QuantLinearLayer, Sequential, capi,
                     linear_backward_hip, linear_backward_hip_f32, linear_hip, linear_i8_hip, matmul_hip_host)


def listed():
    return [
        # The first layer of the MNIST multilayer perceptron at its usual batch, quantized per
        # tensor, weights frozen: the smallest call a program makes, host to host.
        {"name": "mnist_linear_infer", "op": "layer", "m": 64, "n": 256, "k": 784, "mode": PER_TENSOR, "frozen": True},
        # Inference of a three-layer perceptron through Sequential.forward: a batch, and one request.
        {"name": "mlp_infer_256", "op": "mlp", "m": 256, "dims": "4096,11008,4096,1024"},
        {"name": "mlp_infer_1", "op": "mlp", "m": 1, "dims": "4096,11008,4096,1024"},
        # A training step's forward through one large layer: parameters may have changed, so
        # they are uploaded and quantized again.
        {"name": "linear_train_forward", "op": "layer", "m": 256, "n": 11008, "k": 4096, "mode": PER_CHANNEL,
         "frozen": False},
        # Quantize a large tensor per row and bring it back; a ragged one with one scale.
        {"name": "quant_rows_16384", "op": "quant", "m": 16384, "k": 16384, "axis": 0},
        {"name": "quant_tensor_ragged", "op": "quant", "m": 3001, "k": 4099, "axis": -1},
        # The int8 product on codes that are there already.
        {"name": "linear_i8_4096", "op": "linear_i8", "m": 4096, "n": 4096, "k": 4096, "relu": False},
        # One layer of a decoder: a few tokens, and a short prompt.
        {"name": "decode_8", "op": "dynquant", "m": 8, "n": 14336, "k": 4096, "relu": False},
        {"name": "prefill_128", "op": "dynquant", "m": 128, "n": 14336, "k": 4096, "relu": False},
        # Full precision, forward and backward on the device: a large layer.
        {"name": "linear_step_f32", "op": "step", "m": 256, "n": 11008, "k": 4096, "dtype": "float32"},
        # The Linear gate's backward through the host hook at the MNIST size, and la.matmul at the
        # size of the reference's own benchmark (benchmarks/vs_numpy/matmul_bench.v:13,24-47).
        {"name": "mnist_backward_host", "op": "backward", "m": 64, "n": 256, "k": 784, "dtype": "float32"},
        {"name": "matmul_f64_512", "op": "matmul", "m": 512, "n": 512, "k": 512, "dtype": "float64"},
    ]


def _size(rng, lo: int, hi: int) -> int:
    """A size between lo and hi, even over its logarithm; half of them as they come (odd ones
    among them), half a multiple of 64 where the range allows one."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5 and hi >= 64:
        v = (v + 32) // 64 * 64
    return min(hi, max(lo, v))


def draw(rng):
    op = rng.choice(["layer", "layer", "mlp", "mlp", "quant", "quant", "linear_i8", "dynquant", "dynquant", "step",
                     "backward", "matmul"])
    if op == "layer":
        return {"op": op, "m": _size(rng, 1, 256), "n": _size(rng, 64, 11008), "k": _size(rng, 64, 4096),
                "mode": rng.choice([PER_TENSOR, PER_CHANNEL]), "frozen": rng.random() < 0.5}
    if op == "mlp":
        dims = [_size(rng, 256, 4096), _size(rng, 256, 11008), _size(rng, 256, 4096), _size(rng, 16, 1024)]
        return {"op": op, "m": _size(rng, 1, 256), "dims": ",".join(map(str, dims))}
    if op == "quant":
        return {"op": op, "m": _size(rng, 16, 16384), "k": _size(rng, 16, 16384), "axis": rng.choice([-1, 0])}
    if op == "linear_i8":
        return {"op": op, "m": _size(rng, 1, 4096), "n": _size(rng, 64, 4096), "k": _size(rng, 64, 4096),
                "relu": rng.random() < 0.5}
    if op == "dynquant":
        return {"op": op, "m": _size(rng, 1, 256), "n": _size(rng, 256, 14336), "k": _size(rng, 256, 4096),
                "relu": rng.random() < 0.5}
    dtype = rng.choice(["float32", "float64"])
    if op == "step":
        return {"op": op, "m": _size(rng, 16, 256), "n": _size(rng, 64, 11008), "k": _size(rng, 64, 4096), "dtype": dtype}
    if op == "backward":
        return {"op": op, "m": _size(rng, 16, 256), "n": _size(rng, 16, 2048), "k": _size(rng, 16, 2048), "dtype": dtype}
    return {"op": op, "m": _size(rng, 32, 1024), "n": _size(rng, 32, 1024), "k": _size(rng, 32, 1024), "dtype": dtype}


# -- inputs ---------------------------------------------------------------------------

def _normal(gen, *shape, std=1.0, dtype="float32"):
    return torch.randn(*shape, generator=gen, device="cuda", dtype=getattr(torch, dtype)) * std


def _uniform(gen, *shape, lo=0.0, hi=1.0):
    return torch.rand(*shape, generator=gen, device="cuda") * (hi - lo) + lo


def _host(t) -> np.ndarray:
    return t.cpu().numpy()


def _device(t) -> HipTensor:
    """A HipTensor of its own with the values of a torch tensor."""
    t = t.contiguous()
    h = HipTensor.empty(list(t.shape), np.dtype(str(t.dtype).removeprefix("torch.")))
    torch.cuda.synchronize()
    capi.call("vtl_hip_memcpy_d2d", h.ptr, t.data_ptr(), t.numel() * t.element_size())
    capi.call("vtl_hip_sync")
    return h


class _Shared:
    """The memory of a HipTensor as torch sees it, for as long as the torch tensor lives."""

    def __init__(self, t: HipTensor):
        self.owner = t
        self.__cuda_array_interface__ = {"shape": tuple(t.shape), "typestr": t.dtype.str, "data": (t.ptr, False),
                                         "version": 2}


def _view(t: HipTensor) -> torch.Tensor:
    return torch.as_tensor(_Shared(t), device="cuda")


def _outlier_rows(gen, rows, cols):
    """~N(0, 1) with one element in a thousand multiplied by 20."""
    x = _normal(gen, rows, cols)
    step = max(1, (1 << 26) // cols)
    for r in range(0, rows, step):
        part = x[r:r + step]
        part[torch.rand(part.shape, generator=gen, device="cuda") < 0.001] *= 20.0
    return x


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    op = case["op"]
    s = {"op": op, **{k: case[k] for k in ("relu", "axis", "frozen") if k in case}}
    if op == "layer":
        m, n, k = case["m"], case["n"], case["k"]
        s["x"] = _host(_uniform(gen, m, k))
        s["layer"] = QuantLinearLayer(_host(_normal(gen, n, k, std=(2.0 / k) ** 0.5)), _host(_normal(gen, 1, n, std=0.02)),
                                      mode=case["mode"], requires_grad=not case["frozen"])
        if case["frozen"]:
            s["layer"].quantized()
    elif op == "mlp":
        dims = [int(d) for d in case["dims"].split(",")]
        net = Sequential().input([dims[0]])
        for i in range(1, len(dims)):
            net.linear(dims[i], weights=_host(_normal(gen, dims[i], dims[i - 1], std=(2.0 / dims[i - 1]) ** 0.5)))
            if i + 1 < len(dims):
                net.relu()
        s["x"], s["net"] = _host(_normal(gen, case["m"], dims[0])), net
    elif op == "quant":
        s["x"] = _device(_outlier_rows(gen, case["m"], case["k"]))
    elif op == "linear_i8":
        m, n, k = case["m"], case["n"], case["k"]
        codes = lambda r: _device(torch.randint(-127, 128, (r, k), generator=gen, device="cuda", dtype=torch.int8))  # noqa: E731
        s["a"], s["w"] = codes(m), codes(n)
        s["sa"] = _device(_uniform(gen, m, lo=0.5 / 127, hi=1.5 / 127))
        s["sw"] = _device(_uniform(gen, n, lo=0.5 / 127, hi=1.5 / 127))
        s["bias"] = _device(_normal(gen, n, std=0.02))
    elif op == "dynquant":
        m, n, k = case["m"], case["n"], case["k"]
        s["layer"] = QuantLinearLayer(_host(_normal(gen, n, k, std=0.02)), requires_grad=False)
        s["layer"].quantized()
        s["x"], s["session"] = _device(_normal(gen, m, k)), HipSession()
    elif op == "step":
        m, n, k, t = case["m"], case["n"], case["k"], case["dtype"]
        s["x"], s["w"] = _device(_normal(gen, m, k, dtype=t)), _device(_normal(gen, n, k, std=k ** -0.5, dtype=t))
        s["bias"], s["grad"] = _device(_normal(gen, n, std=0.02, dtype=t)), _device(_normal(gen, m, n, dtype=t))
    elif op == "backward":
        m, n, k, t = case["m"], case["n"], case["k"], case["dtype"]
        os.environ["VTL_USE_HIP"] = os.environ["VTL_HIP_BACKWARD"] = "1"    # the hook's opt-in
        s["x"], s["w"] = _host(_normal(gen, m, k, dtype=t)), _host(_normal(gen, n, k, std=k ** -0.5, dtype=t))
        s["grad"] = _host(_normal(gen, m, n, dtype=t))
    else:
        m, n, k, t = case["m"], case["n"], case["k"], case["dtype"]
        s["a"], s["b"] = _host(_normal(gen, m, k, dtype=t)), _host(_normal(gen, k, n, dtype=t))
    return s


def run(s):
    op = s["op"]
    if op == "layer":
        return s["layer"].forward(s["x"])
    if op == "mlp":
        return s["net"].forward(s["x"], no_grad=True)
    if op == "quant":
        q, scales = s["x"].quantize_i8(s["axis"])
        back = q.dequantize(scales, s["axis"])
        return _view(q), _view(scales), _view(back)
    if op == "linear_i8":
        return _view(linear_i8_hip(s["a"], s["sa"], s["w"], s["sw"], s["bias"], relu=s["relu"]))
    if op == "dynquant":
        return _view(s["layer"].forward_device(s["x"], relu=s["relu"], session=s["session"]))
    if op == "step":
        y = linear_hip(s["x"], s["w"], s["bias"])
        return [_view(y)] + [_view(g) for g in linear_backward_hip(s["grad"], s["x"], s["w"])]
    if op == "backward":
        return linear_backward_hip_f32(s["grad"], s["x"], s["w"], True)
    return matmul_hip_host(s["a"], s["b"])


def work(case):
    op, m, k = case["op"], case["m"], case.get("k")
    if op == "quant":
        scales = 4 * (m if case["axis"] == 0 else 1)
        return {"bytes": 4 * m * k + m * k + 2 * scales + m * k + 4 * m * k, "flops": 3 * m * k}
    if op == "mlp":
        d = [int(v) for v in case["dims"].split(",")]
        weights = sum(d[i] * d[i + 1] + 8 * d[i + 1] for i in range(len(d) - 1))
        return {"bytes": 4 * m * (d[0] + d[-1]) + weights,
                "flops": 2 * m * sum(d[i] * d[i + 1] for i in range(len(d) - 1))}
    n = case["n"]
    if op == "layer":
        return {"bytes": 4 * m * k + 4 * m * n + (1 if case["frozen"] else 4) * n * k + 4 * n, "flops": 2 * m * n * k}
    if op == "linear_i8":
        return {"bytes": m * k + n * k + 4 * m * n + 4 * (m + 2 * n), "flops": 2 * m * n * k}
    if op == "dynquant":
        return {"bytes": 4 * m * k + n * k + 4 * m * n + 8 * n, "flops": 2 * m * n * k}
    e = 4 if case["dtype"] == "float32" else 8
    if op == "step":
        return {"bytes": e * (2 * m * k + 2 * n * k + 2 * m * n + 2 * n), "flops": 6 * m * n * k}
    if op == "backward":
        return {"bytes": e * (2 * m * k + 2 * n * k + m * n + n), "flops": 4 * m * n * k}
    return {"bytes": e * (m * k + k * n + m * n), "flops": 2 * m * n * k}


def tolerance(case):
    if case.get("dtype") == "float64":
        return {"rel": 1e-13, "max": 1e-11}     # f64 sums in another order
    if case.get("dtype") == "float32":
        return {"rel": 1e-6, "max": 1e-5}       # f64 sums rounded to f32 once
    # Codes and int32 sums are whole numbers with one right value; what follows is a few f32
    # operations in a stated order.
    return {"rel": 1e-6, "max": 1e-5, "differ": 0.0}
