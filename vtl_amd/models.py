"""`Sequential` builder restricted to what the INT8 path needs: the Python
mirror of nn/models/sequential.v:52-220 for input / linear / relu / forward.

`linear(n)` takes its input width from the previous layer
(nn/models/sequential_info.v:53-60); `forward` loops over the layers
(sequential.v:204-215), here inside one library call: between Linear layers
the activations stay on the device, as per-token int8 codes when the next layer
is a Linear again (as f32 rows for up to 32 rows), and ReLU is folded into the
producing Linear's epilogue, in the spirit of the reference's GPU activation
chain (autograd_cuda/device_session_gpu_d_cuda.v:88-181).
"""
from __future__ import annotations

import numpy as np

from . import capi
from .layers import PER_CHANNEL, HipSession, QuantLinearLayer, forward_host, kaiming_normal
from .storage import HipParams

_RELU = capi.Layer(capi.LAYER_RELU)


class Sequential:
    def __init__(self, mode: str = PER_CHANNEL, seed: int = 0, params: HipParams | None = None):
        self.mode = mode
        self.params = params or HipParams()
        self.rng = np.random.Generator(np.random.Philox(seed))
        self.layers: list = []          # ("input", [k]) | ("linear", layer) | ("relu",)
        self._width: int | None = None
        self.session = HipSession(self.params)

    def input(self, shape) -> "Sequential":
        if len(shape) != 1:
            raise ValueError("only flat inputs reach a Linear layer")
        self._width = int(shape[0])
        self.layers.append(("input", list(shape)))
        return self

    def linear(self, output_size: int, weights: np.ndarray | None = None,
               bias: np.ndarray | None = None) -> "Sequential":
        if self._width is None:
            raise ValueError("Sequential.linear: add an input layer first")
        if weights is None:
            weights = kaiming_normal([output_size, self._width], self.rng)
        weights = np.asarray(weights, np.float32)
        if list(weights.shape) != [output_size, self._width]:
            raise ValueError(f"weights {list(weights.shape)}, expected {[output_size, self._width]}")
        self.layers.append(("linear", QuantLinearLayer(weights, bias, self.mode, self.params)))
        self._width = output_size
        return self

    def relu(self) -> "Sequential":
        self.layers.append(("relu",))
        return self

    def forward(self, x: np.ndarray, no_grad: bool = False) -> np.ndarray:
        """`no_grad` is the Context's flag (autograd/context.v:19-21): under it the layers'
        quantized weights are kept from one forward to the next, otherwise every trainable
        layer uploads and quantizes its parameters again (QuantLinearLayer.quantized)."""
        x = np.asarray(x, np.float32)
        if x.ndim != 2:
            raise ValueError("Matrix expected")
        capi.call("vtl_hip_set_device", self.params.device_id)
        stack, width, codes = [], x.shape[1], {}
        for layer in self.layers:
            if layer[0] == "linear":
                qw = codes.get(layer[1])    # a layer that stands in the stack twice is quantized once
                if qw is None:
                    qw = codes[layer[1]] = layer[1].enqueue_quantized(no_grad)
                stack.append(qw.layer)
                width = qw.out_features
            elif layer[0] == "relu":
                stack.append(_RELU)
        y = forward_host(x, stack, len(stack), width)
        for qw in codes.values():
            qw.known_complete()
        return y

    def release(self) -> None:
        for l in self.layers:
            if l[0] == "linear":
                l[1].release()
        self.session.release()
