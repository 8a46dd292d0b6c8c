"""Linear layer on the INT8 HIP path: the Python mirror of the V files
`nn/layers/hip_config.v`, `linear_hip_hooks_d_hip.v` and `linear_hip_d_hip.v`.

The reference's f32 Linear is `y = x.W^T + b` with W stored
`[out_features, in_features]` and bias `[1, out_features]`
(nn/layers/linear.v:10-33); its backend hook is
`linear_forward_f32` (nn/layers/linear_forward_f32.v:7-14), which asks
`linear_forward_f32_use_<backend>()` and tries the device path.  This module
adds the HIP branch of that hook.  The device path returns host tensors, like
every GPU path of the reference (docs/DEVICE_MEMORY.md:9-16), unless the
caller chains layers on the device explicitly (`forward_device`).

There is no CPU arithmetic in here: a failing device call raises
`capi.VtlHipError`.  (In V the hook site keeps the reference's own
`or { return linear_forward_f32_cpu(...) }`, which is VTL's code, not this
library's.)
"""
from __future__ import annotations

import ctypes as C
import os

import numpy as np

from . import capi
from .storage import HipParams, HipStorage, host_array
from .tensor import (HipTensor, _dynquant_workspace, linear_backward_hip, linear_f32_dynquant_hip, linear_hip, linear_i8_hip,
                     matmul_hip)


# -- nn/layers/hip_config.v (cf. vulkan_config.v:12-24, cuda_config.v:11-23) ----

def hip_linear_enabled() -> bool:
    """True when the user opts in with VTL_USE_HIP=1 (and the build has `-d hip`)."""
    return os.environ.get("VTL_USE_HIP") == "1"


def hip_tests_enabled() -> bool:
    """Gate for device tests, VTL_TEST_HIP=1 (cf. vulkan_tests_enabled)."""
    return os.environ.get("VTL_TEST_HIP") == "1"


def linear_forward_f32_use_hip() -> bool:
    """Hook consulted by linear_forward_f32 (cf. linear_vulkan_hooks_d_vulkan.v:9)."""
    return hip_linear_enabled()


# -- quantization granularity ------------------------------------------------------

PER_TENSOR = "per_tensor"      # one scale for x, one for W
PER_CHANNEL = "per_channel"    # one scale per row of x (token) and per row of W (output channel)


def hip_backward_enabled() -> bool:
    """Linear gate gradients on the device: VTL_USE_HIP=1 and VTL_HIP_BACKWARD=1
    (cf. cuda_backward_enabled, autograd_cuda/gpu_config.v:20-23)."""
    return os.environ.get("VTL_USE_HIP") == "1" and os.environ.get("VTL_HIP_BACKWARD") == "1"


def linear_gate_use_hip_backward() -> bool:
    """Hook asked by LinearGate.backward (cf. linear_gate_use_vulkan_backward,
    nn/gates/layers/linear_gate_vulkan_hooks_d_vulkan.v:6-8)."""
    return hip_backward_enabled() and capi.device_count() > 0


class HipSession:
    """Reusable device buffers for one Context, cf. DeviceSession
    (autograd_cuda/device_session.v:13-24) and GpuDevBuf.ensure
    (autograd_cuda/device_session_gpu_d_cuda.v:24-39): a buffer grows when a
    larger request arrives and is otherwise reused."""

    def __init__(self, params: HipParams | None = None):
        self.params = params or HipParams()
        self._bufs: dict[str, HipStorage] = {}

    def ensure(self, name: str, nbytes: int) -> HipStorage:
        cur = self._bufs.get(name)
        if cur is not None and cur.size >= nbytes:
            return cur
        if cur is not None:
            cur.release()
        buf = HipStorage.empty(max(int(nbytes), 256), np.uint8, self.params)
        self._bufs[name] = buf
        return buf

    def release(self) -> None:
        for b in self._bufs.values():
            b.release()
        self._bufs.clear()


def content_fingerprint(t: np.ndarray) -> int:
    """Cheap fingerprint of a parameter tensor's contents: FNV-1a over the bit patterns of
    up to 64 elements at even strides plus the last one, and the element count.  It is
    the second line of defence of the weight cache (the first is the frozen rule of
    QuantLinearLayer.quantized): an in-place edit of a frozen parameter - a checkpoint
    loaded into the same tensor, a manual `set` - changes it with near certainty when
    the edit touches most elements, as every optimizer step and every load does."""
    flat = np.ascontiguousarray(t, None if t.dtype.itemsize in (4, 8) else np.float64)
    h = C.c_uint64()
    capi.call("vtl_hip_content_fingerprint", flat.ctypes.data, flat.size, flat.itemsize, C.byref(h))
    return h.value


# Weights of up to so many bytes, which one host thread makes codes of, and from so many on, which several do, go to the call that quantizes
# them on their way to the device and takes the bias along.  (us of a forward, uploaded and then quantized, and so: 16 x 256 x 256 46 and 42,
# 64 x 512 x 512 80 and 63, 64 x 600 x 1024 118 and 82.  Codes are ahead in between too, 64 x 400 x 1024 100 and 78, but those sizes still
# take the upload.)
_QUANTIZED_UP_TO, _QUANTIZED_FROM = 1 << 20, 2 << 20


class QuantizedWeights:
    """Device-resident int8 weights of one Linear layer, derived from the f32
    parameter.  `source` / `bias_source` are the host tensors the device copies
    were made from, `fingerprint` / `bias_fingerprint` their content fingerprints at
    that moment and `frozen` whether the parameters were frozen then (see
    QuantLinearLayer.quantized for the rule that decides re-use).

    Codes whose row length is no multiple of 16 lie on the device twice where there are 2**18 of them or
    more: dense (`w_q`), and in padded rows (`w_rows`).

    The device copies are complete on return, for work on any stream.  With `wait` False they
    are on their way, in order for the library's next calls; wait() makes up for it."""

    def __init__(self, weights: np.ndarray, bias: np.ndarray | None, mode: str,
                 params: HipParams | None = None, frozen: bool = False, wait: bool = True):
        if weights.ndim != 2:
            raise ValueError("Matrix expected")
        if mode not in (PER_TENSOR, PER_CHANNEL):
            raise ValueError(f"unknown quantization mode {mode!r}")
        self.mode = mode
        self.source = weights
        self.bias_source = bias
        self.frozen = frozen
        # What says whether the parameters are as they were: their addresses (both tensors are
        # held, so they stay), sizes and fingerprints.
        parts = [t for t in (weights, bias) if t is not None]
        self._watchable = all(type(t) is np.ndarray and t.flags.c_contiguous and t.itemsize in (4, 8) for t in parts)
        self.fingerprint = content_fingerprint(weights)
        self.bias_fingerprint = None if bias is None else content_fingerprint(np.asarray(bias))
        if self._watchable:
            self._watch = (capi.Watch * len(parts))(*[
                capi.Watch(t.ctypes.data, t.size, t.itemsize, h)
                for t, h in zip(parts, (self.fingerprint, self.bias_fingerprint))])
        self.out_features, self.in_features = weights.shape
        w = np.asarray(weights, np.float32)
        b = None if bias is None else np.asarray(bias, np.float32).reshape(-1)
        if b is not None and b.size != self.out_features:
            raise ValueError(f"bias has {b.size} entries, expected {self.out_features}")
        # enqueued, without a wait: only the library's next calls use them
        w = np.ascontiguousarray(w)
        self.bias, extra = None, (None, None, 0)
        if b is not None:
            b = np.ascontiguousarray(b)
            self.bias = HipTensor.empty(b.shape, np.float32, params)
            extra = (self.bias.ptr, b.ctypes.data, b.nbytes)
        if 0 < w.nbytes <= _QUANTIZED_UP_TO or w.nbytes >= _QUANTIZED_FROM:
            per_row = mode == PER_CHANNEL
            self.w_q = HipTensor.empty(w.shape, np.int8, params)
            self.sw = HipTensor.empty([self.out_features if per_row else 1], np.float32, params)
            capi.call("vtl_hip_upload_quantized", w.ctypes.data, self.out_features, self.in_features, int(per_row), self.w_q.ptr,
                      self.sw.ptr, *extra)
        else:
            w_dev = HipTensor.empty(w.shape, np.float32, params)
            try:
                capi.call("vtl_hip_upload_two", w_dev.ptr, w.ctypes.data, w.nbytes, *extra)
                self.w_q, self.sw = w_dev.quantize_i8(0 if mode == PER_CHANNEL else -1)
            finally:
                w_dev.release()
        # Rows of codes that the fast kernels do not take as they are get a padded copy, made with
        # the codes instead of by every forward (8 tokens x 14336 x 4095: 39.7 -> 18.6 us).  Small ones don't: kernels
        # that take rows of any length are as fast there.
        self.w_rows, row_bytes = None, 0
        if self.in_features % 16 and self.w_q.size >= 1 << 18:
            row_bytes = capi.lib().vtl_hip_padded_row(self.in_features)
            self.w_rows = HipTensor.empty([self.out_features, row_bytes], np.int8, params)
            capi.call("vtl_hip_pad_rows_i8", self.w_q.ptr, self.out_features, self.in_features, self.w_rows.ptr)
        self.layer = capi.Layer(capi.LAYER_LINEAR, mode == PER_CHANNEL, self.out_features, self.in_features,
                                (self.w_q if self.w_rows is None else self.w_rows).ptr, self.sw.ptr,
                                self.bias.ptr if self.bias is not None else None, row_bytes)
        self._complete = False
        if wait:
            self.wait()

    def wait(self) -> None:
        """Returns when the device copies are complete."""
        if not self._complete:
            capi.call("vtl_hip_sync")
            self._complete = True

    def known_complete(self) -> None:
        """Says that something has been waited for that was enqueued after the device copies."""
        self._complete = True

    def unchanged(self) -> bool:
        """Whether the parameters still have the contents that the codes were made from."""
        if self._watchable:
            return capi.lib().vtl_hip_contents_unchanged(len(self._watch), self._watch) == 1
        return (self.fingerprint == content_fingerprint(self.source) and
                (self.bias_source is None or self.bias_fingerprint == content_fingerprint(np.asarray(self.bias_source))))

    def release(self) -> None:
        self.w_q.release()
        self.sw.release()
        for t in (self.bias, self.w_rows):
            if t is not None:
                t.release()


def linear_forward_hip_i8_device(x: HipTensor, qw: QuantizedWeights, relu: bool = False,
                                 session: HipSession | None = None) -> HipTensor:
    """x[M,K] f32 on the device -> y[M,N] f32 on the device."""
    if len(x.shape) != 2:
        raise ValueError("Matrix expected")
    if x.shape[1] != qw.in_features:
        raise ValueError(
            f"Invalid shapes for matrix multiplication {x.shape} and {[qw.in_features, qw.out_features]}")
    if qw.mode == PER_CHANNEL:
        ws = None
        if session is not None:
            ws = session.ensure("dynquant", _dynquant_workspace(*x.shape))
        if qw.w_rows is not None:
            x._assert(np.float32, what="linear input")
            own = HipStorage.empty(_dynquant_workspace(*x.shape), np.uint8, x.data.params) if ws is None else None
            y = HipTensor.empty([x.shape[0], qw.out_features], np.float32, x.data.params)
            try:
                use = own or ws
                capi.call("vtl_hip_layer_f32", C.byref(qw.layer), x.ptr, y.ptr, x.shape[0], int(relu), use.ptr, use.size)
            finally:
                if own is not None:
                    own.release()
            return y
        return linear_f32_dynquant_hip(x, qw.w_q, qw.sw, qw.bias, relu=relu, workspace=ws)
    x_q, sx = x.quantize_i8(-1)
    try:
        return linear_i8_hip(x_q, sx, qw.w_q, qw.sw, qw.bias, relu=relu)
    finally:
        x_q.release()
        sx.release()


def linear_forward_hip_f32(x: np.ndarray, weights: np.ndarray, bias: np.ndarray | None,
                           mode: str = PER_CHANNEL) -> np.ndarray:
    """`linear_forward_hip_f32(x, weights, bias) !&vtl.Tensor[f32]`: the HIP entry
    of the f32 hook (cf. linear_forward_vulkan_f32, linear_vulkan_d_vulkan.v:7-12).
    Uploads, quantizes both operands, runs the int8 linear, returns a host tensor."""
    if not hip_linear_enabled():
        raise RuntimeError("linear_forward_hip_f32: set VTL_USE_HIP=1 to enable")
    return _linear_host_roundtrip(x, weights, bias, mode)


def _linear_host_roundtrip(x, weights, bias, mode) -> np.ndarray:
    x = np.asarray(x, np.float32)
    if x.ndim != 2 or np.ndim(weights) != 2:
        raise ValueError("Matrix expected")
    qw = QuantizedWeights(weights, bias, mode, wait=False)
    try:
        return forward_host(x, [qw.layer], 1, qw.out_features)
    finally:
        qw.release()


def forward_host(x: np.ndarray, layers, count: int, out_features: int) -> np.ndarray:
    """x[M, K] through `count` layers (`capi.Layer`) whose parameters are on the current device, host
    to host in one call."""
    x = np.ascontiguousarray(x)
    rows, cols = x.shape
    first = next((l for l in layers if l.kind == capi.LAYER_LINEAR), None)
    if first is not None and cols != first.in_features:
        raise ValueError(
            f"Invalid shapes for matrix multiplication {[rows, cols]} and {[first.in_features, first.out_features]}")
    y, host = host_array(rows * out_features, x.dtype)
    if type(layers) is list:
        layers = (capi.Layer * count)(*layers)
    capi.call("vtl_hip_forward_i8_host", x.ctypes.data, rows, cols, layers, count, host)
    return y.reshape(rows, out_features)


class QuantLinearLayer:
    """`LinearLayer[f32]` (nn/layers/linear.v:17-74) whose forward runs on the
    INT8 HIP path.  Parameters stay on the host as f32 (as in the reference);
    the int8 copy on the device is derived state.

    `requires_grad` mirrors the flag of the layer's weight Variable
    (autograd/variable.v:64, default true): while it is set an optimizer may
    change the parameters between any two forwards, and most of the reference's
    optimizers do so IN PLACE (SGD: nn/optimizers/sgd.v:46-53 ->
    nn/internal/optimizers.v:6-12 `value.set`; likewise adagrad.v:60, adamw.v:95,
    rmsprop.v:81), only Adam assigns a new tensor (adam.v:115,136).  So the
    tensor's identity says nothing about its contents, and a trainable layer
    uploads and quantizes its parameters on every forward, as the reference's
    own device chain uploads them on every forward
    (autograd_cuda/device_session_gpu_d_cuda.v:107).  The codes are kept from
    one forward to the next only for frozen parameters (requires_grad false, or
    a forward under no_grad)."""

    def __init__(self, weights: np.ndarray, bias: np.ndarray | None = None, mode: str = PER_CHANNEL,
                 params: HipParams | None = None, requires_grad: bool = True):
        weights = np.asarray(weights, np.float32)
        if weights.ndim != 2:
            raise ValueError("Matrix expected")
        self.weights = weights                                   # [out, in]
        self.bias = (np.zeros((1, weights.shape[0]), np.float32) if bias is None
                     else np.asarray(bias, np.float32).reshape(1, -1))  # [1, out]
        self.mode = mode
        self.params = params or HipParams()
        self.requires_grad = requires_grad
        self.quantize_count = 0      # how often the parameters were uploaded and quantized (tests)
        self._cache: QuantizedWeights | None = None

    def output_shape(self):
        return [self.weights.shape[0]]

    def variables(self):
        return [self.weights, self.bias]

    def invalidate(self) -> None:
        """Drops the device copy: the next forward uploads and quantizes again.  For
        callers that edit a frozen parameter in place."""
        if self._cache is not None:
            self._cache.release()
            self._cache = None

    def quantized(self, no_grad: bool = False) -> QuantizedWeights:
        """The layer's int8 weights for one forward.  Re-used from the previous forward only
        when ALL of these hold: the parameters are frozen now (`requires_grad` false, or this
        forward runs under `no_grad`) and were frozen when the copy was made, `weights` and
        `bias` are still the same tensor objects, and their content fingerprints have not
        changed.  Otherwise the parameters are uploaded and quantized again."""
        qw = self.enqueue_quantized(no_grad)
        qw.wait()
        return qw

    def enqueue_quantized(self, no_grad: bool = False) -> QuantizedWeights:
        """quantized() without its wait, for a call whose own end is waited for (known_complete)."""
        frozen = no_grad or not self.requires_grad
        c = self._cache
        fresh = (c is not None and frozen and c.frozen and c.source is self.weights
                 and c.bias_source is self.bias and c.unchanged())
        if not fresh:
            if c is not None:
                c.release()
            self._cache = QuantizedWeights(self.weights, self.bias, self.mode, self.params, frozen=frozen,
                                           wait=False)
            self.quantize_count += 1
        return self._cache

    def forward_device(self, x: HipTensor, relu: bool = False,
                       session: HipSession | None = None, no_grad: bool = False) -> HipTensor:
        return linear_forward_hip_i8_device(x, self.quantized(no_grad), relu=relu, session=session)

    def forward(self, x: np.ndarray, no_grad: bool = False) -> np.ndarray:
        x = np.asarray(x, np.float32)
        if x.ndim != 2:
            raise ValueError("Matrix expected")
        capi.call("vtl_hip_set_device", self.params.device_id)
        qw = self.enqueue_quantized(no_grad)
        y = forward_host(x, [qw.layer], 1, qw.out_features)
        qw.known_complete()
        return y

    def release(self) -> None:
        if self._cache is not None:
            self._cache.release()
            self._cache = None


def kaiming_normal(shape, rng: np.random.Generator) -> np.ndarray:
    """Weight initialiser of linear_layer (nn/layers/linear.v:25, nn/internal/init.v:21-70):
    N(0, sqrt(2 / fan_in)) where compute_fans multiplies both fans by shape[1]."""
    f0 = shape[0] * int(np.prod(shape[1:]))
    std = np.sqrt(2.0 / f0)
    return (rng.standard_normal(shape) * std).astype(np.float32)


# -- la.matmul / Linear forward and backward in full precision -----------------

def _as_float_matrix(t, what: str) -> np.ndarray:
    a = np.asarray(t)
    if a.dtype not in (np.float32, np.float64):
        raise TypeError(f"{what}: f32 or f64 tensor expected, got {a.dtype}")
    if a.ndim != 2:
        raise ValueError("Matrix expected")
    return a


def matmul_hip_host(a: np.ndarray, b: np.ndarray) -> np.ndarray:
    """`la.matmul[T](a, b)` (la/la.v:38-55) through the device: upload both
    operands, f64-accumulating matmul, download.  Shape errors carry the
    reference's message."""
    a = _as_float_matrix(a, "matmul")
    b = _as_float_matrix(b, "matmul")
    if a.shape[1] != b.shape[0]:
        raise ValueError(f"Invalid shapes for matrix multiplication {list(a.shape)} and {list(b.shape)}")
    a = np.ascontiguousarray(a)
    b = np.ascontiguousarray(b, a.dtype)
    m, k = a.shape
    n = b.shape[1]
    capi.call("vtl_hip_set_device", 0)
    c, host = host_array(m * n, a.dtype)
    capi.call("vtl_hip_matmul_host_f32" if a.itemsize == 4 else "vtl_hip_matmul_host_f64", a.ctypes.data, b.ctypes.data,
              host, m, n, k)
    return c.reshape(m, n)


def linear_forward_hip_exact(x: np.ndarray, weights: np.ndarray, bias: np.ndarray | None) -> np.ndarray:
    """The unquantized Linear forward on the device with the arithmetic of
    linear_forward_f32_cpu (nn/layers/linear_forward_f32.v:16-18): matmul(x, W^T)
    through f64, then the bias added in the tensor's type."""
    x = _as_float_matrix(x, "linear")
    w = _as_float_matrix(weights, "linear").astype(x.dtype, copy=False)
    x_dev, w_dev = HipTensor.from_host(x), HipTensor.from_host(w)
    b_dev = None if bias is None else HipTensor.from_host(np.asarray(bias, x.dtype).reshape(1, -1))
    try:
        y_dev = linear_hip(x_dev, w_dev, b_dev)
        try:
            return y_dev.cpu()
        finally:
            y_dev.release()
    finally:
        for t in (x_dev, w_dev, b_dev):
            if t is not None:
                t.release()


def linear_backward_hip_f32(grad: np.ndarray, input: np.ndarray, weight: np.ndarray,
                            bias_needs_grad: bool):
    """`linear_backward_hip_f32(grad, input, weight, bias_needs_grad) ![]&vtl.Tensor[f32]`:
    [d_input, d_weight, d_bias] of a Linear layer, the HIP counterpart of
    linear_backward_vulkan_f32 (nn/internal/linear_vulkan_backward_d_vulkan.v:9-38)
    and linear_backward_f64 (autograd_cuda/linear_backward_cuda_d_cuda.v:9-36).
    d_bias is [1, out_features]: the column sums of grad, or zeros when the bias
    needs no gradient.  Works for f32 and f64 host tensors alike."""
    if not hip_backward_enabled():
        raise RuntimeError("linear_backward_hip_f32: set VTL_USE_HIP=1 and VTL_HIP_BACKWARD=1")
    g = _as_float_matrix(grad, "linear backward")
    x = _as_float_matrix(input, "linear backward").astype(g.dtype, copy=False)
    w = _as_float_matrix(weight, "linear backward").astype(g.dtype, copy=False)
    m, n = g.shape
    k = x.shape[1]
    if x.shape != (m, k) or w.shape != (n, k):
        raise ValueError(f"linear_backward_hip: grad {list(g.shape)}, input {list(x.shape)}, weight {list(w.shape)}")
    g, x, w = np.ascontiguousarray(g), np.ascontiguousarray(x), np.ascontiguousarray(w)
    capi.call("vtl_hip_set_device", 0)
    (dx, dx_ptr), (dw, dw_ptr) = host_array(m * k, g.dtype), host_array(n * k, g.dtype)
    db, db_ptr = host_array(n, g.dtype) if bias_needs_grad else (np.zeros(n, g.dtype), None)
    capi.call("vtl_hip_linear_backward_host_f32" if g.itemsize == 4 else "vtl_hip_linear_backward_host_f64",
              g.ctypes.data, x.ctypes.data, w.ctypes.data, dx_ptr, dw_ptr, db_ptr, m, n, k)
    return [dx.reshape(m, k), dw.reshape(n, k), db.reshape(1, n)]


# -- activation hooks (cf. relu_forward_f32 / sigmoid_forward_f32,
#    nn/layers/activation_forward_f32.v:7-24, and their Vulkan bodies
#    nn/layers/activation_vulkan_d_vulkan.v:16-29) ---------------------------------

def _activation_host_roundtrip(x, op: str) -> np.ndarray:
    a = np.asarray(x)
    if a.dtype not in (np.float32, np.float64):
        raise TypeError(f"{op}: f32 or f64 tensor expected, got {a.dtype}")
    if a.size == 0:
        return a.copy()
    t = HipTensor.from_host(a)
    try:
        if op == "relu":
            return t.relu_().cpu()
        out = t.sigmoid_hip()
        try:
            return out.cpu()
        finally:
            out.release()
    finally:
        t.release()


def relu_forward_hip_f32(x: np.ndarray) -> np.ndarray:
    """`relu_forward_hip_f32(x) !&vtl.Tensor[f32]`: ReLU through the device (x < 0 -> 0,
    nn/internal/activation.v:63-70); the HIP body of relu_forward_f32's device branch."""
    if not hip_linear_enabled():
        raise RuntimeError("relu_forward_hip_f32: set VTL_USE_HIP=1 to enable")
    return _activation_host_roundtrip(x, "relu")


def sigmoid_forward_hip_f32(x: np.ndarray) -> np.ndarray:
    """`sigmoid_forward_hip_f32(x) !&vtl.Tensor[f32]`: 1 / (1 + exp(-x)) through the device
    with the arithmetic of nn/internal/activation.v:35-40."""
    if not hip_linear_enabled():
        raise RuntimeError("sigmoid_forward_hip_f32: set VTL_USE_HIP=1 to enable")
    return _activation_host_roundtrip(x, "sigmoid")


def matmul_gate_backward_hip(grad: np.ndarray, a: np.ndarray, b: np.ndarray):
    """`MatMulGate.backward` (autograd/gates_blas.v:43-48) through the device:
    [grad . b^T, a^T . grad], the transposes taken by flag instead of `.t()` copies."""
    if not hip_backward_enabled():
        raise RuntimeError("matmul_gate_backward_hip: set VTL_USE_HIP=1 and VTL_HIP_BACKWARD=1")
    g = _as_float_matrix(grad, "matmul backward")
    av = _as_float_matrix(a, "matmul backward").astype(g.dtype, copy=False)
    bv = _as_float_matrix(b, "matmul backward").astype(g.dtype, copy=False)
    if av.shape[1] != bv.shape[0] or g.shape != (av.shape[0], bv.shape[1]):
        raise ValueError(f"Invalid shapes for matrix multiplication {list(av.shape)} and {list(bv.shape)}")
    g_dev, a_dev, b_dev = HipTensor.from_host(g), HipTensor.from_host(av), HipTensor.from_host(bv)
    outs = []
    try:
        outs.append(matmul_hip(g_dev, b_dev, False, True))    # [M,N] . [K,N]^T -> [M,K]
        outs.append(matmul_hip(a_dev, g_dev, True, False))    # [M,K]^T . [M,N] -> [K,N]
        return HipTensor.cpu_all(outs)
    finally:
        for t in (g_dev, a_dev, b_dev, *outs):
            t.release()
