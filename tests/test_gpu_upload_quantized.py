"""Rows that are quantized on their way to the device, by the host's threads or as they come over the link: the same bits as an upload and the quantizer behind it.  (Beside tests that name
streams each call waits for its end; without a wait, and with transfers behind it: test_gpu_null_stream.py.)"""
import numpy as np
import pytest

from helpers import dev
from vtl_amd import PER_CHANNEL, PER_TENSOR, QuantLinearLayer, capi
from vtl_amd.layers import QuantizedWeights
from vtl_amd.tensor import HipTensor

pytestmark = pytest.mark.gpu


# By the host's threads, rows of any of these lengths: more and less than what one thread makes, rows that do not divide the pieces a transfer is cut into
# (rows are not cut).  By the device, 32 MiB and more in rows of 2048 to 8192 values as they come over the link: edges of a workgroup's registers, rows
# that do not divide the pieces; less, longer, shorter and odd rows go in two steps.
@pytest.mark.parametrize("rows,cols", [(8192, 1024), (8191, 1024), (8200, 1028), (4096, 2048), (4095, 2048), (4200, 2044), (4100, 2052), (3000, 2800), (2049, 4096), (2100, 4100),
                                       (1024, 8192), (1031, 8188), (1030, 8196), (33000, 256), (8300, 1023), (300, 1024), (1, 4)])
@pytest.mark.parametrize("extra", [0, 4096 + 20])
def test_same_bits_as_upload_and_quantize(hip, rows, cols, extra):
    rng = np.random.default_rng(rows + cols)
    x = rng.standard_normal((rows, cols)).astype(np.float32) * np.float32(10.0) ** rng.integers(-3, 4, (rows, 1)).astype(np.float32)
    x[rows // 2] = 0.0
    x[rows // 3, :: 5] = np.nan
    x[-1, cols // 2] = np.inf
    more = rng.integers(0, 256, extra, dtype=np.uint8)
    print("rows", rows, cols, extra, flush=True)
    for per_row in (1, 0):
        xd = dev(x)
        want_q, want_s = xd.quantize_i8(0 if per_row else -1)
        q, s = HipTensor.empty([rows, cols], np.int8), HipTensor.empty([rows if per_row else 1], np.float32)
        room = HipTensor.empty([extra + 64], np.uint8)
        for _ in range(2):
            capi.call("vtl_hip_upload_quantized", x.ctypes.data, rows, cols, per_row, q.ptr, s.ptr, room.ptr + 16 if extra else None,
                      more.ctypes.data if extra else None, extra)
            assert np.array_equal(q.cpu(), want_q.cpu())
            assert np.array_equal(s.cpu().view(np.int32), want_s.cpu().view(np.int32))
            assert np.array_equal(room.cpu()[16:16 + extra], more)
        for t in (xd, want_q, want_s, q, s, room):
            t.release()


# Whatever processors the machine has: the rows of 32 MiB and more, by the device's kernel and by the host's threads
@pytest.mark.parametrize("rows,cols", [(4096, 2048), (4095, 2048), (4200, 2044), (4100, 2052), (3000, 2800), (2049, 4096), (2100, 4100), (1024, 8192), (1031, 8188),
                                       (1030, 8196)])
@pytest.mark.parametrize("extra", [0, 4096 + 20])
@pytest.mark.parametrize("by_host", ["0", "1"])
def test_same_bits_by_the_host_and_on_the_link(hip, knobs, rows, cols, extra, by_host):
    knobs.setenv("VTL_HIP_HOST_QUANTIZE", by_host)
    test_same_bits_as_upload_and_quantize(hip, rows, cols, extra)


def test_errors(hip):
    x, q = np.zeros((4, 8), np.float32), HipTensor.empty([4, 8], np.int8)
    s = HipTensor.empty([4], np.float32)
    for args in ((None, 4, 8, 1, q.ptr, s.ptr, None, None, 0), (x.ctypes.data, -1, 8, 1, q.ptr, s.ptr, None, None, 0),
                 (x.ctypes.data, 4, 8, 1, None, s.ptr, None, None, 0), (x.ctypes.data, 4, 8, 1, q.ptr, None, None, None, 0),
                 (x.ctypes.data, 4, 8, 1, q.ptr, s.ptr, None, x.ctypes.data, 4)):
        assert capi.status("vtl_hip_upload_quantized", *args) == capi.ERR_INVALID_ARG
    for t in (q, s):
        t.release()


# The same by the host's units and by the device's: what one thread makes and what several do, pieces that rows do not divide, rows too short
# for it, one scale for all, and whole forwards whose first layer takes codes (more than 32 rows, dense and padded)
@pytest.mark.parametrize("rows,cols", [(64, 784), (33, 15), (300, 1023), (257, 1021), (263, 4099), (1000, 17), (70, 70001), (5000, 1027),
                                       (4, 100), (20, 800), (32, 512), (33, 497), (64, 256), (65, 256), (128, 128), (18, 900), (1000, 16)])
def test_by_the_host_and_by_the_device(hip, knobs, rows, cols):
    rng = np.random.default_rng(rows * 31 + cols)
    x = rng.standard_normal((rows, cols)).astype(np.float32)
    x[rows // 3, :: 5] = np.nan
    w = rng.standard_normal((40, cols)).astype(np.float32)
    bias = rng.standard_normal((1, 40)).astype(np.float32)
    print("rows", rows, cols, flush=True)
    got = []
    for by_host in ("0", "1"):
        knobs.setenv("VTL_HIP_HOST_QUANTIZE", by_host)
        out = []
        for mode in (PER_CHANNEL, PER_TENSOR):
            qw = QuantizedWeights(x, None, mode)
            out += [qw.w_q.cpu().copy(), qw.sw.cpu().view(np.int32).copy()]
            qw.release()
            layer = QuantLinearLayer(w, bias, mode=mode, requires_grad=False)
            out += [layer.forward(x).copy(), layer.forward(x[: rows // 2]).copy()]
            layer.release()
        got.append(out)
    for a, b in zip(*got):
        assert np.array_equal(a, b, equal_nan=a.dtype == np.float32)


# Forwards and weights where sizes say who quantizes, by them and by the device: few dense rows with one scale that are no whole vectors, and short rows
@pytest.mark.parametrize("rows,cols", [(2, 1023), (2, 1025), (3, 255), (3, 257), (8, 300), (8, 2047), (8, 2049), (5, 4001), (9, 1372),
                                       (264, 31), (265, 31), (512, 32), (513, 32), (86, 191), (86, 192), (129, 128), (341, 192), (64, 256), (64, 257), (8456, 31),
                                       (8457, 32)])
def test_same_bits_whoever_quantizes(hip, knobs, rows, cols):
    rng = np.random.default_rng(rows * 37 + cols)
    x, w = rng.standard_normal((rows, cols)).astype(np.float32), rng.standard_normal((40, cols)).astype(np.float32)
    print("rows", rows, cols, flush=True)
    got = []
    for who in ("0", "2"):
        knobs.setenv("VTL_HIP_HOST_QUANTIZE", who)
        out = []
        for mode in (PER_CHANNEL, PER_TENSOR):
            qw = QuantizedWeights(x, None, mode)
            layer = QuantLinearLayer(w, None, mode=mode, requires_grad=False)
            out += [qw.w_q.cpu().copy(), qw.sw.cpu().view(np.int32).copy(), layer.forward(x).copy()]
            qw.release()
            layer.release()
        got.append(out)
    for a, b in zip(*got):
        assert np.array_equal(a, b)
