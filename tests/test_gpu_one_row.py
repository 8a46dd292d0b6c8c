"""One row through layers with one scale for all weights, and a few short rows: in one launch a layer, the same bits as the same rows
quantized by themselves and then multiplied, which the other tests hold against the CPU oracle.  (Beside tests that name streams a host
call's rows are uploaded; over the link: test_gpu_null_stream.py.)"""
import numpy as np
import pytest

import oracle
from helpers import dev, h2d, raw_device_buffer
from vtl_amd import PER_CHANNEL, PER_TENSOR, capi
from vtl_amd.layers import QuantizedWeights, forward_host, linear_forward_hip_i8_device
from vtl_amd.tensor import HipTensor, linear_i8_hip

pytestmark = pytest.mark.gpu


# whole, ragged and padded rows (2^18 codes and more), rows that are too long for the matrix-vector kernels, inputs that are uploaded first
@pytest.mark.parametrize("dims", [(16, 16), (1, 1), (17, 5), (784, 256), (1001, 300), (4096, 100), (1000, 1000), (1001, 1000), (6000, 70),
                                  (20000, 33), (20001, 40), (300, 500, 64), (64, 1001, 300, 7)], ids=str)
@pytest.mark.parametrize("bias", [True, False])
def test_one_row_per_tensor(hip, dims, bias):
    rng = np.random.default_rng(sum(dims))
    modes = [(PER_TENSOR, PER_CHANNEL)[i % 3 == 1] for i in range(len(dims) - 1)]
    x = rng.standard_normal((1, dims[0])).astype(np.float32)
    weights = [QuantizedWeights((rng.standard_normal((n, k)) / np.sqrt(k)).astype(np.float32),
                                rng.standard_normal(n).astype(np.float32) if bias else None, m, frozen=True)
               for k, n, m in zip(dims, dims[1:], modes)]
    print("one row", dims, bias, flush=True)
    want = x
    for w in weights:
        xd = dev(want)
        q, s = xd.quantize_i8(-1)
        y = linear_i8_hip(q, s, w.w_q, w.sw, w.bias)
        want = y.cpu().copy()
        for t in (xd, q, s, y):
            t.release()
    for _ in range(2):
        got = forward_host(x, [w.layer for w in weights], len(weights), dims[-1])
        assert np.array_equal(got.view(np.int32), want.view(np.int32))
    for w in weights:
        w.release()


@pytest.mark.parametrize("k", [15, 16, 17, 31, 33, 100, 127, 238, 255, 257])
@pytest.mark.parametrize("n", [1, 7, 65, 1003])
def test_few_short_rows(hip, n, k):
    """Rows that start at any byte, shorter than the kernels' pieces, from host to host: one or two of them quantized in the
    launch of the product, more in one before it."""
    rng = np.random.default_rng(n + k)
    w = QuantizedWeights(rng.standard_normal((n, k)).astype(np.float32), rng.standard_normal(n).astype(np.float32), PER_CHANNEL, frozen=True)
    for m in (1, 2, 3, 4, 5, 8):
        x = rng.standard_normal((m, k)).astype(np.float32)
        print("short rows", m, n, k, flush=True)
        xd = dev(x)
        q, s = xd.quantize_i8(0)
        y = linear_i8_hip(q, s, w.w_q, w.sw, w.bias)
        want = y.cpu().copy()
        for t in (xd, q, s, y):
            t.release()
        for _ in range(2):
            assert np.array_equal(forward_host(x, [w.layer], 1, n).view(np.int32), want.view(np.int32))
    w.release()


# edges of the kernels for 2, 4 and 8 rows and of where they are taken, one weight row and more than a wave has
@pytest.mark.parametrize("k", [16, 17, 31, 33, 100, 127, 238, 255])
def test_few_short_rows_in_device_memory(hip, guard_bands, k):
    """Dense codes at odd addresses and f32 rows that are not 16-byte aligned, quantized in the launch of the product (and in one of
    their own beyond the last size of each number of rows): the oracle's bits, nothing written beside them."""
    rng = np.random.default_rng(k)
    for n, off, rows in ((1, 1, (2, 3, 5, 8)), (7, 2, (2, 4, 7)), (65, 3, (2, 3, 4, 5, 6, 7, 8)), (1003, 1, (1, 2, 3, 8)), (2048, 5, (4, 5, 8)),
                         (2049, 7, (4, 8)), (8192, 3, (3,)), (8193, 1, (2, 4))):
        codes, sw = rng.integers(-127, 128, (n, k), dtype=np.int8), rng.uniform(1e-3, 2e-3, n).astype(np.float32)
        bias = rng.standard_normal(n).astype(np.float32)
        held, swd, bd = raw_device_buffer(n * k + off), dev(sw), dev(bias)
        h2d(held.ptr + off, codes)
        for m in rows:
            print("short rows on the device", m, n, k, flush=True)
            x = rng.standard_normal((m, k)).astype(np.float32)
            want = oracle.linear_f32_dynquant(x, codes, sw, bias, threads=4)
            xd, y = raw_device_buffer(4 * m * k + 4), HipTensor.empty([m, n], np.float32)
            h2d(xd.ptr + 4, x)
            capi.call("vtl_hip_linear_f32_dynquant", xd.ptr + 4, held.ptr + off, swd.ptr, bd.ptr, y.ptr, m, n, k, 0, None, 0)
            assert np.array_equal(y.cpu().view(np.int32), want.view(np.int32)), (m, n, k)
            xd.release()
            y.release()
        for t in (held, swd, bd):
            t.release()


@pytest.mark.parametrize("n,k", [(2500, 110), (2700, 100), (8192, 33), (16384, 17), (16385, 18), (20000, 238)])
def test_few_short_rows_of_padded_weights(hip, n, k):
    """The same of a layer whose rows of codes are padded."""
    rng = np.random.default_rng(n + k)
    w = rng.standard_normal((n, k)).astype(np.float32)
    codes, sw = oracle.quantize(w, True)
    bias = rng.standard_normal(n).astype(np.float32)
    qw = QuantizedWeights(w, bias, PER_CHANNEL, frozen=True)
    assert qw.w_rows is not None
    for m in (1, 2, 3, 4, 5, 8):
        print("short padded rows", m, n, k, flush=True)
        x = rng.standard_normal((m, k)).astype(np.float32)
        xd = dev(x)
        y = linear_forward_hip_i8_device(xd, qw)
        assert np.array_equal(y.cpu().view(np.int32), oracle.linear_f32_dynquant(x, codes, sw, bias, threads=4).view(np.int32)), m
        for t in (xd, y):
            t.release()
    qw.release()


@pytest.mark.parametrize("dims", [(100, 200, 250, 64), (33, 17, 255, 31), (100, 20000, 65)], ids=str)
def test_few_short_rows_through_several_layers(hip, dims):
    """Rows over the link, in device memory, and results over the link, each in the form that is taken there."""
    rng = np.random.default_rng(sum(dims))
    weights = [rng.standard_normal((n, k)).astype(np.float32) for k, n in zip(dims, dims[1:])]
    qw = [QuantizedWeights(w, None, PER_CHANNEL, frozen=True) for w in weights]
    for m in (1, 2, 3, 4, 8):
        x = rng.standard_normal((m, dims[0])).astype(np.float32)
        want = x
        for w in weights:
            codes, sw = oracle.quantize(w, True)
            want = oracle.linear_f32_dynquant(want, codes, sw, np.zeros(len(w), np.float32), threads=4)
        print("short rows through layers", m, dims, flush=True)
        got = forward_host(x, [w.layer for w in qw], len(qw), dims[-1])
        assert np.array_equal(got, want), m
    for w in qw:
        w.release()


def test_rows_of_a_layer_with_one_scale_stay_refused(hip):
    w = QuantizedWeights(np.ones((8, 16), np.float32), None, PER_TENSOR, frozen=True)
    x, y = dev(np.ones((1, 16), np.float32)), dev(np.zeros((1, 8), np.float32))
    assert capi.status("vtl_hip_layer_f32", w.layer, x.ptr, y.ptr, 1, 0, None, 0) == capi.ERR_INVALID_ARG
    for t in (w, x, y):
        t.release()
