"""One row through layers with one scale for all weights: in one launch a layer, the same bits as the same row quantized by
itself and then multiplied, which the other tests hold against the CPU oracle."""
import numpy as np
import pytest

from helpers import dev
from vtl_amd import PER_CHANNEL, PER_TENSOR, capi
from vtl_amd.layers import QuantizedWeights, forward_host
from vtl_amd.tensor import linear_i8_hip

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
    """Rows that start at any byte, shorter than the kernels' pieces: quantized in the launch of the product."""
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


def test_rows_of_a_layer_with_one_scale_stay_refused(hip):
    w = QuantizedWeights(np.ones((8, 16), np.float32), None, PER_TENSOR, frozen=True)
    x, y = dev(np.ones((1, 16), np.float32)), dev(np.zeros((1, 8), np.float32))
    assert capi.status("vtl_hip_layer_f32", w.layer, x.ptr, y.ptr, 1, 0, None, 0) == capi.ERR_INVALID_ARG
    for t in (w, x, y):
        t.release()
