"""What the library does only while a process uses the null stream alone, checked in a process of its
own: other tests of this run name streams, and from then on those paths are off."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
import os
os.environ["VTL_USE_HIP"] = os.environ["VTL_HIP_BACKWARD"] = "1"
import numpy as np
import oracle
from vtl_amd import PER_TENSOR, QuantLinearLayer, linear_backward_hip_f32
rng = np.random.default_rng(7)
# Linear backward, host to host: gradients below and above the 128 KiB from which the device writes them into
# pinned memory itself; operands below and above the 1 MiB up to which an upload is one piece
for m, n, k, dt in ((5, 33, 17, np.float32), (64, 256, 784, np.float32), (16, 1023, 401, np.float64),
                    (31, 700, 1301, np.float32), (48, 130, 1, np.float32)):
    for turn in range(3):
        g, x, w = (rng.standard_normal(s).astype(dt) for s in ((m, n), (m, k), (n, k)))
        got = linear_backward_hip_f32(g, x, w, True)
        eps = np.finfo(dt).eps
        g64, x64, w64 = g.astype(np.float64), x.astype(np.float64), w.astype(np.float64)
        for out, want, size in ((got[0], g64 @ w64, abs(g64) @ abs(w64)), (got[1], g64.T @ x64, abs(g64).T @ abs(x64)),
                                (got[2], g64.sum(0)[None], abs(g64).sum(0)[None])):
            # one rounding to the type, and sums of up to max(m, n) f64 products in two orders
            bound = eps * abs(want) + 2 * max(m, n) * np.finfo(np.float64).eps * size
            assert (abs(out - want) <= bound).all(), (m, n, k, dt, turn)
    print("backward", m, n, k, np.dtype(dt).name, "ok", flush=True)
# one scale for x, read over the link by the quantizer (up to 1 MiB, 262144 elements) or uploaded
for m, k in ((1, 16), (64, 784), (3, 21845), (70, 1000), (3, 87381), (2, 131072), (5, 52429)):
    w = rng.standard_normal((40, k), dtype=np.float32)
    layer = QuantLinearLayer(w, mode=PER_TENSOR)
    for turn in range(3):
        x = rng.standard_normal((m, k), dtype=np.float32)
        xq, sx = oracle.quantize(x, False)
        wq, sw = oracle.quantize(w, False)
        acc = xq.astype(np.int64) @ wq.astype(np.int64).T
        want = acc.astype(np.float32) * (sx.reshape(()) * sw.reshape(())) + np.float32(0)
        assert np.array_equal(layer.forward(x), want), (m, k, turn)
    layer.release()
    print("layer", m, k, "ok", flush=True)
# a scale per row: the same from 33 rows on, in one pass and (ragged rows) in two
for m, k in ((32, 785), (33, 785), (33, 788), (64, 4095), (64, 4096), (65, 4033), (128, 2049)):
    w = rng.standard_normal((40, k), dtype=np.float32)
    wq, sw = oracle.quantize(w, True)
    layer = QuantLinearLayer(w)
    for turn in range(3):
        x = rng.standard_normal((m, k), dtype=np.float32)
        assert np.array_equal(layer.forward(x), oracle.linear_f32_dynquant(x, wq, sw, np.zeros(40, np.float32))), (m, k, turn)
    layer.release()
    print("rows", m, k, "ok", flush=True)
"""


THREADS = r"""
import threading
import numpy as np
from vtl_amd import capi
from vtl_amd.tensor import HipTensor, matmul_hip
rng = np.random.default_rng(11)
# products whose K is cut over the grid, from several threads of a program that has the null stream alone
bad = []
def products(seed):
    r = np.random.default_rng(seed)
    capi.call("vtl_hip_set_device", 0)
    for m, n, k in ((64, 256, 784), (16, 256, 1024), (64, 64, 4096), (33, 65, 777)) * 6:
        a, b = r.integers(-8, 9, (m, k)).astype(np.float32), r.integers(-8, 9, (k, n)).astype(np.float32)
        da, db = HipTensor.from_host(a), HipTensor.from_host(b)
        c = [matmul_hip(da, db) for _ in range(4)]
        want = (a.astype(np.float64) @ b).astype(np.float32)
        if not all(np.array_equal(t.cpu(), want) for t in c):
            bad.append((seed, m, n, k))
        for t in (da, db, *c):
            t.release()
threads = [threading.Thread(target=products, args=(s,)) for s in range(4)]
for t in threads:
    t.start()
for t in threads:
    t.join()
assert not bad, bad
print("ok")
"""


RESULTS = r"""
import sys
import threading
import numpy as np
import oracle
from vtl_amd import PER_CHANNEL, PER_TENSOR, QuantLinearLayer, Sequential, capi, matmul_hip_host
# Results that the last launch writes to the host itself: pieces of eight (up to 8 rows, 2048 results) and ordinary stores
# behind it, results in staging memory and in the library's own (from 128 KiB on), in 8 MiB and more; the kernels
# for a few rows, small products, 32-row blocks, tiles, K cut over the grid; inputs over the link (few rows: at most 20 KiB or
# past 32 KiB) and uploaded
LAYERS = [(1, 1, 64), (1, 2048, 300), (1, 2049, 512), (2, 1024, 256), (2, 1025, 1100), (3, 9, 1700), (8, 256, 640), (8, 40, 1024),
          (5, 700, 2100), (17, 2050, 512), (33, 100, 784), (40, 900, 1024), (64, 300, 2100), (65, 4100, 640), (200, 801, 1664),
          (256, 8191, 72), (256, 8193, 72),
          (256, 4096, 72), (256, 4128, 72), (100, 6553, 72), (100, 6554, 72)]   # either side of what is written directly
def layers(seed):
    rng = np.random.default_rng(seed)
    for m, n, k in LAYERS:
        w, b = rng.standard_normal((n, k), dtype=np.float32), rng.standard_normal((1, n), dtype=np.float32)
        for mode in (PER_CHANNEL, PER_TENSOR):
            layer = QuantLinearLayer(w, b, mode=mode, requires_grad=False)
            wq, sw = oracle.quantize(w, mode == PER_CHANNEL)
            for turn in range(3):
                x = rng.standard_normal((m, k), dtype=np.float32)
                xq, sx = oracle.quantize(x, mode == PER_CHANNEL)
                want = oracle.epilogue(oracle.gemm_i8_i32(xq, wq, threads=4), sx, sw, b.reshape(-1))
                assert np.array_equal(layer.forward(x), want), (m, n, k, mode, turn)
            layer.release()
def network(seed):   # a ReLU folded into the last layer, and one more that is not
    rng = np.random.default_rng(seed)
    w1, w2 = rng.standard_normal((70, 130), dtype=np.float32), rng.standard_normal((40, 70), dtype=np.float32)
    for relus in (0, 1, 2):
        net = Sequential().input([130]).linear(70, weights=w1).relu().linear(40, weights=w2)
        for _ in range(relus):
            net.relu()
        for m in (1, 6, 40):
            x = rng.standard_normal((m, 130), dtype=np.float32)
            y = x
            for w, r in ((w1, True), (w2, relus > 0)):
                wq, sw = oracle.quantize(w, True)
                y = oracle.linear_f32_dynquant(y, wq, sw, np.zeros(len(w), np.float32), relu=r)
            assert np.array_equal(net.forward(x, no_grad=True), y), (relus, m)
        net.release()
def products(seed):   # whole numbers: every sum is exact; whole tiles of 128, K cut, results past 8 MiB
    rng = np.random.default_rng(seed)
    for m, n, k, dt in ((1, 1, 1, "f4"), (37, 41, 100, "f8"), (33, 257, 3000, "f4"), (128, 256, 64, "f8"), (180, 183, 32, "f4"),
                        (1024, 1024, 8, "f8"), (1030, 1030, 8, "f8"), (300, 655, 40, "f4"), (300, 656, 40, "f4"),
                        # operands that go up together: in one launch (640 KiB in all), in turn (1 MiB each) or in pieces, several a
                        # launch, odd addresses
                        (80, 80, 1024, "f4"), (80, 81, 1024, "f4"), (256, 256, 1024, "f4"), (257, 256, 1024, "f4"), (64, 64, 2048, "f4"), (64, 65, 2048, "f4"), (401, 403, 777, "f8"), (701, 903, 1201, "f4"),
                        (2051, 65, 1103, "f8")):
        for turn in range(2):
            a, b = rng.integers(-8, 9, (m, k)).astype(dt), rng.integers(-8, 9, (k, n)).astype(dt)
            assert np.array_equal(matmul_hip_host(a, b), (a.astype("f8") @ b.astype("f8")).astype(dt)), (m, n, k, dt, turn)
capi.call("vtl_hip_set_device", 0)
for part in (layers, network, products):
    part(1)
    print(part.__name__, flush=True)
bad = []
def guarded(part, seed):
    try:
        part(seed)
    except BaseException as e:
        bad.append((part.__name__, seed, repr(e)))
threads = [threading.Thread(target=guarded, args=(p, s)) for s, p in enumerate((layers, layers, network, products), 2)]
for t in threads:
    t.start()
for t in threads:
    t.join()
assert not bad, bad
print("ok")
"""


def test_results_written_by_the_last_launch(hip):
    done = subprocess.run([sys.executable, "-c", RESULTS], cwd=ROOT, stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                          text=True, timeout=110)
    assert done.returncode == 0 and done.stdout.strip().endswith("ok"), done.stdout[-2000:]


GRADIENTS = r"""
import ctypes as C
import itertools
import threading
import numpy as np
from vtl_amd import capi
# Every set of gradients that can be asked for.  The last product tells the host that all of them are there (dX's, or dW's where there
# is no dX), or a launch behind (dB alone, dX or dW too large to be written over the link), and what was not written over the
# link comes down.  Memory of the caller's own: through staging memory, 1 MiB for the three together; of
# vtl_hip_host_alloc: written in place beyond 4 KiB and up to 8 MiB.  Whole numbers: every sum is exact.
SIZES = [(3, 5, 7), (64, 256, 784), (40, 700, 1001), (17, 1030, 2100), (600, 64, 2100), (2, 2049, 1024)]
def memory(count, dt, pool, kept):
    if not pool:
        return np.empty(count, dt)
    at = C.c_void_p()
    capi.call("vtl_hip_host_alloc", C.byref(at), count * dt.itemsize)
    kept.append(at)
    return np.frombuffer((C.c_char * (count * dt.itemsize)).from_address(at.value), dt)
def gradients(seed):
    rng = np.random.default_rng(seed)
    for (m, n, k), dt in itertools.product(SIZES, (np.dtype("f4"), np.dtype("f8"))):
        for pools in ((0, 0, 0), (1, 1, 1), (1, 0, 0), (0, 1, 0)):
            kept = []
            for wanted in range(1, 8):
                g, x, w = (rng.integers(-9, 10, s).astype(dt) for s in ((m, n), (m, k), (n, k)))
                want = [g @ w, g.T @ x, g.sum(0)]
                out = [memory(a.size, dt, p, kept) if wanted >> i & 1 else None for i, (a, p) in enumerate(zip(want, pools))]
                for o in out:
                    if o is not None:
                        o[:] = -12345
                capi.call("vtl_hip_linear_backward_host_" + ("f32" if dt.itemsize == 4 else "f64"), g.ctypes.data,
                          x.ctypes.data if wanted & 2 else None, w.ctypes.data if wanted & 1 else None,
                          *(None if o is None else o.ctypes.data for o in out), m, n, k)
                for name, o, a in zip(("dx", "dw", "db"), out, want):
                    assert o is None or np.array_equal(o, a.reshape(-1)), (m, n, k, dt, pools, wanted, name)
            for at in kept:
                capi.call("vtl_hip_host_free", at)
capi.call("vtl_hip_set_device", 0)
gradients(1)
print("null stream", flush=True)
bad = []
def guarded(seed, stream=None):
    try:
        if stream:
            capi.call("vtl_hip_set_stream", stream)
        gradients(seed)
    except BaseException as e:
        bad.append((seed, repr(e)))
def at_once(*calls):
    threads = [threading.Thread(target=guarded, args=c) for c in calls]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, bad
at_once((2,), (3,))
print("two threads", flush=True)
hiprt = C.CDLL("libamdhip64.so")
stream = C.c_void_p()
assert hiprt.hipStreamCreateWithFlags(C.byref(stream), C.c_uint(1)) == 0
at_once((4, stream))
print("ok")
"""


def test_every_set_of_gradients(hip):
    done = subprocess.run([sys.executable, "-c", GRADIENTS], cwd=ROOT, stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                          text=True, timeout=110)
    assert done.returncode == 0 and done.stdout.rstrip().endswith("ok"), done.stdout[-3000:]


SMALL_GRADIENTS = r"""
import os
os.environ["VTL_USE_HIP"] = os.environ["VTL_HIP_BACKWARD"] = "1"
import threading
import numpy as np
from vtl_amd import capi, linear_backward_hip_f32
# Operands of up to 640 KiB in all go up together and one launch has every gradient: either side of that, and sizes that the one
# launch does not take (a row or a column of one).  Whole numbers: every sum is exact.
SIZES = {"f4": [(64, 345, 346), (64, 346, 346), (513, 64, 64), (40, 700, 64)], "f8": [(64, 229, 229), (64, 230, 230), (513, 33, 47)]}
def gradients(seed):
    rng = np.random.default_rng(seed)
    for dt in SIZES:
        for m, n, k in [(1, 1, 1), (1, 2, 3), (5, 1, 7), (3, 9, 1), (17, 33, 65), (64, 64, 64), (16, 256, 256)] + SIZES[dt]:
            for bias in (True, False):
                for turn in range(2):
                    g, x, w = (rng.integers(-8, 9, s).astype(dt) for s in ((m, n), (m, k), (n, k)))
                    dx, dw, db = linear_backward_hip_f32(g, x, w, bias)
                    assert np.array_equal(dx, g @ w) and np.array_equal(dw, g.T @ x), (dt, m, n, k)
                    assert np.array_equal(db.reshape(-1), g.sum(axis=0) if bias else np.zeros(n)), (dt, m, n, k)
capi.call("vtl_hip_set_device", 0)
gradients(1)
print("one thread", flush=True)
bad = []
def guarded(seed):
    try:
        gradients(seed)
    except BaseException as e:
        bad.append((seed, repr(e)))
threads = [threading.Thread(target=guarded, args=(s,)) for s in (2, 3)]
for t in threads:
    t.start()
for t in threads:
    t.join()
assert not bad, bad
print("ok")
"""


def test_small_gradients_in_one_upload_and_one_launch(hip):
    done = subprocess.run([sys.executable, "-c", SMALL_GRADIENTS], cwd=ROOT, stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                          text=True, timeout=110)
    assert done.returncode == 0 and done.stdout.rstrip().endswith("ok"), done.stdout[-3000:]


ONE_ROW = r"""
import numpy as np
import oracle
from vtl_amd import PER_CHANNEL, PER_TENSOR, capi
from vtl_amd.layers import QuantizedWeights, forward_host
# One row through layers with one scale for their weights, and a few short rows, read over the link by the launch that quantizes
# them or (20 to 32 KiB) uploaded: whole, ragged and padded rows, rows too long for the matrix-vector kernels, several layers
capi.call("vtl_hip_set_device", 0)
rng = np.random.default_rng(5)
for dims, rows in [((16, 16), (1,)), ((1, 1), (1,)), ((17, 5), (1, 2, 8)), ((784, 256), (1,)), ((1001, 300), (1, 2)), ((1000, 1000), (1,)), ((1001, 1000), (1,)),
                   ((6000, 70), (1,)), ((20000, 33), (1,)), ((20001, 40), (1,)), ((300, 500, 64), (1,)), ((64, 1001, 300, 7), (1, 3)),
                   ((100, 2700), (1, 2, 3, 8)), ((238, 1003), (1, 2, 3, 8)), ((100, 16385), (1, 2)), ((100, 200, 250, 64), (1, 2, 4, 8))]:
    for mode in (PER_TENSOR, PER_CHANNEL):
        weights = [(rng.standard_normal((n, k)) / np.sqrt(k)).astype(np.float32) for k, n in zip(dims, dims[1:])]
        qw = [QuantizedWeights(w, None, mode, frozen=True) for w in weights]
        for m in rows if mode == PER_CHANNEL else (1,):
            for turn in range(3):
                x = rng.standard_normal((m, dims[0])).astype(np.float32)
                y = x
                for w in weights:
                    wq, sw = oracle.quantize(w, mode == PER_CHANNEL)
                    xq, sx = oracle.quantize(y, mode == PER_CHANNEL)
                    y = oracle.epilogue(oracle.gemm_i8_i32(xq, wq, threads=4), sx, sw, None)
                assert np.array_equal(forward_host(x, [w.layer for w in qw], len(qw), dims[-1]), y), (dims, mode, m, turn)
        for w in qw:
            w.release()
    print(dims, flush=True)
print("ok")
"""


def test_one_row_and_short_rows_over_the_link(hip):
    done = subprocess.run([sys.executable, "-c", ONE_ROW], cwd=ROOT, stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                          text=True, timeout=110)
    assert done.returncode == 0 and done.stdout.rstrip().endswith("ok"), done.stdout[-3000:]


QUANTIZED_UPLOADS = r"""
import numpy as np
import oracle
from vtl_amd import capi
from vtl_amd.tensor import HipTensor
# Rows that are quantized on their way to the device, without a wait: the caller's memory is its own again on return, and small
# and large transfers come directly behind, through the same staging memory
capi.call("vtl_hip_set_device", 0)
rng = np.random.default_rng(9)
def tensor(shape, dtype):
    return HipTensor.empty(shape, dtype)
for rows, cols, extra in ((8192, 1024, 0), (8200, 1028, 4100), (4096, 2048, 0), (4111, 2048, 4100), (2049, 4096, 65537), (1031, 8188, 20), (4100, 2052, 3 << 20), (300, 1024, 64)):
    held, waiting = [], []
    for turn in range(2):
        x = rng.standard_normal((rows, cols), dtype=np.float32)
        x[rows // 2] = 0.0
        more, small, large = (rng.integers(0, 256, n, dtype=np.uint8) for n in (extra, 5000, 21 << 20))
        want = oracle.quantize(x, True, threads=8) + (more.copy(), small.copy(), large.copy())
        q, s, e, a, b = tensor([rows, cols], np.int8), tensor([rows], np.float32), tensor([extra + 16], np.uint8), tensor([5000], np.uint8), tensor([21 << 20], np.uint8)
        capi.call("vtl_hip_upload_quantized", x.ctypes.data, rows, cols, 1, q.ptr, s.ptr, e.ptr if extra else None,
                  more.ctypes.data if extra else None, extra)
        x[:] = np.nan
        more[:] = 0
        for t, src in ((a, small), (b, large))[:: 1 - 2 * turn]:
            capi.call("vtl_hip_upload", t.ptr, src.ctypes.data, src.nbytes)
            src[:] = 0
        waiting.append(((q, s, e, a, b), want))
    for tensors, want in waiting:
        for t, w in zip(tensors, want):
            assert np.array_equal(t.cpu().reshape(-1)[:w.size], w.reshape(-1)), (rows, cols, extra)
            t.release()
    print(rows, cols, extra, flush=True)
print("ok")
"""


def test_uploads_behind_rows_quantized_on_their_way(hip):
    done = subprocess.run([sys.executable, "-c", QUANTIZED_UPLOADS], cwd=ROOT, stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                          text=True, timeout=110)
    assert done.returncode == 0 and done.stdout.rstrip().endswith("ok"), done.stdout[-3000:]


@pytest.mark.parametrize("by_host", ["0", "1"])      # as they come over the link, and by the host's threads (with up to 64 KiB beside them)
def test_uploads_behind_rows_quantized_by_the_host_and_on_the_link(hip, monkeypatch, by_host):
    monkeypatch.setenv("VTL_HIP_HOST_QUANTIZE", by_host)     # (of the process that it starts)
    test_uploads_behind_rows_quantized_on_their_way(hip)


def test_products_from_several_threads_on_the_null_stream(hip):
    done = subprocess.run([sys.executable, "-c", THREADS], cwd=ROOT, stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                          text=True, timeout=100)
    assert done.returncode == 0 and done.stdout.strip().endswith("ok"), done.stdout[-2000:]


OTHER_STREAM = r"""
import ctypes as C
import numpy as np
import oracle
from vtl_amd import QuantLinearLayer, capi
from vtl_amd.tensor import HipTensor
hiprt = C.CDLL("libamdhip64.so")
capi.call("vtl_hip_set_device", 0)
stream = C.c_void_p()
assert hiprt.hipStreamCreateWithFlags(C.byref(stream), C.c_uint(1)) == 0     # non-blocking
pinned = C.c_void_p()
capi.call("vtl_hip_host_alloc", C.byref(pinned), 40 << 20)
def read(t):
    assert hiprt.hipMemcpyAsync(pinned, C.c_void_p(t.ptr), C.c_size_t(t.data.size), C.c_int(2), stream) == 0
    assert hiprt.hipStreamSynchronize(stream) == 0
    return np.frombuffer((C.c_uint8 * t.data.size).from_address(pinned.value), t.dtype).reshape(t.shape)
rng = np.random.default_rng(3)
for n in (1, 1000, 262144, 262145, 5 << 20, 9 << 20):
    x = rng.standard_normal(n, dtype=np.float32)
    t = HipTensor.from_host(x)
    assert np.array_equal(read(t), x), n
    t.release()
for n, k in ((300, 1024), (1000, 1023), (2048, 4096)):
    w = rng.standard_normal((n, k), dtype=np.float32)
    qw = QuantLinearLayer(w, requires_grad=False).quantized()
    codes, scales = oracle.quantize(w, True)
    assert np.array_equal(read(qw.w_q), codes) and np.array_equal(read(qw.sw), scales), (n, k)
    if qw.w_rows is not None:
        assert np.array_equal(read(qw.w_rows)[:, :k], codes)
    qw.release()
assert hiprt.hipStreamDestroy(stream) == 0
print("ok")
"""


def test_uploads_are_there_for_streams_the_library_does_not_know(hip):
    done = subprocess.run([sys.executable, "-c", OTHER_STREAM], cwd=ROOT, stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                          text=True, timeout=100)
    assert done.returncode == 0 and done.stdout.strip().endswith("ok"), done.stdout[-2000:]


def test_paths_of_a_program_without_streams(hip):
    done = subprocess.run([sys.executable, "-c", PROGRAM], cwd=ROOT, stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                          text=True, timeout=100)
    assert done.returncode == 0, done.stdout[-2000:]
    assert done.stdout.count("ok") == 19, done.stdout[-2000:]
