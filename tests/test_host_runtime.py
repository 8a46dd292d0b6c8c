"""What the library enqueues where, without a GPU: each test runs a program of its own on a HIP runtime
that keeps count of devices, streams and memory and runs no kernel
(tests/host_runtime/fake_runtime.cpp)."""
import os
import subprocess
import sys

import numpy as np
import pytest

from vtl_amd import capi, layers
from vtl_amd.layers import PER_CHANNEL, PER_TENSOR, QuantizedWeights, QuantLinearLayer

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

_PRELUDE = r"""
import ctypes as C, sys
fake = C.CDLL(sys.argv[2], mode=C.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[1])
from vtl_amd import capi

def runtime(devices=1, capturing=False, refuse_memory=False, wait_ms=0):
    fake.fake_set(devices, int(capturing), int(refuse_memory), wait_ms)

def lines():
    buf = C.create_string_buffer(1 << 20)
    n = fake.fake_log(buf, C.c_size_t(len(buf)))
    return [l.split() for l in buf.raw[:n].decode().splitlines()]

def events():
    return [(l[0], int(l[1]), int(l[2]), int(l[3])) for l in lines()]

def count(what, log):
    return sum(1 for e in log if e[0] == what)

def malloc_on(device, nbytes):
    p = C.c_void_p()
    capi.call("vtl_hip_malloc_on", device, C.byref(p), nbytes)
    return p.value
"""


@pytest.fixture(scope="module")
def fake_runtime(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("runtime") / "libfake_runtime.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "host_runtime", "fake_runtime.cpp"), "-o", out], check=True)
    return out


def _run(fake, program):
    res = subprocess.run([sys.executable, "-c", _PRELUDE + program, ROOT, fake], stdout=subprocess.PIPE,
                         stderr=subprocess.STDOUT, text=True, timeout=100)
    assert res.returncode == 0 and res.stdout.strip().endswith("done"), res.stdout[-3000:]


_PRODUCTS = r"""
runtime()
p = malloc_on(0, 1 << 20)
def product(name, m, n, k):
    events()
    st = capi.status("vtl_hip_matmul_" + name, p, p, p, m, n, k, 0, 0)
    return st, events()
SHORT = [(64, 256, 784), (16, 256, 1024), (64, 256, 2000), (1, 33, 513), (32, 32, 2047)]
"""


def test_short_products_share_no_scratch_between_streams(fake_runtime):
    """Matmuls with K below 2048 need no memory of the library's once a stream has been named: one
    launch each, also while the stream records a graph that nothing has warmed up for."""
    _run(fake_runtime, _PRODUCTS + r"""
capi.call("vtl_hip_set_stream", 4096)
for capturing in (False, True):
    runtime(capturing=capturing)
    for name in ("f32", "f64"):
        for m, n, k in SHORT:
            st, log = product(name, m, n, k)
            assert st == capi.OK, (capturing, name, m, n, k, st)
            assert [e[0] for e in log] == ["launch"] and log[0][2] == 4096, (capturing, name, m, n, k, log)
print("done")
""")


def test_products_in_slices_without_memory_run_in_one_piece(fake_runtime):
    """Where K would be cut and there is no memory for the partial sums, or a capture forbids to get
    it, the product runs unsliced."""
    _run(fake_runtime, _PRODUCTS + r"""
for name in ("f32", "f64"):
    st, log = product(name, 64, 256, 784)
    assert st == capi.OK and count("launch", log) == 2, log      # slices and their sum
capi.call("vtl_hip_trim")
runtime(refuse_memory=True)
for name in ("f32", "f64"):
    for m, n, k in SHORT + [(64, 64, 4096)]:
        st, log = product(name, m, n, k)
        assert st == capi.OK and count("launch", log) == 1, (name, m, n, k, st, log)
runtime(capturing=True)
capi.call("vtl_hip_set_stream", 4096)
for name in ("f32", "f64"):
    st, log = product(name, 64, 64, 4096)
    assert st == capi.OK and [e[0] for e in log] == ["launch"], (name, st, log)
print("done")
""")


def test_long_products_take_vector_loads(fake_runtime):
    """Only rows too long for a lane's 32-bit offset are loaded element by element: how many rows there are, or how long K is
    where it runs across them, does not matter (a forward over five million rows, its dW)."""
    _run(fake_runtime, _PRODUCTS + r"""
import re
def checked(name, m, n, k, ta, tb):
    events()
    assert capi.status("vtl_hip_matmul_" + name, p, p, p, m, n, k, ta, tb) == capi.OK     # no kernel runs here
    flags = [re.search(r"direct_kernelI\wLi.*?Lb(\d)ELb(\d)ELb(\d)E", l[4]) for l in lines() if l[0] == "launch"]
    flags = [f.groups() for f in flags if f]
    assert len(flags) == 1 and flags[0][:2] == (str(ta), str(tb)), flags
    return flags[0][2] == "1"
MANY = 5000000
for name, size in (("f32", 4), ("f64", 8)):
    along, across = ((1 << 32) - 1) // (64 * size), ((1 << 32) - 1) // (16 * size)
    for case in [(MANY, 64, 64, 0, 1), (MANY, 64, 64, 0, 0), (64, 64, MANY, 1, 0), (64, MANY, 64, 0, 1), (MANY, 7, 5, 1, 0), (5, MANY, 64, 0, 0),
                 (64, 64, MANY, 0, 0), (64, 64, along, 0, 1), (across, 3, 5, 1, 0), (3, across, 5, 0, 0), (64, 64, 1 << 28, 1, 0)]:
        assert not checked(name, *case), (name, case)
    for case in [(64, 64, along + 1, 0, 1), (64, 64, along + 1, 0, 0), (64, 64, along + 1, 1, 1), (across + 1, 3, 5, 1, 0),
                 (3, across + 1, 5, 0, 0), (1, 64, 64, 1, 0), (64, 1, 64, 0, 0)]:
        assert checked(name, *case), (name, case)
print("done")
""")


def test_copies_run_where_the_memory_is(fake_runtime):
    """Memory of device 0 is copied after something was allocated on device 1: the kernel that carries the
    bytes runs on device 0, and device 1 is current again afterwards.  On a stream of the caller's the copy is
    the runtime's, which takes memory of any device."""
    _run(fake_runtime, r"""
runtime(devices=2)
BIG = 3 << 20
p = malloc_on(0, BIG + 4096)
q = malloc_on(1, BIG + 4096)
host = C.create_string_buffer(BIG)
def here():
    d = C.c_int(-1)
    fake.hipGetDevice(C.byref(d))
    return d.value
def downloads(*device):
    n = len(device)
    return "vtl_hip_download", (n, (C.c_void_p * n)(*[C.addressof(host)] * n), (C.c_void_p * n)(*device), (C.c_size_t * n)(*[4096] * n))
for size in (100, 4096, BIG):
    for name, args in (("vtl_hip_memcpy_h2d", (p + 5, host, size)), ("vtl_hip_upload", (p + 5, host, size)),
                       ("vtl_hip_memcpy_d2h", (host, p + 5, size)), ("vtl_hip_memcpy_d2d", (p, p + 2048, 1024)),
                       downloads(p + 64, p)):
        events()
        capi.status(name, *args)      # no kernel runs here, so whoever waits for one reports that
        log = [e for e in events() if e[0] in ("launch", "copy")]
        assert log and all(e[1] == 0 for e in log), (name, size, log)
        assert here() == 1, name
# of both devices in one call, each on its own
events()
name, args = downloads(q, p)
args[3][0] = 0
capi.status(name, *args)
assert {e[1] for e in events() if e[0] == "launch"} == {0}
# device to device between the two: no kernel
events()
capi.call("vtl_hip_memcpy_d2d", q, p, 4096)
assert [e[0] for e in events()] == ["copy"]
capi.call("vtl_hip_set_stream", 4096)
for name, args in (("vtl_hip_memcpy_h2d", (p, host, 4096)), ("vtl_hip_upload", (p, host, BIG)),
                   ("vtl_hip_memcpy_d2h", (host, p, BIG)), downloads(p, q)):
    events()
    capi.status(name, *args)
    log = [e for e in events() if e[0] in ("launch", "copy")]
    assert log and log[0][0] == "copy" and log[0][2] == 4096, (name, log)
    assert here() == 1, name
print("done")
""")


def test_tensors_from_the_host_are_there_on_return(fake_runtime):
    """HipStorage.from_cpu waits for what it enqueued, so that work on streams the library knows
    nothing of finds the bytes."""
    _run(fake_runtime, r"""
import numpy as np
from vtl_amd.storage import HipStorage
runtime()
def waited(log):
    enqueued = max(i for i, e in enumerate(log) if e[0] in ("launch", "copy"))
    return any(e[0] in ("sync", "device_sync") for e in log[enqueued:])
def run(f, *args, **kw):
    events()
    try:
        f(*args, **kw)
    except capi.VtlHipError:      # the wait for a kernel that no one runs
        pass
    return events()
for nbytes in (1, 4096, 1 << 20, (1 << 20) + 1, 5 << 20):
    assert waited(run(HipStorage.from_cpu, np.zeros(nbytes, np.uint8))), nbytes
print("done")
""")


def test_gradients_in_the_memory_of_w_wait_for_its_upload(fake_runtime):
    """The backward from host to host lets launches write dW and db to the host while it still has W to copy: never to
    memory that W lies in (dW is all of it, or db its last row)."""
    _run(fake_runtime, r"""
runtime()
M, N, K = 64, 2048, 64
NK = N * K
arena = C.c_void_p()
capi.call("vtl_hip_host_alloc", C.byref(arena), 4 * (NK + N) + 8192)
host = (C.c_float * (M * (N + K) + NK))()
grad, x, other = C.addressof(host), C.addressof(host) + 4 * M * N, C.addressof(host) + 4 * M * (N + K)
w = arena.value + 4096
def written(dx, dw, db):
    events()
    capi.status("vtl_hip_linear_backward_host_f32", grad, x, w, dx, dw, db, M, N, K)    # no kernel runs here
    return [int(l[5]) for l in lines() if len(l) > 5]
W = range(w, w + 4 * NK)
assert written(None, w, None) == [w]                     # W is not read at all
for dw, db in ((w, None), (w - 4096, None), (w + 4 * 1024, None), (None, w), (None, w + 4 * (NK - N)), (w, w + 4 * NK)):
    early = written(other, dw, db)[:-1]                  # all but dX, which comes behind the upload
    assert len(early) == (dw is not None) + (db is not None), (dw, db, early)
    assert not any(p in W for p in early), (dw, db, early)
assert w + 4 * NK in written(other, w, w + 4 * NK)       # behind W: straight to the host
print("done")
""")


def test_a_call_that_fails_keeps_no_memory(fake_runtime):
    """Whole host calls that end in an error between their first step and their last, whichever it is: the pinned memory that
    the result was to come through, and the device memory, serve the next call."""
    _run(fake_runtime, r"""
runtime()
p = malloc_on(0, 1 << 20)
host = (C.c_float * 65536)()
def forward(rows, row_bytes):
    layer = capi.Layer(0, 1, 64, 100, p, p, None, row_bytes)      # a linear, one scale per row
    return capi.status("vtl_hip_forward_i8_host", host, rows, 100, C.byref(layer), 1, host)
for rows in (1, 16, 64):
    for again in range(4):
        events()
        assert forward(rows, 100) == capi.ERR_INVALID_ARG       # rows of a layer are padded to whole 16 bytes
        log = events()
        assert again == 0 or not count("host_malloc", log) + count("malloc", log), (rows, again, log)
runtime(refuse_memory=True)
capi.call("vtl_hip_trim")
for again in range(4):      # device memory runs out behind the lease of what results come through
    events()
    assert capi.status("vtl_hip_linear_backward_host_f32", host, host, host, host, host, host, 64, 64, 64) == capi.ERR_OUT_OF_MEMORY
    assert not count("host_malloc", events()), again
print("done")
""")


def test_whole_host_calls_share_no_scratch_between_threads(fake_runtime):
    """Whole host calls run in several threads at once: what two of their launches meet in is memory of the call's own, not
    the library's one buffer per purpose (32 MiB at least, where these calls take a few)."""
    _run(fake_runtime, r"""
runtime()
p = malloc_on(0, 1 << 20)
host = (C.c_float * (1 << 20))()
def shared(name, *args):
    events()
    capi.status(name, *args)                                                  # no kernel runs here
    log = events()
    assert count("launch", log) > 1, (name, args, log)
    return [e for e in log if e[0] == "malloc" and e[3] >= 32 << 20]
for per_channel in (0, 1):
    for rows, n, k, row in ((256, 1000, 72, 80), (256, 1000, 72, 0), (64, 1000, 1001, 1008), (64, 1024, 4096, 0)):
        layer = capi.Layer(0, per_channel, n, k, p, p, None, row)             # a linear
        assert not shared("vtl_hip_forward_i8_host", host, rows, k, C.byref(layer), 1, host), (per_channel, rows, n, k)
for name in ("f32", "f64"):
    backward = "vtl_hip_linear_backward_host_" + name
    assert not shared(backward, host, host, host, host, host, host, 256, 64, 16), name    # gradients in one launch
    assert not shared(backward, host, host, host, host, host, host, 2048, 64, 16), name   # column sums in splits
    capi.status(backward, host, host, host, host, host, host, 2048, 64, 16)
    assert any("colsum_finalize_kernel" in l[4] for l in lines() if l[0] == "launch"), name
print("done")
""")


def test_a_small_backward_on_a_stream_of_its_own_waits_for_no_other(fake_runtime):
    """Once a stream has been named a release waits for the whole device: a backward from host to host releases nothing while it
    still has something to launch."""
    _run(fake_runtime, r"""
runtime()
host, dx, dw, db = [(C.c_float * 65536)() for _ in range(4)]
capi.call("vtl_hip_set_stream", 4096)
for name in ("f32", "f64"):
    for m, n, k in ((16, 24, 40), (64, 64, 64), (600, 16, 16)):
        for want_db in (db, None):
            events()
            capi.status("vtl_hip_linear_backward_host_" + name, host, host, host, dx, dw, want_db, m, n, k)    # no kernel runs here
            log = [e[0] for e in events()]
            last = max(i for i, e in enumerate(log) if e == "launch")
            assert "device_sync" not in log[:last], (name, m, n, k, log)
print("done")
""")


def test_a_forward_on_a_stream_of_its_own_waits_for_no_other(fake_runtime):
    """Nor does a forward from host to host whose results are flagged by a launch of their own."""
    _run(fake_runtime, r"""
runtime()
p = malloc_on(0, 8 << 20)
host, y = (C.c_float * (1 << 16))(), (C.c_float * (1 << 16))()
capi.call("vtl_hip_set_stream", 4096)
for per_channel in (0, 1):
    for rows, n, k in ((1, 3358, 150), (1, 3358, 160), (1, 64, 64), (2, 3271, 50), (8, 3000, 512)):
        for row in (0, (k + 15) // 16 * 16):
            layer = capi.Layer(0, per_channel, n, k, p, p, None, row)
            events()
            capi.status("vtl_hip_forward_i8_host", host, rows, k, C.byref(layer), 1, y)    # no kernel runs here
            log = [e[0] for e in events()]
            last = max(i for i, e in enumerate(log) if e == "launch")
            assert "device_sync" not in log[:last], (per_channel, rows, n, k, row, log)
print("done")
""")


def test_column_sums_within_their_input_come_behind_all_of_it(fake_runtime):
    """Sums that are written into the tensor they are made from, from 128 rows on: by a launch behind the one that reads it, for other
    workgroups still read what one has summed."""
    _run(fake_runtime, r"""
runtime()
p = malloc_on(0, 8 << 20)
def kernels(name, *args):
    events()
    assert capi.status(name, *args) == capi.OK
    return [k for l in lines() if l[0] == "launch" for k in ("colsum_finalize", "13colsum_kernel", "colsum_short") if k in l[4]]
for name, size in (("f32", 4), ("f64", 8)):
    for rows, cols in ((128, 700), (300, 64), (512, 129)):
        for out in (p + 5 * size, p + size * (rows * cols - 1), p + size * 3 * cols):
            assert kernels("vtl_hip_colsum_" + name, p, rows, cols, out) == ["13colsum_kernel", "colsum_finalize"], (name, rows, cols, out - p)
            x, w, dx, dw = (p + (i << 20) for i in range(2, 6))
            got = kernels("vtl_hip_linear_backward_" + name, p, x, w, dx, dw, out, rows, cols, 16)
            assert got == ["13colsum_kernel", "colsum_finalize"], (name, rows, cols, out - p)
        assert kernels("vtl_hip_colsum_" + name, p, rows, cols, p + size * rows * cols) == ["colsum_short"]     # behind it
print("done")
""")


def test_results_over_what_they_are_made_from_come_behind_the_quantizer(fake_runtime):
    """A quantized linear whose Y lies over X, or over the weights, is not made by tiles that read their rows while others are stored."""
    _run(fake_runtime, r"""
import re
runtime()
p = malloc_on(0, 16 << 20)
far = p + (8 << 20)
def kernels(x, y, m, n, k, row=0, w=p + (4 << 20)):
    events()
    layer = capi.Layer(0, 1, n, k, w, far, None, row)
    st = capi.status("vtl_hip_layer_f32", C.byref(layer), x, y, m, 0, None, 0)
    found = [re.search("linear_small|linear_gemv|quantize|gemm_i8_small", l[4]) for l in lines() if l[0] == "launch"]
    return [f.group() for f in found if f]
for m, n, k, row in ((64, 256, 256, 0), (33, 1000, 512, 0), (64, 128, 500, 512), (20, 100, 256, 0)):
    assert kernels(p, far, m, n, k, row) == ["linear_small"]
    ends = p + 4 * m * k
    for y in (p, p + 16, ends - 4, p + 64):
        assert kernels(p, y, m, n, k, row)[0] == "quantize", (m, n, k, y - p)
        assert kernels(y, p + 16, m, n, k, row)[0] == ("quantize" if p + 16 + 4 * m * n > y else "linear_small"), (m, n, k, y - p)
    assert kernels(p, ends, m, n, k, row) == ["linear_small"]                     # behind it
    assert kernels(p, p + (4 << 20) + 16, m, n, k, row)[0] == "quantize"
assert kernels(p, far, 8, 14336, 256) == ["linear_small"] and kernels(p, p, 8, 14336, 256, w=p + (1 << 20)) == ["linear_gemv"]
print("done")
""")


def test_products_over_their_operands_come_behind_all_of_them(fake_runtime):
    """Slices of K meet within their launch only where C is memory of its own: elsewhere a launch behind it adds them up."""
    _run(fake_runtime, r"""
runtime()
p = malloc_on(0, 32 << 20)
far = p + (16 << 20)
def launches(name, *args):
    events()
    assert capi.status(name, *args) == capi.OK
    return count("launch", events())
for name, size in (("f32", 4), ("f64", 8)):
    for m, n, k in ((64, 256, 2000), (64, 64, 4096), (32, 1024, 1024)):
        a, b = p, p + m * k * size
        end = b + n * k * size
        assert launches("vtl_hip_matmul_" + name, a, b, far, m, n, k, 0, 0) == 1, (name, m, n, k)
        assert launches("vtl_hip_matmul_" + name, a, b, end, m, n, k, 0, 1) == 1
        for c in (a, a + 4 * size, b - size, b, end - size):
            assert launches("vtl_hip_matmul_" + name, a, b, c, m, n, k, 0, 0) == 2, (name, m, n, k, c - p)
            assert launches("vtl_hip_linear_" + name, a, b, None, c, m, n, k, 0) == 2, (name, m, n, k, c - p)
print("done")
""")


def test_int8_products_over_their_operands_come_behind_all_of_them(fake_runtime):
    """Small int8 products whose K the tile kernels cut: with the results over an operand they are cut, and added up behind it."""
    _run(fake_runtime, r"""
import re
runtime()
p = malloc_on(0, 32 << 20)
far = p + (16 << 20)
def kernels(name, *args):
    events()
    assert capi.status(name, *args) == capi.OK
    found = [re.search("gemm_i8_small|gemm_i8|finalize", l[4]) for l in lines() if l[0] == "launch"]
    return [f.group() for f in found if f]
for m, n, k in ((100, 500, 3312), (64, 640, 3312)):
    a, b = p, p + m * k
    for y, want in ((far, ["gemm_i8_small"]), (b + n * k, ["gemm_i8_small"]), (a, ["gemm_i8", "finalize"]), (b - 16, ["gemm_i8", "finalize"]),
                    (b + n * k - 16, ["gemm_i8", "finalize"])):
        assert kernels("vtl_hip_linear_i8_f32", a, far + (8 << 20), 1, b, far + (9 << 20), 1, None, y, m, n, k, 0) == want, (m, n, k, y - p)
        assert kernels("vtl_hip_gemm_i8_i32", a, b, y, m, n, k) == want, (m, n, k, y - p)
print("done")
""")


def test_where_gradients_share_a_launch(fake_runtime):
    """Not where dW is few rows of millions of values, or large enough for shapes of its own."""
    _run(fake_runtime, r"""
runtime()
p = [malloc_on(0, 1 << 20) + (i << 36) for i in range(6)]             # (no kernel runs here)
def in_one(name, m, n, k, dx, db):
    events()
    assert capi.status("vtl_hip_linear_backward_" + name, p[0], p[1], p[2], p[3] if dx else None, p[4], p[5] if db else None, m, n, k) == capi.OK
    found = [l[4] for l in lines() if l[0] == "launch"]
    return "linear_backward" in found[0]                              # (and what adds up slices behind it)
for name, m, n, k, dx, db in (("f32", 64, 256, 640, 1, 1), ("f32", 192, 832, 832, 1, 1), ("f64", 13, 664, 2861, 1, 0), ("f32", 3, 742, 1465, 1, 1), ("f64", 13, 4511, 120, 0, 1)):
    assert in_one(name, m, n, k, dx, db), (name, m, n, k)
for name, m, n, k, dx, db in (("f32", 9, 1899, 2356, 1, 1), ("f64", 7, 927, 4509, 0, 1), ("f32", 2, 1072, 1284, 1, 0), ("f32", 31, 1870, 1608, 1, 1), ("f32", 256, 11008, 4096, 1, 1),
                              ("f64", 442, 6, 3774, 1, 0), ("f32", 88, 1150, 4098, 0, 1), ("f64", 15, 1993, 769, 0, 1)):
    assert not in_one(name, m, n, k, dx, db), (name, m, n, k)
print("done")
""")


def test_small_uploads_share_a_launch_with_little_else(fake_runtime):
    _run(fake_runtime, r"""
runtime()
host = (C.c_float * (1 << 19))()
def launches(*sizes):
    p = [malloc_on(0, n) for n in sizes]
    events()
    assert capi.status("vtl_hip_upload_two", p[0], host, sizes[0], p[1], host, sizes[1]) == capi.OK
    found = [l[4] for l in lines() if l[0] == "launch"]
    assert all("host_copy" in k or "clear_counters" in k for k in found), found
    return sum("host_copy" in k for k in found)
launches(16, 16)
for a, b, n in ((4, 4, 1), (320 << 10, 321 << 10, 2), (2048, 1 << 20, 1), (1 << 20, 64 << 10, 1), (1 << 20, 65 << 10, 2)):    # (a slot's 4 MiB in all)
    assert launches(a, b) == n, (a, b)
print("done")
""")


def test_where_column_sums_take_one_launch(fake_runtime):
    _run(fake_runtime, r"""
runtime()
p = malloc_on(0, 1 << 20)
out = p + (1 << 36)                    # (no kernel runs here)
def kernels(name, rows, cols, off=0):
    events()
    assert capi.status("vtl_hip_colsum_" + name, p + off, rows, cols, out) == capi.OK
    return [k for l in lines() if l[0] == "launch" for k in ("colsum_finalize", "13colsum_kernel", "colsum_short") if k in l[4]]
for name in ("f32", "f64"):
    for rows, cols in ((0, 5), (1, 1), (512, 1), (512, 32768), (127, 32767)):
        assert kernels(name, rows, cols) == ["colsum_short"], (name, rows, cols)
    assert kernels(name, 127, 100003) == kernels(name, 256, 32771) == ["13colsum_kernel"]         # nothing to split
    assert kernels(name, 513, 64) == ["13colsum_kernel", "colsum_finalize"], name
assert kernels("f32", 320, 65536) == kernels("f32", 96, 65536) == ["colsum_short"]
assert kernels("f64", 320, 65536) == ["13colsum_kernel", "colsum_finalize"] and kernels("f64", 96, 65536) == ["13colsum_kernel"]
assert kernels("f32", 96, 65536, 4) == ["13colsum_kernel"]                    # rows that start anywhere
print("done")
""")


def test_small_host_calls_take_the_launches_they_are_to(fake_runtime):
    """While the process uses the null stream alone: a small backward is one upload and one launch, one row through a layer with one scale
    is one launch that reads it over the link, and large weights are quantized as they arrive."""
    _run(fake_runtime, r"""
import re
runtime()
p = malloc_on(0, 64 << 20)
host, dx, dw, db = [(C.c_float * (1 << 20))() for _ in range(4)]
def kernels(name, *args):
    events()
    capi.status(name, *args)                                                  # no kernel runs here
    found = [re.search("host_copy|upload_rows|linear_backward|f64acc_direct|linear_gemv|quantize", l[4]) for l in lines() if l[0] == "launch"]
    names = [f.group() for f in found if f]
    return [n for i, n in enumerate(names) if i == 0 or n != names[i - 1]]    # (a launch's gradients are noted one by one)
one = ["host_copy", "linear_backward"]
for name, fits, beyond in (("f32", (64, 345, 346), (64, 346, 346)), ("f64", (64, 229, 229), (64, 230, 230))):
    backward = "vtl_hip_linear_backward_host_" + name
    assert kernels(backward, host, host, host, dx, dw, db, 64, 64, 64) == one
    assert kernels(backward, host, host, host, dx, dw, db, *fits) == one
    got = kernels(backward, host, host, host, dx, dw, db, *beyond)
    assert got[0] == "host_copy" and "host_copy" in got[2:] and got[-1] != "linear_backward", got
layer = capi.Layer(0, 0, 64, 784, p, p, None, 0)                              # one scale
assert kernels("vtl_hip_forward_i8_host", host, 1, 784, C.byref(layer), 1, host) == ["linear_gemv"]
# that where every workgroup's reading of the row is not the longer, else it is quantized by a launch of its own (uploaded, 20 to 32 KB, for neither)
for n, k, want in ((5500, 4096, 1), (17, 5120, 0), (16, 5120, 1), (17, 5136, 0), (1, 8192, 0), (16, 8208, 1), (17, 8208, 0), (64, 14336, 0), (64, 4999, 1),
                   (4000, 11001, 1), (33, 11017, 0), (32, 14001, 1), (4000, 6001, 2)):
    layer = capi.Layer(0, 0, n, k, p, p, None, 0)
    got = kernels("vtl_hip_forward_i8_host", host, 1, k, C.byref(layer), 1, host)
    assert got[:max(want, 1)] == [["quantize"], ["linear_gemv"], ["host_copy", "linear_gemv"]][want], (n, k, got)
layers = (capi.Layer * 2)(capi.Layer(0, 0, 10000, 16, p, p, None, 0), capi.Layer(0, 0, 64, 10000, p, p, None, 0))
assert kernels("vtl_hip_forward_i8_host", host, 1, 16, layers, 2, host) == ["linear_gemv"]      # twice: the second row is on the device
rows = (C.c_float * (9 << 20))()
got = [kernels("vtl_hip_upload_quantized", rows, n, k, 1, p, p, None, None, 0) for n, k in ((4200, 2044), (4096, 2048))]
assert "upload_rows" not in got[0] and got[1] == ["upload_rows"], got        # (in short rows too little would be on its way)
print("done")
""")


def test_narrow_weight_gradients_have_a_launch_of_their_own(fake_runtime):
    """Many rows of a few bytes, which a launch that writes over the link as it computes would send one by one."""
    _run(fake_runtime, r"""
runtime()
host, dx, dw, db = [(C.c_float * (1 << 20))() for _ in range(4)]
def in_one(name, m, n, k):
    events()
    capi.status("vtl_hip_linear_backward_host_" + name, host, host, host, dx, dw, db, m, n, k)    # no kernel runs here
    return not any("f64acc_direct" in l[4] for l in lines() if l[0] == "launch")                 # that of dX
for name, m, n, k in (("f32", 5, 48, 3), ("f32", 5, 128, 4), ("f32", 5, 400, 9), ("f32", 5, 1024, 8), ("f32", 3, 1024, 17), ("f32", 3, 2048, 33),
                      ("f64", 5, 128, 2), ("f64", 5, 1024, 4), ("f64", 3, 400, 5), ("f64", 3, 1024, 7), ("f64", 3, 2048, 16)):
    assert in_one(name, m, n, k), (name, m, n, k)
for name, m, n, k in (("f32", 5, 49, 2), ("f32", 10, 778, 2), ("f32", 64, 1500, 5), ("f32", 5, 129, 6), ("f32", 5, 401, 10), ("f32", 3, 1025, 16),
                      ("f32", 3, 2049, 40), ("f64", 10, 778, 3), ("f64", 3, 2000, 4), ("f64", 3, 401, 5), ("f64", 3, 2049, 16)):
    assert not in_one(name, m, n, k), (name, m, n, k)
print("done")
""")


_SHORT_ROWS = r"""
import re
runtime()
p = malloc_on(0, 64 << 20)
host = (C.c_float * (1 << 20))()
def in_one(name, *args):
    events()
    assert capi.status(name, *args) == capi.OK, args
    kernels = [l[4] for l in lines() if l[0] == "launch"]
    return len(kernels) == 1 and "linear_gemv" in kernels[0]
def dense(m, n, k):
    return in_one("vtl_hip_linear_f32_dynquant", p, p, p, None, p, m, n, k, 0, None, 0)
def padded(m, n, k):
    return in_one("vtl_hip_layer_f32", C.byref(capi.Layer(0, 1, n, k, p, p, None, (k + 15) & ~15)), p, p, m, 0, None, 0)
"""


def test_where_short_rows_are_quantized(fake_runtime):
    """A few rows of fewer than 256 codes that start anywhere: in the launch of the product where that is the faster form for this many
    rows, weights and the memory they lie in."""
    _run(fake_runtime, _SHORT_ROWS + r"""
for m, n in ((1, 14336), (2, 16384), (3, 8192), (4, 8192), (5, 2048), (8, 2048), (8, 1)):
    for k in (17, 100, 239):
        assert dense(m, n, k) and padded(m, n, k), (m, n, k)
for m, n in ((2, 16385), (3, 8193), (4, 16384), (5, 2049), (6, 14336), (8, 16384)):
    for k in (17, 100):
        assert not dense(m, n, k) and not padded(m, n, k), (m, n, k)
# weights that a call in two launches pads: three
for m, n, k, one in ((1, 100000, 100, 1), (2, 40000, 100, 1), (2, 25000, 200, 1), (4, 40000, 100, 1), (4, 60000, 200, 1), (4, 60000, 100, 0),
                     (6, 17000, 200, 0)):
    assert dense(m, n, k) == bool(one), (m, n, k)
assert padded(1, 65536, 100) and not padded(1, 80000, 100)
for k in (15, 16, 240):                                        # too short, or whole rows
    assert not dense(8, 64, k), k
# where the rows lie, not which entry point: the first layer reads them over the link, the second has them in device memory, the
# last one's results go over the link
def forward(rows, *dims):
    layers = (capi.Layer * (len(dims) - 1))(*[capi.Layer(0, 1, n, k, p, p, None, 0) for k, n in zip(dims, dims[1:])])
    events()
    capi.status("vtl_hip_forward_i8_host", host, rows, dims[0], layers, len(dims) - 1, host)     # no kernel runs here
    found = [re.search("linear_gemv|quantize", l[4]) for l in lines() if l[0] == "launch"]
    return [f.group() for f in found if f]
assert forward(2, 100, 200, 300, 64) == ["linear_gemv"] * 3
assert forward(1, 100, 20000) == ["quantize"]
assert forward(4, 100, 200, 250, 64) == ["quantize", "linear_gemv", "quantize"]
print("done")
""")


def test_a_kernel_that_is_asked_for_is_the_one(fake_runtime):
    """The switches that name a kernel for a few rows, or for more, come before the rule for rows that each tile quantizes."""
    _run(fake_runtime, r"""
import os, re
runtime()
p = malloc_on(0, 64 << 20)
def kernels(m, n, k, **knobs):
    os.environ.update(knobs)
    capi.call("vtl_hip_reload_env")
    for name in knobs:
        del os.environ[name]
    events()
    capi.status("vtl_hip_linear_f32_dynquant", p, p + (16 << 20), p, None, p + (32 << 20), m, n, k, 0, None, 0)
    found = [re.search("linear_small|linear_gemv_rows|quantize|skinny|streamk|gemm_i8", l[4]) for l in lines() if l[0] == "launch"]
    return [f.group() for f in found if f]
for m, n, k in ((8, 4000, 512), (8, 8192, 512), (5, 600, 256), (3, 4000, 256), (8, 14336, 256)):
    assert kernels(m, n, k) == ["linear_small"], (m, n, k)
    assert kernels(m, n, k, VTL_HIP_GEMV_ROWS="1") == ["linear_gemv_rows"], (m, n, k)
    got = kernels(m, n, k, VTL_HIP_GEMV_ROWS="0")
    assert "linear_gemv_rows" not in got and "linear_small" not in got, (m, n, k, got)
for m, n, k in ((64, 256, 512), (33, 1000, 256)):
    assert kernels(m, n, k) == kernels(m, n, k, VTL_HIP_GEMV_ROWS="1") == ["linear_small"], (m, n, k)
    assert kernels(m, n, k, VTL_HIP_SKINNY_TILED="1") == ["quantize", "skinny"], (m, n, k)
print("done")
""")


def test_short_rows_are_not_refused_for_want_of_scratch(fake_runtime):
    """Where a call that would take two launches may not allocate, the launch that needs no scratch serves."""
    _run(fake_runtime, _SHORT_ROWS + r"""
capi.call("vtl_hip_set_stream", 4096)
runtime(capturing=True)
for m, n, k in ((2, 20000, 100), (4, 9000, 239), (4, 60000, 100), (8, 8000, 239)):
    assert dense(m, n, k), (m, n, k)
for m, n, k in ((1, 80000, 100), (2, 20000, 100)):
    assert padded(m, n, k), (m, n, k)
# the caller's workspace, and none for padded weights
events()
assert capi.status("vtl_hip_linear_f32_dynquant", p, p, p, None, p, 4, 60000, 100, 0, p, 1 << 20) == capi.OK
assert "linear_gemv" in lines()[-1][4]
print("done")
""")


def test_a_transfer_that_waits_for_the_device_costs_no_host_time(fake_runtime):
    """A large upload whose staging memory is not free yet: neither the caller nor the threads that help
    with the copying spin until it is."""
    _run(fake_runtime, r"""
import time
import numpy as np
runtime(wait_ms=600)
p = malloc_on(0, 64 << 20)
src = np.zeros(64 << 20, np.uint8)
src += 1
runtime()                                      # what is made on first use does not wait
small = np.zeros(4, np.uint8)
capi.call("vtl_hip_upload", p, small.ctypes.data, 4)
runtime(wait_ms=600)
cpu, wall = time.process_time(), time.monotonic()
st = capi.status("vtl_hip_upload", p, src.ctypes.data, src.nbytes)
cpu, wall = time.process_time() - cpu, time.monotonic() - wall
assert st == capi.ERR_RUNTIME and wall > 0.6   # no kernel ever frees a slot here
assert cpu < 0.25, (cpu, wall)
print("done")
""")


@pytest.mark.parametrize("mode", [PER_CHANNEL, PER_TENSOR])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("cols", [1024, 1023])
def test_int8_parameters_are_there_on_return(monkeypatch, cols, bias, mode):
    """The last of the calls that make a layer's codes waits for all of them; a forward from host to host leaves
    that to its own end."""
    calls = []

    def call(name, *args):
        calls.append(name)
        if name == "vtl_hip_content_fingerprint":     # no device needed
            assert capi.status(name, *args) == capi.OK

    monkeypatch.setattr(capi, "call", call)
    w, b = np.ones((300, cols), np.float32), np.zeros(300, np.float32) if bias else None
    QuantizedWeights(w, b, mode)
    assert "vtl_hip_quantize_f32_i8" in calls and ("vtl_hip_pad_rows_i8" in calls) == (cols % 16 != 0)
    assert calls[-1] == "vtl_hip_sync", calls
    calls.clear()
    layer = QuantLinearLayer(w, b, mode, requires_grad=False)
    layer.forward(np.zeros((4, cols), np.float32))
    assert calls[-1] == "vtl_hip_forward_i8_host" and "vtl_hip_sync" not in calls
    calls.clear()
    layer.quantized()
    assert "vtl_hip_sync" not in calls                 # the forward has waited
    layer.invalidate()
    calls.clear()
    monkeypatch.setattr(layers, "forward_host", lambda *a: calls.append("failed") or 1 / 0)
    with pytest.raises(ZeroDivisionError):
        layer.forward(np.zeros((4, cols), np.float32))
    del calls[:calls.index("failed") + 1]
    layer.quantized()
    assert calls == ["vtl_hip_sync"]                   # no copies a second time, but the wait
