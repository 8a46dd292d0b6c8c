"""Device memory that is handed out again (vtl_hip_malloc / vtl_hip_free), on the null stream
in a process that names no other, and on streams of the caller's."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

from helpers import d2h, h2d
from vtl_amd import capi
from vtl_amd.tensor import HipTensor

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _malloc(nbytes):
    p = C.c_void_p()
    capi.call("vtl_hip_malloc", C.byref(p), nbytes)
    return p.value


_NULL_STREAM_ONLY = r"""
import ctypes as C, sys
import numpy as np
sys.path.insert(0, sys.argv[1])
from vtl_amd import capi
from vtl_amd.tensor import HipTensor
capi.call("vtl_hip_set_device", 0)
def malloc(n):
    p = C.c_void_p()
    capi.call("vtl_hip_malloc", C.byref(p), n)
    return p.value
# sizes around the edges of the size classes: what comes back is at least as large as asked, the
# block comes round again for the next request of its class, never while it is in use
for n in (1, 511, 512, 513, 4095, 4096, 4097, 65535, 65536, 73728, 73729, (1 << 20) + 1, (33 << 20) - 3):
    a, b = malloc(n), malloc(n)
    assert a and b and a != b and a % 256 == 0
    for p, v in ((a, 0x11), (b, 0x22)):
        capi.call("vtl_hip_memset", p, v, n)
    for p, v in ((a, 0x11), (b, 0x22)):
        got = np.empty(n, np.uint8)
        capi.call("vtl_hip_memcpy_d2h", got.ctypes.data, p, n)
        assert np.all(got == v), n
    capi.call("vtl_hip_free", a)
    assert capi.status("vtl_hip_free", a) == capi.ERR_RUNTIME      # released twice
    assert malloc(n) == a
    capi.call("vtl_hip_free", a)
    capi.call("vtl_hip_free", b)
# a block released behind a long kernel and taken at once: the kernel's input stays whole
rng = np.random.default_rng(5)
x = rng.standard_normal((2048, 4096), dtype=np.float32)
want = None
for i in range(8):
    t = HipTensor.from_host(x)
    q, s = t.quantize_i8(0)
    t.release()
    u = HipTensor.empty(x.shape, np.float32)      # the block of t, most likely
    capi.call("vtl_hip_memset", u.ptr, 0x7f, x.nbytes)
    got = q.cpu()
    want = got if want is None else want
    assert np.array_equal(got, want)
    for h in (q, s, u):
        h.release()
capi.call("vtl_hip_trim")
y = HipTensor.from_host(x)
assert np.array_equal(y.cpu(), x)
# uploads that nothing waits for, from memory that is overwritten at once, small and large in turn
import threading
bad = []
def rounds(seed):
    r = np.random.default_rng(seed)
    for i in range(12):
        src = r.integers(0, 255, [100, 70000, (1 << 20) + 5, 3 << 20][i % 4], dtype=np.uint8)
        keep = src.copy()
        t = HipTensor.from_host(src)
        src[:] = 0
        if not np.array_equal(t.cpu(), keep):
            bad.append((seed, i))
        t.release()
rounds(0)
threads = [threading.Thread(target=rounds, args=(k,)) for k in range(1, 5)]
for t in threads:
    t.start()
for t in threads:
    t.join()
assert not bad, bad
print("done")
"""


def test_memory_comes_round_again_on_the_null_stream(hip):
    res = subprocess.run([sys.executable, "-c", _NULL_STREAM_ONLY, ROOT], stdout=subprocess.PIPE,
                         stderr=subprocess.PIPE, text=True, timeout=110)
    assert res.returncode == 0 and res.stdout.strip().endswith("done"), res.stderr[-2000:]


# bytes: single ones, around a vector, where a result's array moves to pinned memory (128 KiB), some in between, where staging
# ends and chunks begin (1 MiB), where chunks have grown to a whole slot (from 3.75 MiB on), once round the ring of 8 slots of 4 MiB and a remainder
@pytest.mark.parametrize("nbytes", [1, 15, 16, 17, 4096, 131072, 131073, (384 << 10) - 1, 384 << 10, 700001, (1 << 20) - 1, 1 << 20, (1 << 20) + 1,
                                    (4 << 20) + 3, (16 << 20) + 4097, (36 << 20) + 13])
@pytest.mark.parametrize("offset", [0, 5])
def test_copies_to_and_from_the_device(hip, nbytes, offset):
    rng = np.random.default_rng(nbytes + offset)
    src = rng.integers(0, 256, nbytes, dtype=np.uint8)
    base = _malloc(nbytes + offset + 64)
    p = C.c_void_p()
    capi.call("vtl_hip_host_alloc", C.byref(p), nbytes + 64)
    pinned = np.frombuffer((C.c_uint8 * (nbytes + 64)).from_address(p.value), np.uint8)
    for up in ("vtl_hip_memcpy_h2d", "vtl_hip_upload"):
        capi.call("vtl_hip_memset", base, 0x5a, nbytes + offset + 64)
        given = src.copy()
        capi.call(up, base + offset, given.ctypes.data, nbytes)
        given[:] = 0
        back = d2h(base, nbytes + offset + 64, np.uint8)                    # memory of numpy's
        assert np.array_equal(back[offset:offset + nbytes], src)
        assert np.all(back[:offset] == 0x5a) and np.all(back[offset + nbytes:] == 0x5a)
        for skew in (offset, 0):                                            # pinned, in step and out of step
            pinned[:] = 0x33
            capi.call("vtl_hip_memcpy_d2h", p.value + skew, base + offset, nbytes)
            assert np.array_equal(pinned[skew:skew + nbytes], src)
            assert np.all(pinned[:skew] == 0x33) and np.all(pinned[skew + nbytes:] == 0x33)
    capi.call("vtl_hip_host_free", p)
    assert capi.status("vtl_hip_host_free", p) == capi.ERR_INVALID_ARG
    capi.call("vtl_hip_free", base)


def test_several_downloads_at_once(hip):
    """More results than one launch carries, empty ones, small and large ones among them."""
    rng = np.random.default_rng(9)
    arrays = [rng.standard_normal(n).astype(np.float32) for n in (3, 0, 300000, 1, 50000, 200000, 250000, 7, 600000)]
    ts = [HipTensor.from_host(a) for a in arrays]
    for got, a in zip(HipTensor.cpu_all(ts), arrays):
        assert np.array_equal(got, a)
    for t in ts:
        t.release()


def test_results_beyond_the_pinned_memory_are_ordinary_arrays(hip):
    """Kept results use up the pinned memory; the ones after that still arrive."""
    x = np.arange(40 << 20, dtype=np.float32)       # 160 MiB
    t = HipTensor.from_host(x)
    kept = [t.cpu() for _ in range(8)]
    assert all(np.array_equal(k, x) for k in kept)
    p = C.c_void_p()
    assert capi.status("vtl_hip_host_alloc", C.byref(p), 512 << 20) == capi.ERR_OUT_OF_MEMORY
    del kept
    capi.call("vtl_hip_host_alloc", C.byref(p), 512 << 20)
    capi.call("vtl_hip_host_free", p)
    t.release()


def test_release_waits_for_streams_of_the_caller(hip):
    """Memory that work on a non-blocking stream still reads is released and taken again by the null
    stream: the release waits, so the new owner's writes come after the reads."""
    hiprt = C.CDLL("libamdhip64.so")
    stream = C.c_void_p()
    assert hiprt.hipStreamCreateWithFlags(C.byref(stream), C.c_uint(1)) == 0
    rng = np.random.default_rng(6)
    x = rng.standard_normal((4096, 4096), dtype=np.float32)
    n = x.nbytes
    dst = _malloc(n)
    try:
        for _ in range(4):
            src = _malloc(n)
            h2d(src, x)
            capi.call("vtl_hip_set_stream", stream)
            for _ in range(4):
                capi.call("vtl_hip_memcpy_d2d", dst, src, n)
            capi.call("vtl_hip_free", src)
            capi.call("vtl_hip_set_stream", None)
            again = _malloc(n)
            capi.call("vtl_hip_memset", again, 0, n)
            capi.call("vtl_hip_sync")
            assert np.array_equal(d2h(dst, x.shape, np.float32), x)
            capi.call("vtl_hip_free", again)
    finally:
        capi.call("vtl_hip_set_stream", None)
        assert hiprt.hipStreamDestroy(stream) == 0
        capi.call("vtl_hip_free", dst)
        capi.call("vtl_hip_trim")
