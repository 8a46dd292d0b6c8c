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
print("done")
"""


def test_memory_comes_round_again_on_the_null_stream(hip):
    res = subprocess.run([sys.executable, "-c", _NULL_STREAM_ONLY, ROOT], stdout=subprocess.PIPE,
                         stderr=subprocess.PIPE, text=True, timeout=110)
    assert res.returncode == 0 and res.stdout.strip().endswith("done"), res.stderr[-2000:]


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
