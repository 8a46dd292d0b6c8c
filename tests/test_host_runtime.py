"""What the library enqueues where, without a GPU: each test runs a program of its own on a HIP runtime
that keeps count of devices, streams and memory and runs no kernel
(tests/host_runtime/fake_runtime.cpp)."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

_PRELUDE = r"""
import ctypes as C, sys
fake = C.CDLL(sys.argv[2], mode=C.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[1])
from vtl_amd import capi

def runtime(devices=1, capturing=False, refuse_memory=False, wait_ms=0):
    fake.fake_set(devices, int(capturing), int(refuse_memory), wait_ms)

def events():
    buf = C.create_string_buffer(1 << 20)
    n = fake.fake_log(buf, C.c_size_t(len(buf)))
    lines = [l.split() for l in buf.raw[:n].decode().splitlines()]
    return [(l[0], int(l[1]), int(l[2]), int(l[3])) for l in lines]

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
