"""The host's quantizer makes the codes and scales that the oracle does, bit for bit, and which calls take it."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import oracle
from test_host_runtime import _run, fake_runtime  # noqa: F401

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vtl_amd", "csrc")

_WRAPPER = r"""
#include "host_quant.hip"
using namespace vtlhip;
extern "C" int quantize(int wide, const float *x, long rows, long cols, int per_row, int8_t *q, long row, float *scales, unsigned csr)
{
    const HostQuantizer *h = host_quantizer();
    if (!h || (wide && h != &kAvx512))
        return 0;
    h = wide ? &kAvx512 : &kAvx2;
    const unsigned before = _mm_getcsr();
    _mm_setcsr(csr);
    if (per_row) {
        h->rows(x, rows, cols, q, row, scales);
    } else {
        scales[0] = h->scale(h->absmax(x, rows * cols));
        h->scaled(x, rows, cols, q, row, scales[0]);
    }
    const int kept = _mm_getcsr() == csr;
    _mm_setcsr(before);
    return kept ? 1 : -1;
}
"""


@pytest.fixture(scope="module")
def quantizer(tmp_path_factory):
    d = tmp_path_factory.mktemp("host_quant")
    (d / "q.cpp").write_text(_WRAPPER)
    subprocess.run(["g++", "-std=c++17", "-O3", "-ffp-contract=off", "-fPIC", "-shared", "-I", CSRC, str(d / "q.cpp"), "-o", str(d / "q.so")],
                   check=True)
    return C.CDLL(str(d / "q.so")).quantize


def rows_to_try(rows, cols):
    """Magnitudes from subnormal to the largest, rows of zeros, quotients at and beside ties, NaNs and infinities."""
    rng = np.random.default_rng(rows * 7919 + cols)
    x = rng.standard_normal((rows, cols)).astype(np.float32)
    for r in range(rows):
        kind = r % 9
        if kind == 1:
            x[r] = 0.0
        elif kind == 2:                                    # ties: the largest is 127, so the scale is 1
            x[r] = rng.integers(-126, 126, cols) + np.float32(0.5)
            x[r, 0] = 127.0
        elif kind == 3:
            x[r] = np.nextafter(rng.integers(-126, 126, cols) + np.float32(0.5), np.float32(rng.choice([-200.0, 200.0])))
            x[r, -1] = -127.0
        elif kind == 4:
            x[r] *= np.float32(1e-41)                      # subnormal values and scales
        elif kind == 5:
            x[r] *= np.float32(3e37)
        elif kind == 6:
            x[r, rng.integers(0, cols)] = np.nan
        elif kind == 7:
            x[r, rng.integers(0, cols)] = -np.inf
        elif kind == 8:
            x[r] *= np.float32(2.0) ** np.float32(rng.integers(-105, -95))      # either side of where division takes over
    return x


# the vectors' steps of 32 and 64 values and what is left of a row; DAZ, FTZ and rounding towards zero in the calling thread
@pytest.mark.parametrize("cols", [1, 16, 31, 32, 33, 63, 64, 65, 127, 784, 4099])
@pytest.mark.parametrize("wide", [0, 1])
@pytest.mark.parametrize("csr", [0x1f80, 0xffc0])
def test_same_bits_as_the_oracle(quantizer, cols, wide, csr):
    x = rows_to_try(54, cols)
    for per_row, groups in ((1, [x]), (0, [x[r:r + 1] for r in range(54)] + [x[0:1].repeat(5, 0), x[::9].copy()])):
        for v in groups:
            for row in (cols, (cols + 15) & ~15):
                q = np.full((len(v), row), 99, np.int8)
                s = np.zeros(len(v) if per_row else 1, np.float32)
                st = quantizer(wide, v.ctypes.data_as(C.c_void_p), C.c_long(len(v)), C.c_long(cols), per_row, q.ctypes.data_as(C.c_void_p),
                               C.c_long(row), s.ctypes.data_as(C.c_void_p), C.c_uint(csr))
                if st == 0:
                    pytest.skip("no such vector units here")
                assert st == 1
                with np.errstate(all="ignore"):
                    want_q, want_s = oracle.quantize(v, bool(per_row))
                assert np.array_equal(q[:, :cols], want_q) and not q[:, cols:].any(), (cols, per_row)
                assert np.array_equal(s.view(np.int32), np.asarray(want_s).reshape(-1).view(np.int32))


def test_which_calls_the_host_quantizes_for(fake_runtime):  # noqa: F811
    """Where it is to, rows of 16 values and more and more rows than the product's launch would quantize itself go up as
    codes; a stream that is capturing, longer and shorter rows take the ways they took."""
    _run(fake_runtime, r"""
import os, re
runtime()
p = malloc_on(0, 64 << 20)
host = (C.c_float * (9 << 20))()
def kernels(name, *args):
    events()
    capi.status(name, *args)                                                  # no kernel runs here
    found = [re.search("host_copy|upload_rows|linear_gemv|quantize|gemm_i8|pad_rows", l[4]) for l in lines() if l[0] == "launch"]
    names = [f.group() for f in found if f]
    return [n for i, n in enumerate(names) if i == 0 or n != names[i - 1]]
def weights(rows, cols, per_row=1, extra=0):
    return kernels("vtl_hip_upload_quantized", host, rows, cols, per_row, p, p, p if extra else None, host if extra else None, extra)
def forward(rows, cols, per_channel, row_bytes=0):
    layer = capi.Layer(0, per_channel, 256, cols, p, p, None, row_bytes)
    return kernels("vtl_hip_forward_i8_host", host, rows, cols, C.byref(layer), 1, host)
for on in (0, 1):
    os.environ["VTL_HIP_HOST_QUANTIZE"] = str(on)
    capi.call("vtl_hip_reload_env")
    device = [] if on else ["quantize"]
    for per_row in (0, 1):
        for extra in (0, 1024, 65536):
            assert weights(8, 784, per_row, extra) == ["host_copy"] + device, (on, per_row, extra)
        assert weights(8, 16, per_row) == ["host_copy"] + device
        assert weights(8, 15, per_row) == ["host_copy", "quantize"]
        assert weights(8, 784, per_row, 65540) == ["host_copy", "quantize"]
        assert forward(33, 784, per_row)[:2] == (["host_copy"] if on else ["quantize"]) + ["gemm_i8"]
        assert forward(32, 784, per_row)[0] == ("host_copy" if on else "quantize")
        assert forward(64, 256, per_row)[0] == forward(16, 1008, 0)[0] == ("gemm_i8" if on else "quantize")     # 16 KiB of codes: read over the link
        assert forward(65, 256, per_row)[0] == forward(17, 1008, 0)[0] == ("host_copy" if on else "quantize")
        assert forward(16, 1000, per_row, 1008)[0] == ("gemm_i8" if on else "quantize")
        assert forward(1, 784, per_row) == ["linear_gemv"] and forward(8, 240, 1)[0] == "quantize"
        got = forward(40, 1000, per_row, 1008)
        assert got[:2] == (["host_copy", "gemm_i8"] if on else ["quantize", "pad_rows"]), (on, per_row, got)
        assert forward(40, 1000, per_row, 8)[-1:] != ["gemm_i8"]               # rows that do not fit are refused either way
print("done")
""")
    _run(fake_runtime, r"""
import os
os.environ["VTL_HIP_HOST_QUANTIZE"] = "1"
runtime()
p = malloc_on(0, 64 << 20)
host = (C.c_float * (9 << 20))()
events()
capi.status("vtl_hip_upload_quantized", host, 4200, 2048, 1, p, p, None, None, 0)
names = [l[4] for l in lines() if l[0] == "launch"]
assert any("host_copy" in n for n in names) and not any("upload_rows" in n or "quantize" in n for n in names), names
print("done")
""")
    _run(fake_runtime, r"""
import os
os.environ["VTL_HIP_HOST_QUANTIZE"] = "1"
runtime()
p = malloc_on(0, 1 << 20)
host = (C.c_float * (8 * 784))()
capi.call("vtl_hip_set_stream", 4096)
for capturing in (False, True):
    runtime(capturing=capturing)
    events()
    capi.status("vtl_hip_upload_quantized", host, 8, 784, 1, p, p, None, None, 0)
    assert any("host_copy" in l[4] for l in lines() if l[0] == "launch") != capturing
print("done")
""")


# (a process for each: no kernel empties a slot here)
@pytest.mark.parametrize("per_row,extra", [(0, 0), (0, 4096), (0, 65536), (1, 0), (1, 4096), (1, 65536)])
def test_little_beside_codes_takes_no_launch_of_its_own(fake_runtime, per_row, extra):  # noqa: F811
    """A bias, and the scale of all rows, go up with the first of three launches of codes."""
    _run(fake_runtime, r"""
import os
os.environ["VTL_HIP_HOST_QUANTIZE"] = "1"
runtime()
p = malloc_on(0, 64 << 20)
host = (C.c_float * (1 << 20))()
events()
extra = EXTRA
assert capi.status("vtl_hip_upload_quantized", host, 768, 512, PER_ROW, p, p, p if extra else None, host if extra else None, extra) == capi.OK
log = [l[4] for l in lines() if l[0] == "launch"]
assert sum("host_copy" in k for k in log) == 3, log
print("done")
""".replace("PER_ROW", str(per_row)).replace("EXTRA", str(extra)))


def test_few_ragged_rows_are_not_read_as_codes_over_the_link(fake_runtime):  # noqa: F811
    """Two to eight rows with one scale that are no whole vectors, from 256 values on (two rows: 1024) and up to 16 KiB of codes: a launch of the device's quantizes them."""
    _run(fake_runtime, r"""
import os, re
os.environ["VTL_HIP_HOST_QUANTIZE"] = "2"
runtime()
p = malloc_on(0, 64 << 20)
host = (C.c_float * (1 << 20))()
def first(rows, cols, per_channel=0, row_bytes=0, n=61):
    layer = capi.Layer(0, per_channel, n, cols, p, p, None, row_bytes)
    events()
    capi.status("vtl_hip_forward_i8_host", host, rows, cols, C.byref(layer), 1, host)
    found = [re.search("host_copy|linear_gemv|quantize|gemm_i8|pad_rows", l[4]) for l in lines() if l[0] == "launch"]
    return [f.group() for f in found if f][0]
for rows in range(2, 9):
    start = 1024 if rows == 2 else 256
    for cols in (17, 250, 255, 257, 1001, 1023, 1025, 1372, 2047, 4001):
        got = first(rows, cols)
        assert (got == "quantize") == (cols >= start and rows * cols <= 16384), (rows, cols, got)     # more codes are carried up
    assert first(rows, 1372, 0, 1376) != "quantize" and first(rows, 1376) != "quantize"    # padded, whole
assert first(9, 1372) != "quantize"
os.environ["VTL_HIP_HOST_QUANTIZE"] = "1"
capi.call("vtl_hip_reload_env")
assert first(8, 1372) != "quantize"
print("done")
""")


_SHORT_ROWS = r"""
import os
os.environ["VTL_HIP_HOST_QUANTIZE"] = "WHO"
runtime()
p = malloc_on(0, 64 << 20)
host = (C.c_float * (3 << 20))()
events()
if "WHAT" == "forward":
    layer = capi.Layer(0, PER_ROW, 24, NCOLS, p, p, None, 0)
    capi.status("vtl_hip_forward_i8_host", host, NROWS, NCOLS, C.byref(layer), 1, host)
else:
    capi.status("vtl_hip_upload_quantized", host, NROWS, NCOLS, PER_ROW, p, p, None, None, 0)
by = "device" if any("quantize" in l[4] for l in lines() if l[0] == "launch") else "host"
assert by == "BY", by
print("done")
"""


# (a process for each call: no kernel empties a slot here)
@pytest.mark.parametrize("what,per_row,device,host", [
    ("forward", 1, [(1000, 31), (178, 160), (2100, 48), (104, 256), (341, 192), (1400, 187), (9000, 31)],
     [(342, 192), (513, 128), (64, 257), (120, 2000), (9000, 32)]),
    ("forward", 0, [(1000, 31), (1000, 63), (9000, 31)], [(257, 64), (9000, 32)]),
    ("weights", 1, [(300, 31), (513, 32), (178, 160), (86, 191), (1400, 127), (9000, 31)], [(264, 31), (512, 32), (86, 192), (129, 128), (9000, 32)]),
    ("weights", 0, [(1000, 31), (9000, 31)], [(500, 31), (1000, 32), (9000, 32)])])
def test_short_rows_are_quantized_by_the_device(fake_runtime, what, per_row, device, host):  # noqa: F811
    """Rows that cost the host's units more than the link saves: activations, and weights."""
    calls = [(r, c, 2, "device") for r, c in device] + [(r, c, 2, "host") for r, c in host] + [(*device[0], 1, "host")]
    for rows, cols, asked, by in calls:
        program = _SHORT_ROWS
        for name, value in (("WHO", asked), ("WHAT", what), ("PER_ROW", per_row), ("NROWS", rows), ("NCOLS", cols), ("BY", by)):
            program = program.replace(name, str(value))
        _run(fake_runtime, program)


def test_few_ragged_rows_go_up_as_codes_on_a_stream(fake_runtime):  # noqa: F811
    """Once a stream has been named a launch that quantizes them would have an upload in front."""
    _run(fake_runtime, r"""
import os
os.environ["VTL_HIP_HOST_QUANTIZE"] = "2"
runtime()
p = malloc_on(0, 64 << 20)
host = (C.c_float * (1 << 16))()
capi.call("vtl_hip_set_stream", 4096)
events()
layer = capi.Layer(0, 0, 61, 1372, p, p, None, 0)
capi.status("vtl_hip_forward_i8_host", host, 8, 1372, C.byref(layer), 1, host)
names = [l[4] for l in lines() if l[0] == "launch"]
assert any("host_copy" in n for n in names) and not any("quantize" in n for n in names), names
print("done")
""")
