"""Device storage: the Python mirror of the V file `storage/hip_d_hip.v`.

Follows `CudaStorage[T]` (storage/cuda_d_cuda.v:19-107): a raw device pointer
with byte size and element count, created from host memory with a blocking
copy, copied back with `cpu()` / `to_array()`, and released explicitly
(nothing frees on garbage collection in the reference; here `__del__` is a
safety net only).  A numpy array stands in for `CpuStorage[T]`.
"""
from __future__ import annotations

import ctypes as C
from dataclasses import dataclass

import numpy as np

from . import capi


@dataclass
class HipParams:
    """`@[params] HipParams{device_id int = 0}` (cf. CudaParams, storage/cuda_d_cuda.v:9-11)."""
    device_id: int = 0


_SUPPORTED = (np.float32, np.int8, np.int32, np.float64, np.uint8)
_DTYPES = {t: np.dtype(t) for t in _SUPPORTED} | {np.dtype(t): np.dtype(t) for t in _SUPPORTED}


# Results of more bytes than this are arrays over pinned memory of the library, which the device
# writes itself; smaller ones are copied into ordinary memory, which the allocator recycles
# (from 128 KiB on it would map fresh pages for each).
_PINNED_FROM = 128 << 10


class _HostBlock:
    """Pinned memory under one result array; goes back to the library with the array."""

    __slots__ = ("ptr", "__array_interface__")

    def __init__(self, ptr: int, count: int, dt: np.dtype):
        self.ptr = ptr
        self.__array_interface__ = {"shape": (count,), "typestr": dt.str, "data": (ptr, False), "version": 3}

    def __del__(self):
        capi._lib.vtl_hip_host_free(self.ptr)


def host_array(count: int, dt: np.dtype):
    """An uninitialised array for a download and its address."""
    nbytes = count * dt.itemsize
    if nbytes > _PINNED_FROM:
        ptr = C.c_void_p(0)
        if capi.lib().vtl_hip_host_alloc(C.byref(ptr), nbytes) == capi.OK:
            return np.asarray(_HostBlock(ptr.value, count, dt)), ptr.value
    out = np.empty(count, dt)
    return out, out.ctypes.data


_PARAMS: dict = {}


class HipStorage:
    """`HipStorage[T]{ptr voidptr; size int; count int; device_id int}`."""

    def __init__(self, ptr: int, size: int, count: int, dtype, device_id: int = 0):
        self.ptr = ptr
        self.size = size      # bytes
        self.count = count    # elements
        self.dtype = dtype if type(dtype) is np.dtype else np.dtype(dtype)
        self.device_id = device_id

    # -- construction ------------------------------------------------------
    @staticmethod
    def empty(count: int, dtype, params: HipParams | None = None) -> "HipStorage":
        """Uninitialised memory.  It may be a released storage's, which calls enqueued before still use: a
        stream that the library was never told of (vtl_hip_set_stream) waits for vtl_hip_sync before it writes there."""
        device_id = params.device_id if params is not None else 0
        dt = _DTYPES.get(dtype)
        if dt is None:
            dt = np.dtype(dtype)
            if dt.type not in _SUPPORTED:
                raise TypeError(f"HipStorage: unsupported element type {dt}")
        count = int(count)
        nbytes = count * dt.itemsize
        ptr = capi.alloc(device_id, nbytes)    # an address in one call: small operations on tensors are made of such calls
        if not ptr:
            ptr = C.c_void_p()
            capi.call("vtl_hip_malloc_on", device_id, C.byref(ptr), nbytes)
            ptr = ptr.value or 0
        return HipStorage(ptr, nbytes, count, dt, device_id)

    @staticmethod
    def from_cpu(arr: np.ndarray, params: HipParams | None = None) -> "HipStorage":
        """`(cpu &CpuStorage[T]) hip(params) !&HipStorage[T]` (storage/cuda_d_cuda.v:32-55).  The bytes
        are there on return, for work on any stream."""
        flat = np.ascontiguousarray(arr).reshape(-1)
        st = HipStorage.empty(flat.size, flat.dtype, params)
        if st.size:
            capi.call("vtl_hip_memcpy_h2d", st.ptr, flat.ctypes.data, st.size)
        return st

    @property
    def params(self) -> HipParams:
        """What makes another storage on the same device."""
        p = _PARAMS.get(self.device_id)
        if p is None:
            p = _PARAMS[self.device_id] = HipParams(self.device_id)
        return p

    def hip(self, params: HipParams | None = None) -> "HipStorage":
        """Identity, for chaining (storage/cuda_d_cuda.v:62-65)."""
        return self

    # -- transfer back -------------------------------------------------------
    def cpu(self) -> np.ndarray:
        """`.cpu() !&CpuStorage[T]` (storage/cuda_d_cuda.v:68-81)."""
        if self.count and not self.ptr:
            raise capi.VtlHipError("HipStorage.cpu", capi.ERR_INVALID_ARG, "null pointer")
        out, host = host_array(self.count, self.dtype)
        if self.size:
            capi.call("vtl_hip_memcpy_d2h", host, self.ptr, self.size)
        return out

    @staticmethod
    def cpu_all(storages) -> list:
        """`.cpu()` of several storages with one wait for all of them."""
        n = len(storages)
        outs = [host_array(s.count, s.dtype) for s in storages]
        capi.call("vtl_hip_download", n, (C.c_void_p * n)(*[o[1] for o in outs]),
                  (C.c_void_p * n)(*[s.ptr for s in storages]), (C.c_size_t * n)(*[s.size for s in storages]))
        return [o[0] for o in outs]

    def to_array(self) -> np.ndarray:
        """`.to_array() ![]T` (storage/cuda_d_cuda.v:84-95)."""
        return self.cpu()

    def release(self) -> None:
        """`.release()` (storage/cuda_d_cuda.v:98-102)."""
        if self.ptr:
            capi.call("vtl_hip_free", self.ptr)
            self.ptr = 0

    def __del__(self):  # safety net; the reference relies on explicit release()
        try:
            if self.ptr:
                capi._lib.vtl_hip_free(self.ptr)
                self.ptr = 0
        except Exception:
            pass


def hip_available() -> bool:
    """True when the library loads and reports at least one device."""
    try:
        return capi.device_count() > 0
    except (OSError, FileNotFoundError):
        return False
