// A HIP runtime for one test process without a GPU: it keeps count of devices, streams and
// allocations (in host memory), writes down what is enqueued where, and runs no kernel.  Loaded with
// RTLD_GLOBAL before libvtlhip.so, its functions take the place of the real ones.
#include <hip/hip_runtime_api.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <unistd.h>

#include <map>
#include <mutex>
#include <string>

namespace {

std::mutex g_lock;
std::string g_log;
int g_devices = 2, g_capturing = 0, g_refuse_memory = 0, g_wait_ms = 0;
thread_local int g_device = 0;
struct Range {
    size_t bytes;
    int device;
};
std::map<const char *, Range> g_memory;
std::map<const void *, std::string> g_kernels;   // mangled names

void note(const char *what, void *stream, unsigned long long n, const std::string &more = "")
{
    char line[128];
    snprintf(line, sizeof line, "%s %d %llu %llu", what, g_device, (unsigned long long)(uintptr_t)stream, n);
    std::lock_guard<std::mutex> hold(g_lock);
    g_log += line + more + "\n";
}

struct Call {
    dim3 grid, block;
    size_t shared;
    hipStream_t stream;
};
thread_local Call g_call;

}  // namespace

extern "C" {

void fake_set(int devices, int capturing, int refuse_memory, int wait_ms)
{
    g_devices = devices;
    g_capturing = capturing;
    g_refuse_memory = refuse_memory;
    g_wait_ms = wait_ms;
}

// The lines "<event> <device> <stream> <number>" since the last call; of a launch also the kernel's name and, of
// the f64-accumulating matmul and the column sums, the address they write to.
size_t fake_log(char *out, size_t cap)
{
    std::lock_guard<std::mutex> hold(g_lock);
    const size_t n = g_log.size() < cap ? g_log.size() : cap;
    memcpy(out, g_log.data(), n);
    g_log.clear();
    return n;
}

hipError_t hipGetDeviceCount(int *n) { *n = g_devices; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = g_device; return hipSuccess; }
hipError_t hipSetDevice(int d) { g_device = d; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }

hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }

hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }

hipError_t hipMalloc(void **p, size_t bytes)
{
    note("malloc", nullptr, bytes);
    if (g_refuse_memory)
        return hipErrorOutOfMemory;
    *p = aligned_alloc(4096, (bytes + 4095) / 4096 * 4096);
    std::lock_guard<std::mutex> hold(g_lock);
    g_memory[static_cast<char *>(*p)] = {bytes, g_device};
    return hipSuccess;
}

hipError_t hipFree(void *p)
{
    note("free", nullptr, 0);
    std::lock_guard<std::mutex> hold(g_lock);
    g_memory.erase(static_cast<char *>(p));
    free(p);
    return hipSuccess;
}

hipError_t hipHostMalloc(void **p, size_t bytes, unsigned)
{
    note("host_malloc", nullptr, bytes);
    *p = aligned_alloc(4096, (bytes + 4095) / 4096 * 4096);
    return hipSuccess;
}

hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }

hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p)
{
    std::lock_guard<std::mutex> hold(g_lock);
    auto it = g_memory.upper_bound(static_cast<const char *>(p));
    if (it == g_memory.begin())
        return hipErrorInvalidValue;
    --it;
    if (static_cast<const char *>(p) >= it->first + it->second.bytes)
        return hipErrorInvalidValue;
    memset(a, 0, sizeof *a);
    a->type = hipMemoryTypeDevice;
    a->device = it->second.device;
    a->devicePointer = const_cast<void *>(p);
    return hipSuccess;
}

hipError_t hipGetSymbolAddress(void **p, const void *)
{
    static void *cells = calloc(1, (size_t)64 << 20);
    *p = cells;
    return hipSuccess;
}

hipError_t hipMemcpyAsync(void *, const void *, size_t bytes, hipMemcpyKind, hipStream_t st)
{
    note("copy", st, bytes);
    return hipSuccess;
}

hipError_t hipStreamSynchronize(hipStream_t st)
{
    note("sync", st, 0);
    if (g_wait_ms)
        usleep(1000 * g_wait_ms);
    return hipSuccess;
}

hipError_t hipDeviceSynchronize() { note("device_sync", nullptr, 0); return hipSuccess; }

hipError_t hipStreamIsCapturing(hipStream_t st, hipStreamCaptureStatus *s)
{
    *s = g_capturing && st ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}

hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t st)
{
    g_call = {grid, block, shared, st};
    return hipSuccess;
}

hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *st)
{
    *grid = g_call.grid;
    *block = g_call.block;
    *shared = g_call.shared;
    *st = g_call.stream;
    return hipSuccess;
}

void __hipRegisterFunction(void **, const void *function, char *, const char *name, unsigned, void *, void *, dim3 *, dim3 *,
                           int *)
{
    std::lock_guard<std::mutex> hold(g_lock);
    g_kernels[function] = name;
}

hipError_t hipLaunchKernel(const void *function, dim3 grid, dim3, void **args, size_t, hipStream_t st)
{
    std::string more = " ?";
    auto it = g_kernels.find(function);
    if (it != g_kernels.end())
        more = " " + it->second;
    if (more.find("matmul_f64acc_direct_kernel") != std::string::npos)   // its argument begins with A, B, C
        more += " " + std::to_string((unsigned long long)(uintptr_t) static_cast<void **>(args[0])[2]);
    else if (more.find("13colsum_kernel") != std::string::npos)              // x, rows, cols, rows of a split, out
        more += " " + std::to_string((unsigned long long)(uintptr_t) * static_cast<void **>(args[4]));
    else if (more.find("colsum_short_kernel") != std::string::npos)          // its argument begins with x, rows and cols, out
        more += " " + std::to_string((unsigned long long)(uintptr_t) static_cast<void **>(args[0])[2]);
    else if (more.find("linear_backward_kernel") != std::string::npos) {     // that, and those of two products of 104 bytes each
        void **words = static_cast<void **>(args[0]);
        const std::string name = more;
        for (int at : {3 + 2, 3 + 13 + 2})
            if (words[at])
                note("launch", st, (unsigned long long)grid.x, name + " " + std::to_string((unsigned long long)(uintptr_t)words[at]));
        if (!words[2])
            return hipSuccess;
        more += " " + std::to_string((unsigned long long)(uintptr_t)words[2]);
    }
    note("launch", st, (unsigned long long)grid.x * grid.y * grid.z, more);
    return hipSuccess;
}

}  // extern "C"
