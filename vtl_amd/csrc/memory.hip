// Device memory of the library's callers.
//
// hipMalloc and hipFree cost 12 + 12 us at 16 MiB and 30 + 230 us from 256 MiB on, a hipFree
// waits for the device whatever the size (9 us behind the smallest launch), and two 1 GiB
// results taken in turn cost tens of milliseconds a call: more than the kernels that fill
// them.  So released blocks are kept and handed out again.
#include <exception>
#include <map>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "common.hpp"

namespace vtlhip {

bool stream_is_capturing(hipStream_t st)
{
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &capturing) != hipSuccess) {
        (void)hipGetLastError();
        return true;   // the cautious answer
    }
    return capturing != hipStreamCaptureStatusNone;
}

// Sizes are rounded up to eight steps per power of two, so that tensors of nearly the same size
// share blocks and at most an eighth is wasted.
size_t size_class(size_t bytes)
{
    if (bytes <= 512)
        return 512;
    const int top = 63 - __builtin_clzll((unsigned long long)bytes);
    const size_t step = (size_t)1 << (top < 12 ? 9 : top - 3);
    return (bytes + step - 1) & ~(step - 1);
}

namespace {

// Released blocks are kept per device and size class.  No wait is needed
// while every call of the process has used the null stream of one device (single_stream()): whatever still
// reads or writes a released block was enqueued before the release, and whoever gets the
// block next enqueues behind it.  Once a program has named a stream of its own, a release waits
// for the device first, as hipFree does, so that a block in the pool is idle on every stream.
constexpr size_t kIdleBytesMost = (size_t)8 << 30;      // idle blocks of all devices; the oldest go first
constexpr size_t kPooledBlockMost = (size_t)4 << 30;    // larger blocks go back to the driver at once

struct Block {
    size_t bytes = 0;       // size class, 0: not pooled
    int device = 0;
    bool live = false;
    bool idle = false;      // in the pool, and no stream works on it any more
    uint64_t stamp = 0;     // when it was released
};

struct DevicePool {
    std::mutex lock;
    std::unordered_map<void *, Block> blocks;
    std::map<std::pair<int, size_t>, std::vector<void *>> free_list;
    size_t idle_bytes = 0;
    uint64_t clock = 0;
};

// Never destroyed: blocks may be released by destructors that run while the process ends.
DevicePool &device_pool()
{
    static DevicePool *p = new DevicePool;
    return *p;
}

// Takes blocks out of the pool (lock held), the oldest first, until at most `keep` bytes are left.
void take_oldest(DevicePool &p, size_t keep, std::vector<void *> &out)
{
    while (p.idle_bytes > keep) {
        void *oldest = nullptr;
        uint64_t stamp = ~(uint64_t)0;
        for (auto &e : p.free_list)
            for (void *b : e.second)
                if (p.blocks[b].stamp < stamp) {
                    stamp = p.blocks[b].stamp;
                    oldest = b;
                }
        if (!oldest)
            return;
        const Block b = p.blocks[oldest];
        std::vector<void *> &list = p.free_list[{b.device, b.bytes}];
        for (size_t i = 0; i < list.size(); i++)
            if (list[i] == oldest) {
                list[i] = list.back();
                list.pop_back();
                break;
            }
        p.idle_bytes -= b.bytes;
        p.blocks.erase(oldest);
        out.push_back(oldest);
    }
}

}  // namespace

void trim_device_pool()
{
    DevicePool &p = device_pool();
    std::vector<void *> out;
    {
        std::lock_guard<std::mutex> hold(p.lock);
        take_oldest(p, 0, out);
    }
    for (void *b : out)
        (void)hipFree(b);
    (void)hipGetLastError();
}

hipError_t malloc_or_trim(void **ptr, size_t bytes)
{
    hipError_t e = hipMalloc(ptr, bytes);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        try {
            trim_device_pool();
        } catch (const std::exception &) {
        }
        e = hipMalloc(ptr, bytes);
    }
    return e;
}

}  // namespace vtlhip

using namespace vtlhip;

extern "C" {

int vtl_hip_malloc(void **dptr, size_t bytes)
try {
    if (!dptr || bytes == 0)
        return VTL_HIP_ERR_INVALID_ARG;
    *dptr = nullptr;
    int dev = 0;
    VTL_HIP_TRY(hipGetDevice(&dev));
    note_device(dev);
    DevicePool &p = device_pool();
    const bool pooled = bytes <= kPooledBlockMost && (single_stream() || !stream_is_capturing(current_stream()));
    const size_t cls = pooled ? size_class(bytes) : bytes;
    if (pooled) {
        std::lock_guard<std::mutex> hold(p.lock);
        auto it = p.free_list.find({dev, cls});
        if (it != p.free_list.end() && !it->second.empty()) {
            void *b = it->second.back();
            Block &rec = p.blocks[b];
            if (!rec.idle && !single_stream()) {
                // released while only the null stream was in use: wait once for all such blocks
                VTL_HIP_TRY(hipDeviceSynchronize());
                for (auto &e : p.free_list)
                    if (e.first.first == dev)
                        for (void *q : e.second)
                            p.blocks[q].idle = true;
            }
            it->second.pop_back();
            p.idle_bytes -= cls;
            rec.live = true;
            rec.idle = false;
            *dptr = b;
            return VTL_HIP_OK;
        }
    }
    VTL_HIP_TRY(malloc_or_trim(dptr, cls));
    std::lock_guard<std::mutex> hold(p.lock);
    Block &rec = p.blocks[*dptr];
    rec = Block();
    rec.bytes = pooled ? cls : 0;
    rec.device = dev;
    rec.live = true;
    return VTL_HIP_OK;
} catch (const std::exception &) {   // the pool's own bookkeeping found no host memory
    if (*dptr)
        (void)hipFree(*dptr);
    *dptr = nullptr;
    return VTL_HIP_ERR_OUT_OF_MEMORY;
}

int vtl_hip_malloc_on(int device_id, void **dptr, size_t bytes)
{
    if (!dptr)
        return VTL_HIP_ERR_INVALID_ARG;
    *dptr = nullptr;
    const int st = vtl_hip_set_device(device_id);
    return st != VTL_HIP_OK || bytes == 0 ? st : vtl_hip_malloc(dptr, bytes);
}

void *vtl_hip_alloc(int device_id, size_t bytes)
{
    void *dptr = nullptr;
    return vtl_hip_malloc_on(device_id, &dptr, bytes) == VTL_HIP_OK ? dptr : nullptr;
}

int vtl_hip_free(void *dptr)
try {
    if (!dptr)
        return VTL_HIP_OK;  // CudaStorage.release() skips nil too
    DevicePool &p = device_pool();
    bool known = false, pooled = false;
    int dev = 0;
    {
        std::lock_guard<std::mutex> hold(p.lock);
        auto it = p.blocks.find(dptr);
        if (it != p.blocks.end()) {
            if (!it->second.live)   // released twice: the block belongs to the pool
                return record_hip_error(hipErrorInvalidValue, "vtl_hip_free of released memory");
            known = true;
            pooled = it->second.bytes != 0;
            dev = it->second.device;
        }
    }
    bool idle = false;
    if (pooled && !single_stream()) {
        int now = 0;
        if (stream_is_capturing(current_stream()) || hipGetDevice(&now) != hipSuccess || now != dev ||
            hipDeviceSynchronize() != hipSuccess) {
            (void)hipGetLastError();
            pooled = false;
        }
        idle = true;
    }
    std::vector<void *> out;
    if (known) {
        std::lock_guard<std::mutex> hold(p.lock);
        auto it = p.blocks.find(dptr);
        if (it == p.blocks.end() || !it->second.live)
            return record_hip_error(hipErrorInvalidValue, "vtl_hip_free of released memory");
        if (pooled) {
            Block &rec = it->second;
            p.free_list[{rec.device, rec.bytes}].push_back(dptr);
            rec.live = false;
            rec.idle = idle;
            rec.stamp = ++p.clock;
            p.idle_bytes += rec.bytes;
            if (p.idle_bytes > kIdleBytesMost)
                take_oldest(p, kIdleBytesMost, out);
        } else {
            p.blocks.erase(it);
        }
    }
    if (!pooled)
        VTL_HIP_TRY(hipFree(dptr));
    for (void *b : out)
        VTL_HIP_TRY(hipFree(b));
    return VTL_HIP_OK;
} catch (const std::exception &) {
    return VTL_HIP_ERR_OUT_OF_MEMORY;
}

int vtl_hip_trim(void)
try {
    trim_device_pool();
    trim_pinned_pool();
    return VTL_HIP_OK;
} catch (const std::exception &) {
    return VTL_HIP_ERR_OUT_OF_MEMORY;
}

}  // extern "C"
