// Pinned host memory and the copies between host and device.
//
// What bounds them: below a few hundred KiB the latency of the copy engines and of
// hipStreamSynchronize, above it the link (57 GB/s each way from pinned memory; the runtime's copies
// of pageable memory reach 31 to 35 GB/s up and 17 down) and, for results, the page faults of
// fresh host memory (4.7 GB/s).
#include <sched.h>
#include <stdio.h>
#include <string.h>
#include <time.h>

#include <atomic>
#include <condition_variable>
#include <deque>
#include <exception>
#include <map>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

#include "common.hpp"
#include "host_quant.hpp"
#include "quant_device.hpp"

namespace vtlhip {

namespace {

// ---- pinned host memory ----------------------------------------------------------
// Blocks that host tensors are made of (results of downloads): the device writes them directly,
// and a block that comes round again has its pages in place, where fresh memory costs a page
// fault of 0.9 us every 4 KiB (4.7 GB/s).
constexpr size_t kPinnedLiveMost = (size_t)1 << 30;     // beyond, callers use ordinary memory
constexpr size_t kPinnedIdleMost = (size_t)256 << 20;

struct PinnedPool {
    std::mutex lock;
    std::map<uintptr_t, size_t> live;                   // start -> size class
    std::map<size_t, std::vector<void *>> free_list;
    size_t live_bytes = 0, idle_bytes = 0;
};

PinnedPool &pinned_pool()
{
    static PinnedPool *p = new PinnedPool;
    return *p;
}

bool in_pinned_pool(const void *ptr, size_t bytes)
{
    PinnedPool &p = pinned_pool();
    const uintptr_t a = reinterpret_cast<uintptr_t>(ptr);
    std::lock_guard<std::mutex> hold(p.lock);
    auto it = p.live.upper_bound(a);
    if (it == p.live.begin())
        return false;
    --it;
    return a + bytes <= it->first + it->second;
}

// ---- copy kernel -------------------------------------------------------------------
// Copies up to kMaxSegments runs of bytes between device memory and pinned host memory, and, when
// a flag is given, raises it in pinned memory once every byte is there.  Used instead of the copy
// engines because a kernel needs no hand-over between queues: host -> device copy, kernel and
// flag take 11.6 us for 64 KiB and 14.2 us for 196 KiB where the same chain through
// hipMemcpyAsync takes 23.0 and 25.6 us, and from 4 MiB on both run at the link's 50 to 57 GB/s.
// 16 workgroups keep the link full (50.6 GB/s at 4 MiB up, with 64 of them 46.8); only downloads from
// 1 MiB on take 32.
constexpr int kMaxSegments = 4;

struct Segment {
    char *dst;
    const char *src;     // same position within 16 bytes as dst
    size_t nvec;         // 16-byte vectors
    unsigned head, tail; // single bytes before and after them
};

struct LinkSignals {
    DoneSignal done;
    unsigned *behind;    // flag of the launch before this one, which has ended by now, or nullptr
    unsigned behind_value;
    int to_host;         // the bytes have to be visible to the host when the flag is (else: the source is free)
};

struct CopyArgs {
    Segment seg[kMaxSegments];
    int count;
    LinkSignals signals;
};

__device__ __forceinline__ void raise_behind(const LinkSignals &s)
{
    if (s.behind && blockIdx.x == 0 && threadIdx.x == 0)
        __hip_atomic_store(s.behind, s.behind_value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// At the end of a workgroup whose pinned source has been read (or, to_host, whose bytes are there).
__device__ __forceinline__ void raise_done(const LinkSignals &s)
{
    const DoneSignal &done = s.done;
    if (!done.flag)
        return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // every load has returned, every store is acknowledged
    __syncthreads();
    if (threadIdx.x != 0)
        return;
    if (s.to_host) {
        // one system-scope fence per workgroup covers the stores of all of its threads (they
        // happen before it through the barrier); whoever counts last raises the flag
        __threadfence_system();
        const unsigned before = __hip_atomic_fetch_add(done.counter, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        if (before + 1 == done.target)
            __hip_atomic_store(done.flag, done.value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    } else {
        // nothing to publish: the flag says that the pinned source has been read, which the
        // returned loads are enough for (a fence would write the caches back at every chunk)
        const unsigned before = __hip_atomic_fetch_add(done.counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (before + 1 == done.target)
            __hip_atomic_store(done.flag, done.value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// One workgroup's share of a segment.
__device__ __forceinline__ void copy_segment(const Segment &seg)
{
    const size_t first = (size_t)blockIdx.x * 512 + threadIdx.x, step = (size_t)gridDim.x * 512;
    const uint4 *src = reinterpret_cast<const uint4 *>(seg.src + seg.head);
    uint4 *dst = reinterpret_cast<uint4 *>(seg.dst + seg.head);
    size_t i = first;
    for (; i + 3 * step < seg.nvec; i += 4 * step) {   // four reads of the link in flight per lane
        const uint4 a = src[i], b = src[i + step], c = src[i + 2 * step], d = src[i + 3 * step];
        dst[i] = a;
        dst[i + step] = b;
        dst[i + 2 * step] = c;
        dst[i + 3 * step] = d;
    }
    for (; i < seg.nvec; i += step)
        dst[i] = src[i];
    if (blockIdx.x == 0) {
        if (threadIdx.x < seg.head)
            seg.dst[threadIdx.x] = seg.src[threadIdx.x];
        const size_t end = seg.head + seg.nvec * 16;
        if (threadIdx.x < seg.tail)
            seg.dst[end + threadIdx.x] = seg.src[end + threadIdx.x];
    }
}

__global__ __launch_bounds__(512) void host_copy_kernel(const CopyArgs g)
{
    raise_behind(g.signals);
    for (int s = 0; s < g.count; s++)
        copy_segment(g.seg[s]);
    raise_done(g.signals);
}

// f32 rows in pinned memory that arrive as codes and scales, `cols` of the launch each.
struct Rows {
    const float *src;    // 16-byte aligned; nullptr: none
    int8_t *q;
    float *scale;
    int count;
};

struct RowsArgs {
    Rows rows[kMaxSegments];
    Segment seg[kMaxSegments];   // copied as they are
    int count, copies, cols;
    LinkSignals signals;
};

// Per-row quantization of what comes over the link: the f32 rows never lie in device memory, and no launch behind the transfer reads
// them again.  Bound by the link, 56 GB/s as the copy: a workgroup has one row in registers and the next one on its way.  The end of
// a launch, when the last rows are there, is a microsecond longer than a copy's, so it is for transfers of many MiB a
// launch (us, copy and quantizer behind it, and this: 11008 x 4096 3659 and 3614 of a forward, 4096 x 4096 1279 and
// 1265; 512 x 4096 213 and 217, 1000 x 1000 120 and 122).  More workgroups take longer on the link (4096 x 4096 with 16 1270,
// 32 1303, 64 1308).  Of rows of fewer than 2048 values too little is on its way at a time: 8192 x 1024 705 and 1000, 32768 x 1024 2525 and
// 3760, 20000 x 1536 2305 and 2500, x 1800 2710 and 2790; 20000 x 2048 3040 and 3030.  Arithmetic as in quant.hip.
constexpr size_t kRowsFrom = (size_t)32 << 20;
constexpr int kRowsLeastCols = 2048, kRowsMostCols = 8192;

template <int NV>
__global__ __launch_bounds__(512) void upload_rows_kernel(const RowsArgs g)
{
    using namespace qdev;
    __shared__ float smem[2][8];
    raise_behind(g.signals);
    const int tid = (int)threadIdx.x, nv = g.cols >> 2;
    int turn = 0;
    for (int s = 0; s < g.count; s++) {
        const Rows &part = g.rows[s];
        float4_t next[NV];
        auto load = [&](int row) {
#pragma unroll
            for (int i = 0; i < NV; i++) {
                const int idx = i * 512 + tid;
                next[i] = float4_t{0.f, 0.f, 0.f, 0.f};
                if (row < part.count && idx < nv)
                    next[i] = reinterpret_cast<const float4_t *>(part.src)[(size_t)row * nv + idx];
            }
        };
        load((int)blockIdx.x);
        for (int row = (int)blockIdx.x; row < part.count; row += (int)gridDim.x) {
            float4_t v[NV];
#pragma unroll
            for (int i = 0; i < NV; i++)
                v[i] = next[i];
            load(row + (int)gridDim.x);
            float m = 0.0f;
#pragma unroll
            for (int i = 0; i < NV; i++)
                m = absmax4(m, v[i]);
            m = wave_max(m);
            if ((tid & 63) == 0)
                smem[turn][tid >> 6] = m;
            lds_barrier();   // (the next row stays on its way)
            m = smem[turn][0];
#pragma unroll
            for (int i = 1; i < 8; i++)
                m = fmaxf(m, smem[turn][i]);
            turn ^= 1;       // the next row's maxima: others may still read these
            const float scale = m / 127.0f;
            if (tid == 0)
                part.scale[row] = scale;
            const QuantScale p = make_quant_scale(scale);
#pragma unroll
            for (int i = 0; i < NV; i++) {
                const int idx = i * 512 + tid;
                if (idx < nv)
                    reinterpret_cast<unsigned *>(part.q)[(size_t)row * nv + idx] = quant4(v[i], p);
            }
        }
    }
    for (int s = 0; s < g.copies; s++)
        copy_segment(g.seg[s]);
    raise_done(g.signals);
}

void launch_upload_rows(const RowsArgs &g, unsigned blocks, hipStream_t st)
{
    const dim3 grid(blocks), block(512);
    if (g.cols <= 2048)
        hipLaunchKernelGGL((upload_rows_kernel<1>), grid, block, 0, st, g);
    else if (g.cols <= 4096)
        hipLaunchKernelGGL((upload_rows_kernel<2>), grid, block, 0, st, g);
    else
        hipLaunchKernelGGL((upload_rows_kernel<4>), grid, block, 0, st, g);
}

Segment make_segment(void *dst, const void *src, size_t bytes)
{
    Segment s;
    s.dst = static_cast<char *>(dst);
    s.src = static_cast<const char *>(src);
    size_t head = (16 - (reinterpret_cast<uintptr_t>(dst) & 15)) & 15;
    if (head > bytes)
        head = bytes;
    s.head = (unsigned)head;
    s.nvec = (bytes - head) >> 4;
    s.tail = (unsigned)((bytes - head) & 15);
    return s;
}

unsigned copy_blocks(size_t bytes)
{
    const size_t per = (size_t)512 * 16;
    const size_t want = (bytes + per - 1) / per;
    const size_t most = bytes >= ((size_t)1 << 20) ? 32 : 16;
    return (unsigned)(want < 1 ? 1 : want > most ? most : want);
}

constexpr int kMaxDevices = 64;

// A flag in pinned memory, the counter in device memory that its launches count on, and what both
// read when the last launch is done.  One launch at a time.
struct Signal {
    unsigned *flag = nullptr;
    unsigned *counter = nullptr;
    unsigned arrived = 0, value = 0;

    DoneSignal next(unsigned blocks) const { return {counter, arrived + blocks, value + 1, flag}; }
    void attach(LinkSignals &s, unsigned blocks, bool to_host)
    {
        s.done = next(blocks);
        s.to_host = to_host;
    }
    void launched(unsigned blocks)
    {
        arrived += blocks;
        value++;
    }
    bool raised() const { return reached(flag, value); }
    static bool reached(const unsigned *flag, unsigned value)
    {
        return (int)(__atomic_load_n(flag, __ATOMIC_ACQUIRE) - value) >= 0;
    }
};

__global__ void clear_counters_kernel(unsigned *p) { p[threadIdx.x] = 0; }

// Pinned memory that starts with `n` flags, 64 bytes apart, and device counters for them.
constexpr size_t kFlagBytes = 4096;
int make_signals(Signal *sig, int n, size_t pinned_bytes, char *&pinned)
{
    void *host = nullptr, *dev = nullptr;
    hipError_t e = hipHostMalloc(&host, kFlagBytes + pinned_bytes, hipHostMallocDefault);
    if (e == hipSuccess)
        e = malloc_or_trim(&dev, 64 * sizeof(unsigned) * 16);
    int rc = e == hipSuccess ? VTL_HIP_OK : record_hip_error(e, "memory of a host copy");
    if (rc == VTL_HIP_OK) {
        hipLaunchKernelGGL(clear_counters_kernel, dim3(1), dim3(1024), 0, current_stream(), static_cast<unsigned *>(dev));
        rc = check_launch("clear_counters_kernel");
        if (rc == VTL_HIP_OK && hipStreamSynchronize(current_stream()) != hipSuccess)   // the next user may come with another stream
            rc = record_hip_error(hipErrorUnknown, "clear_counters_kernel");
    }
    if (rc != VTL_HIP_OK) {
        if (host)
            (void)hipHostFree(host);
        if (dev)
            (void)hipFree(dev);
        return rc;
    }
    memset(host, 0, kFlagBytes);
    for (int i = 0; i < n; i++) {
        sig[i].flag = static_cast<unsigned *>(host) + 16 * i;
        sig[i].counter = static_cast<unsigned *>(dev) + 16 * i;
    }
    pinned = static_cast<char *>(host) + kFlagBytes;
    return VTL_HIP_OK;
}


// ---- lanes: what a download waits with -----------------------------------------------
// A signal and a staging buffer in pinned memory, leased for the length of one call, so that
// calls on several threads and streams do not meet.
constexpr size_t kLaneStage = (size_t)1 << 20;

struct Lane {
    int device = -1;
    Signal signal;
    char *stage = nullptr;
};

struct Lanes {
    std::mutex lock;
    std::vector<Lane *> spare;
};

Lanes &lanes()
{
    static Lanes *l = new Lanes;
    return *l;
}

int lease_lane(Lane *&out)
{
    int dev = 0;
    VTL_HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices)
        return VTL_HIP_ERR_NO_DEVICE;
    {
        Lanes &l = lanes();
        std::lock_guard<std::mutex> hold(l.lock);
        for (size_t i = l.spare.size(); i-- > 0;)
            if (l.spare[i]->device == dev) {
                out = l.spare[i];
                l.spare.erase(l.spare.begin() + (long)i);
                return VTL_HIP_OK;
            }
    }
    std::unique_ptr<Lane> lane(new Lane);
    lane->device = dev;
    const int rc = make_signals(&lane->signal, 1, kLaneStage, lane->stage);
    if (rc == VTL_HIP_OK)
        out = lane.release();
    return rc;
}

void return_lane(Lane *lane)
{
    Lanes &l = lanes();
    std::lock_guard<std::mutex> hold(l.lock);
    l.spare.push_back(lane);
}

double seconds()
{
    timespec t;
    clock_gettime(CLOCK_MONOTONIC, &t);
    return (double)t.tv_sec + 1e-9 * (double)t.tv_nsec;
}

// Waits for a launch: its flag is polled for two milliseconds, then it is left to the
// runtime, which also reports what went wrong if the launch never ends well.
int wait_flag(const unsigned *flag, unsigned value, hipStream_t st)
{
    const double began = seconds();
    for (;;) {
        for (int i = 0; i < 64; i++) {
            if (Signal::reached(flag, value))
                return VTL_HIP_OK;
            __builtin_ia32_pause();
        }
        if (seconds() - began > 2e-3)
            break;
    }
    VTL_HIP_TRY(hipStreamSynchronize(st));
    return Signal::reached(flag, value) ? VTL_HIP_OK : record_hip_error(hipErrorUnknown, "host copy ended without its flag");
}

// Small uploads enqueued so far and those known to have been read, per device: what a download has
// waited for tells that every upload before it is done with its staging memory.
struct UploadCount {
    std::atomic<uint64_t> enqueued{0}, done{0};
};

UploadCount g_uploads[kMaxDevices];

// Waits for a lane's flag behind which `before` uploads were enqueued.
int wait_behind(Lane *lane, uint64_t before, bool one_stream, hipStream_t st)
{
    const int rc = wait_flag(lane->signal.flag, lane->signal.value, st);
    if (rc == VTL_HIP_OK && one_stream) {
        UploadCount &uploads = g_uploads[lane->device];
        uint64_t seen = uploads.done.load(std::memory_order_relaxed);
        while (seen < before && !uploads.done.compare_exchange_weak(seen, before))
            ;
    }
    return rc;
}

// Enqueues the segments with a flag at the end and waits for it.
int copy_and_wait(CopyArgs &g, size_t bytes, Lane *lane, hipStream_t st)
{
    const bool one_stream = single_stream();
    const uint64_t before = g_uploads[lane->device].enqueued.load(std::memory_order_acquire);
    const unsigned blocks = copy_blocks(bytes);
    lane->signal.attach(g.signals, blocks, true);
    hipLaunchKernelGGL(host_copy_kernel, dim3(blocks), dim3(512), 0, st, g);
    int rc = check_launch("host_copy_kernel");
    if (rc != VTL_HIP_OK)
        return rc;
    lane->signal.launched(blocks);
    return wait_behind(lane, before, one_stream, st);
}

// ---- staging ring ------------------------------------------------------------------------
// Pinned slots that uploads go through (the host copies in, a kernel carries over), and downloads
// into memory that is not the library's.  The last kernel that uses a slot raises its flag: an event
// behind every chunk instead held the next one back for 5.5 us of a 21 us MiB.
constexpr int kSlots = 8;
constexpr size_t kSlotBytes = (size_t)4 << 20;
constexpr size_t kSlotStride = kSlotBytes + 4096;
constexpr size_t kWithAnother = (size_t)64 << 10;
constexpr size_t kManyHelpersFrom = (size_t)16 << 20;   // below, more than three helpers cost more to wake than they do (4 MiB, us of a forward: 157 and 171)
constexpr int kCodesLeastCols = 16;             // rows of fewer values are hardly fewer bytes as codes and a scale
constexpr size_t kSmall = (size_t)1 << 20;      // up to here one host thread copies faster than others wake up

struct Ring {
    std::mutex lock;         // one transfer at a time
    UploadCount *uploads = nullptr;
    char *base = nullptr;
    Signal signal[kSlots];
    int slot = 0;            // slot that small uploads fill
    size_t used = 0;         // bytes of it that are taken

    // What says that a slot is free again: a launch may read several, and raises the flag of its first.
    struct Gate {
        int signal;
        unsigned value;
    } gate[kSlots] = {};

    char *at(int i) { return base + (size_t)i * kSlotStride; }
    bool is_free(int i) const { return Signal::reached(signal[gate[i].signal].flag, gate[i].value); }
    int wait(int i, hipStream_t st) { return wait_flag(signal[gate[i].signal].flag, gate[i].value, st); }
    // Slots on their way up, and no launch yet behind theirs that would raise their flag.
    int waiting = -1;

    // A launch that reads the slots first .. first + count - 1.  On the way up the next launch on the
    // stream raises their flag, which begins when this one has ended (counting workgroups and a flag of its own
    // hold a launch back for about 1.5 us, on a link that a MiB keeps busy for 18); only the last launch (`own`) counts.
    LinkSignals signals_for(int first, unsigned blocks, bool own, bool to_host)
    {
        LinkSignals s = {};
        if (waiting >= 0) {
            s.behind = signal[waiting].flag;
            s.behind_value = signal[waiting].value;
        }
        if (own)
            signal[first].attach(s, blocks, to_host);
        return s;
    }
    void launched(int first, int count, unsigned blocks, bool own)
    {
        if (own)
            signal[first].launched(blocks);
        else
            signal[first].value++;
        waiting = own ? -1 : first;
        for (int i = 0; i < count; i++)
            gate[(first + i) % kSlots] = {first, signal[first].value};
    }
    // After a failure nothing is under way any more and the host raises the flag.
    void give_up(hipStream_t st)
    {
        (void)hipStreamSynchronize(st);
        (void)hipGetLastError();
        if (waiting >= 0)
            __atomic_store_n(signal[waiting].flag, signal[waiting].value, __ATOMIC_RELEASE);
        waiting = -1;
    }
    // Copies with the slot's flag at the end; no bytes: the flag behind the kernels before.
    int launch(int i, void *dst, const void *src, size_t bytes, bool to_host, hipStream_t st)
    {
        CopyArgs g = {};
        if (bytes) {
            g.seg[0] = make_segment(dst, src, bytes);
            g.count = 1;
        }
        const unsigned blocks = copy_blocks(bytes < kSmall || to_host ? bytes : kSmall - 1);
        g.signals = signals_for(i, blocks, true, to_host);
        hipLaunchKernelGGL(host_copy_kernel, dim3(blocks), dim3(512), 0, st, g);
        const int rc = check_launch("host_copy_kernel");
        if (rc == VTL_HIP_OK)
            launched(i, 1, blocks, true);
        return rc;
    }
    // Closes the slot that small uploads were filling; the next transfer starts in a slot of its own.
    int close(hipStream_t st)
    {
        if (used == 0)
            return VTL_HIP_OK;
        const int rc = launch(slot, nullptr, nullptr, 0, false, st);
        slot = (slot + 1) % kSlots;
        used = 0;
        return rc;
    }
};

Ring *ring_of_current_device()
{
    static Ring *rings[kMaxDevices] = {};
    static std::mutex lock;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        (void)hipGetLastError();
        return nullptr;
    }
    std::lock_guard<std::mutex> hold(lock);
    if (!rings[dev]) {
        std::unique_ptr<Ring> r(new Ring);
        if (make_signals(r->signal, kSlots, kSlots * kSlotStride, r->base) != VTL_HIP_OK)
            return nullptr;
        r->uploads = &g_uploads[dev];
        rings[dev] = r.release();
    }
    return rings[dev];
}

// ---- host threads that share a large transfer's copying ------------------------------------
// One thread copies 31 GB/s out of memory that is in no cache and touches 4.7 GB/s of fresh pages; the
// link takes 57.  Three helpers and the caller reach 90 GB/s.  A helper looks for jobs for half a millisecond,
// seven chunks' time on the link, before it sleeps: a transfer that keeps the link busy never waits for one to wake
// (50 us), and one that stands behind a long device queue costs no host time.
constexpr double kHelpersLook = 0.5e-3;

// Up to two numbers from a file, 0 for what is not there.
void read_numbers(const char *path, double &a, double &b)
{
    if (FILE *f = fopen(path, "r")) {
        if (fscanf(f, "%lf %lf", &a, &b) < 1)
            a = 0;
        fclose(f);
    }
}

// Processors that this process may keep busy: those it may run on, or its container's share (both
// generations of control groups) where that is less.
int processors()
{
    cpu_set_t cpus;
    const int have = sched_getaffinity(0, sizeof cpus, &cpus) == 0 ? CPU_COUNT(&cpus) : 1;
    double quota = 0, period = 0, unused = 0;
    read_numbers("/sys/fs/cgroup/cpu.max", quota, period);       // "max <period>" without a limit
    if (period <= 0) {
        read_numbers("/sys/fs/cgroup/cpu/cpu.cfs_quota_us", quota, unused);    // -1 without one
        read_numbers("/sys/fs/cgroup/cpu/cpu.cfs_period_us", period, unused);
    }
    if (quota <= 0 || period <= 0 || quota >= period * have)
        return have;
    return quota < period ? 1 : (int)(quota / period);
}

// Quantization of rows: what a source or a piece of one becomes on its way, if anything (no codes: its bytes are copied).
struct Quantized {
    int8_t *q = nullptr;         // codes on the device
    float *scale = nullptr;      // one for each row there
    size_t unit = 0;             // bytes of a row of f32 (they are not cut)
    // by the host's threads: bytes from one row of codes to the next, and the scale of all rows (with `one`)
    const HostQuantizer *host = nullptr;
    size_t row = 0;
    bool one = false;
    float given = 0.0f;
};

struct Crew {
    struct Job {
        char *dst;
        const char *src;
        size_t bytes;
        std::atomic<int> *left;         // jobs of the same chunk that are not done
        const Quantized *codes;         // makes codes at dst (with none there: the largest magnitude for `scales`) instead of a copy
        float *scales;
    };
    // (us, 180 MB made codes of and their forward, in jobs of 64 / 128 / 256 KiB: 2780 / 1670 / 1480; they meet at the lock)
    static constexpr size_t kJobBytes = (size_t)256 << 10;
    // How many helpers there are, where processors are many, and how many of them a copy takes: the link needs no more, but what reads four
    // bytes to send one does (us, as above with 3 / 7 / 11 helpers: 2240 / 1480 / 1430).
    static constexpr int kHelpers = 7, kCopyHelpers = 3;

    std::mutex lock;
    std::condition_variable wake, wake_more;     // the first kCopyHelpers, and the others
    std::deque<Job> queue;
    std::atomic<int> queued{0};      // jobs in the queue, read without the lock
    std::atomic<int> transfers{0};   // under way
    unsigned begun = 0, begun_more = 0;    // transfers so far, and those that take every helper (lock held)
    bool called = false;             // every helper that sleeps has been notified (lock held)
    bool started = false;

    static Crew &instance()
    {
        static Crew *c = new Crew;   // never destroyed: its threads live as long as the process
        return *c;
    }
    void begin(bool more = false)
    {
        {
            std::lock_guard<std::mutex> hold(lock);
            transfers++;
            begun++;
            begun_more += more;
            called = true;
            if (!started) {
                started = true;
                const int have = processors(), helpers = have > 2 * kHelpers ? kHelpers : have > 4 ? kCopyHelpers : have - 1;
                try {
                    for (int i = 0; i < helpers; i++)
                        std::thread([this, i] { help(i >= kCopyHelpers); }).detach();
                } catch (const std::exception &) {   // no more threads to be had: the callers copy alone
                }
            }
        }
        wake.notify_all();
        if (more)
            wake_more.notify_all();
    }
    void end()
    {
        std::lock_guard<std::mutex> hold(lock);
        transfers--;
    }
    // Cut into jobs of `size` bytes (of whole rows).
    void push(char *dst, const char *src, size_t bytes, std::atomic<int> &left, const Quantized *codes = nullptr, float *scales = nullptr,
              size_t size = kJobBytes)
    {
        left.store((int)((bytes + size - 1) / size), std::memory_order_relaxed);
        std::lock_guard<std::mutex> hold(lock);
        for (size_t at = 0; at < bytes; at += size) {
            Job j = {dst, src + at, bytes - at < size ? bytes - at : size, &left, codes, scales};
            if (!codes) {
                j.dst = dst + at;
            } else if (dst) {
                j.dst = dst + at / codes->unit * codes->row;
                j.scales = scales ? scales + at / codes->unit : nullptr;
            }
            try {
                queue.push_back(j);
                queued++;
            } catch (const std::exception &) {
                run(j);
            }
        }
        if (!called) {       // one went to sleep since the transfer began
            called = true;
            wake.notify_all();
        }
    }
    static void run(const Job &j)
    {
        if (!j.codes) {
            memcpy(j.dst, j.src, j.bytes);
        } else {
            const Quantized &c = *j.codes;
            const float *x = reinterpret_cast<const float *>(j.src);
            const int64_t rows = (int64_t)(j.bytes / c.unit), cols = (int64_t)(c.unit / sizeof(float));
            int8_t *q = reinterpret_cast<int8_t *>(j.dst);
            if (!q)
                raise(j.scales, c.host->absmax(x, (int64_t)(j.bytes / sizeof(float))));
            else if (c.one)
                c.host->scaled(x, rows, cols, q, (int64_t)c.row, c.given);
            else
                c.host->rows(x, rows, cols, q, (int64_t)c.row, j.scales);
        }
        j.left->fetch_sub(1, std::memory_order_release);
    }
    static void raise(float *most, float v)
    {
        float seen;
        __atomic_load(most, &seen, __ATOMIC_RELAXED);
        while (v > seen && !__atomic_compare_exchange(most, &seen, &v, true, __ATOMIC_RELAXED, __ATOMIC_RELAXED))
            ;
    }
    bool work()
    {
        if (queued.load(std::memory_order_acquire) == 0)
            return false;
        Job j;
        {
            // (held for a few instructions: to be put to sleep for it, and woken, takes longer than a job)
            std::unique_lock<std::mutex> hold(lock, std::try_to_lock);
            for (int i = 0; i < 1000 && !hold; i++) {
                __builtin_ia32_pause();
                hold.try_lock();
            }
            if (!hold)
                hold.lock();
            if (queue.empty())
                return false;
            j = queue.front();
            queue.pop_front();
            queued--;
        }
        run(j);
        return true;
    }
    // The caller of a transfer copies too while it would otherwise wait.
    void finish(std::atomic<int> &left)
    {
        while (left.load(std::memory_order_acquire) != 0)
            if (!work())
                __builtin_ia32_pause();
    }
    void help(bool more)
    {
        unsigned seen = 0;
        double since = seconds();
        for (;;) {
            if (work()) {
                since = seconds();
                continue;
            }
            if (transfers.load(std::memory_order_acquire) > 0 && seconds() - since < kHelpersLook) {
                for (int i = 0; i < 16; i++)
                    __builtin_ia32_pause();
                continue;
            }
            std::unique_lock<std::mutex> hold(lock);
            if (more) {
                wake_more.wait(hold, [&] { return begun_more != seen; });
                seen = begun_more;
            } else {
                wake.wait(hold, [&] {
                    const bool stay = begun == seen && queue.empty();
                    if (stay)
                        called = false;
                    return !stay;
                });
                seen = begun;
            }
            since = seconds();
        }
    }
};

// Room for small uploads of `bytes` in all (with the gaps that put_small leaves), behind those before them in
// the current slot (one flag per slot and not one per upload).
size_t small_room(size_t bytes) { return (bytes + 15 + 255) & ~(size_t)255; }

int open_small(Ring *r, size_t room, hipStream_t st)
{
    int rc = VTL_HIP_OK;
    // When a download has waited for everything so far, the slot is filled from its start again:
    // staging memory that is still in the host's caches.
    if (single_stream() && r->uploads->done.load(std::memory_order_acquire) ==
                               r->uploads->enqueued.load(std::memory_order_relaxed))
        r->used = 0;
    if (r->used + room > kSlotBytes)
        rc = r->close(st);
    if (rc == VTL_HIP_OK && r->used == 0)
        rc = r->wait(r->slot, st);
    return rc;
}

// Copies bytes there, `skew` past a 16-byte boundary.
char *put_small(Ring *r, const void *src, size_t bytes, size_t skew)
{
    char *staged = r->at(r->slot) + r->used + skew;
    memcpy(staged, src, bytes);
    r->used += small_room(bytes);
    return staged;
}

// One upload of several.
struct Source : Quantized {
    void *dst;
    const void *src;
    size_t bytes;

    Source() = default;
    Source(void *dst_, const void *src_, size_t bytes_, const Quantized &codes = {}) : Quantized(codes), dst(dst_), src(src_), bytes(bytes_) {}
    // Where it lies in pinned memory, from a 64-byte boundary: bytes or codes as far behind a 16-byte boundary as on the
    // device, and behind the codes that the host has made the scales.
    size_t skew() const { return reinterpret_cast<uintptr_t>(host ? static_cast<void *>(q) : dst) & 15; }
    size_t codes_bytes() const { return bytes / unit * row; }
    size_t scales_at() const { return ((skew() + codes_bytes() + 15) & ~(size_t)15) + (reinterpret_cast<uintptr_t>(scale) & 15); }
    size_t link_bytes() const { return host ? codes_bytes() + (one ? 0 : bytes / unit * sizeof(float)) : bytes; }
    size_t staged_bytes() const { return host ? scales_at() + (one ? 0 : bytes / unit * sizeof(float)) : bytes; }
    // By the calling thread.
    void stage(char *staged) const
    {
        std::atomic<int> left{1};
        Crew::run({staged + skew(), static_cast<const char *>(src), bytes, &left, host ? this : nullptr,
                   host && !one ? reinterpret_cast<float *>(staged + scales_at()) : nullptr});
    }
    // The segments that carry it.
    int segments(char *staged, Segment *seg) const
    {
        seg[0] = host ? make_segment(q, staged + skew(), codes_bytes()) : make_segment(dst, staged + skew(), bytes);
        if (!host || one)
            return 1;
        seg[1] = make_segment(scale, staged + scales_at(), bytes / unit * sizeof(float));
        return 2;
    }
};

// What a launch carries: `staged` in pinned memory.
struct Load {
    RowsArgs rows = {};
    CopyArgs copy = {};

    // `staged`: 16-byte aligned
    void add(const Source &piece, char *staged)
    {
        if (!piece.unit || piece.host) {
            copy.count += piece.segments(staged, copy.seg + copy.count);
            return;
        }
        rows.rows[rows.count++] = {reinterpret_cast<const float *>(staged + piece.skew()), piece.q, piece.scale, (int)(piece.bytes / piece.unit)};
        rows.cols = (int)(piece.unit / sizeof(float));
    }
    int launch(unsigned blocks, const LinkSignals &signals, hipStream_t st)
    {
        if (rows.count == 0) {
            copy.signals = signals;
            hipLaunchKernelGGL(host_copy_kernel, dim3(blocks), dim3(512), 0, st, copy);
            return check_launch("host_copy_kernel");
        }
        rows.signals = signals;
        rows.copies = copy.count;
        for (int i = 0; i < copy.count; i++)
            rows.seg[i] = copy.seg[i];
        launch_upload_rows(rows, blocks, st);
        return check_launch("upload_rows_kernel");
    }
};

// Small uploads, kSmall bytes in all at most, in one launch.
int upload_small(Ring *r, const Source *from, int count, hipStream_t st)
{
    size_t bytes = 0, room = 0;
    for (int i = 0; i < count; i++) {
        bytes += from[i].link_bytes();
        room += small_room(from[i].staged_bytes());
    }
    int rc = open_small(r, room, st);
    if (rc != VTL_HIP_OK)
        return rc;
    CopyArgs g = {};
    for (int i = 0; i < count; i++) {
        char *const staged = r->at(r->slot) + r->used;
        from[i].stage(staged);
        r->used += small_room(from[i].staged_bytes());
        g.count += from[i].segments(staged, g.seg + g.count);
    }
    hipLaunchKernelGGL(host_copy_kernel, dim3(copy_blocks(bytes < kSmall ? bytes : kSmall - 1)), dim3(512), 0, st, g);
    rc = check_launch("host_copy_kernel");
    if (rc == VTL_HIP_OK)
        r->uploads->enqueued.fetch_add(1, std::memory_order_acq_rel);
    return rc;
}

// What goes up in pieces of at most a slot, and the launches that carry up to kMaxSegments pieces each: small ones first, so
// that the link does not wait for the host's first copy, then larger ones, because a launch costs the link about 3 us (one slot
// a launch 53.9 GB/s, four 56.1).  Beyond a slot half as large again each: the host copies what a launch carries
// during the one before, and is not twice as fast as the link.  (180 MB in launches of one slot 3310 us, so 3170; 2 MiB of two
// operands 88 -> 80.)
constexpr size_t kFirstLaunch = (size_t)512 << 10;

struct Pieces {
    struct Piece : Source {
        std::atomic<int> left{0};
        bool last_of_launch;
    };
    std::unique_ptr<Piece[]> piece;
    int count = 0;

    // `host`: the host makes codes of (some of) it, and not the link but the host is what it waits for: launches of one slot at most,
    // and ever smaller ones at the end, where the link has to carry what the threads made last.
    Pieces(const Source *from, int sources, bool host)
    {
        const size_t most = host ? kSlotBytes : kMaxSegments * kSlotBytes;
        const auto segments = [&](int s) { return from[s].host && !from[s].one ? 2 : 1; };   // (codes with a scale a row take two)
        for (int pass = 0; pass < 2; pass++) {
            size_t ahead = 0, launch = kFirstLaunch, room = launch;
            for (int s = 0; s < sources; s++)
                ahead += from[s].bytes;
            int n = 0, in_launch = 0;   // pieces, and segments of the launch that is being filled
            for (int s = 0; s < sources; s++)
                for (size_t at = 0; at < from[s].bytes;) {
                    if (in_launch == 0 && host)
                        room = ahead < 2 * kFirstLaunch ? ahead : ahead / 3 < kFirstLaunch ? kFirstLaunch : ahead / 3 < launch ? ahead / 3 : launch;
                    else if (in_launch == 0 && ahead < launch + launch / 2)   // no small launch at the end
                        room = ahead;
                    size_t take = from[s].bytes - at;
                    if (take > kSlotBytes)
                        take = kSlotBytes;
                    if (take > room)
                        take = room;
                    if (from[s].unit)   // (a slot has room for a row)
                        take = take < from[s].unit ? from[s].unit : take - take % from[s].unit;
                    if (pass) {
                        Source &p = piece[n];
                        p = from[s];
                        p.src = static_cast<const char *>(from[s].src) + at;
                        p.bytes = take;
                        if (p.unit) {
                            p.q += p.host ? at / p.unit * p.row : at / sizeof(float);
                            if (!p.one)
                                p.scale += at / p.unit;
                        } else {
                            p.dst = static_cast<char *>(from[s].dst) + at;
                        }
                    }
                    at += take;
                    ahead -= take;
                    room -= take < room ? take : room;
                    n++;
                    in_launch += segments(s);
                    const size_t unit = at < from[s].bytes ? from[s].unit : 0;   // of what comes next
                    const bool end = ahead == 0 || room < (unit ? unit : 1) ||
                                     in_launch + segments(at < from[s].bytes || s + 1 == sources ? s : s + 1) > kMaxSegments;
                    if (pass)
                        piece[n - 1].last_of_launch = end;
                    if (end) {
                        launch = launch < kSlotBytes ? 2 * launch : (launch + launch / 2) & ~(size_t)4095;
                        if (launch > most)
                            launch = most;
                        room = launch;
                        in_launch = 0;
                    }
                }
            if (!pass)
                piece.reset(new Piece[(size_t)n]);
            count = n;
        }
    }
};

// Of whole rows.
size_t job_bytes(size_t unit) { return unit > Crew::kJobBytes ? unit : Crew::kJobBytes - Crew::kJobBytes % unit; }

// The host threads fill slots while the link empties the ones before them.  launch(first, n, slot of the
// first, last): pieces first .. first + n - 1, in as many consecutive slots.
template <typename Launch>
int send_pieces(Ring *r, Pieces &c, hipStream_t st, Launch launch)   // between Crew::begin() and end()
{
    int rc = r->close(st);
    if (rc != VTL_HIP_OK)
        return rc;
    const int n = c.count, s0 = r->slot;
    Crew &crew = Crew::instance();
    int pushed = 0, issued = 0;
    while (issued < n && rc == VTL_HIP_OK) {
        int end = issued;
        while (!c.piece[end++].last_of_launch)
            ;
        // what this launch carries, and as much of the next ones as there are free slots for
        while (pushed < n && pushed - issued < kSlots) {
            const int slot = (s0 + pushed) % kSlots;
            if (!r->is_free(slot)) {
                if (pushed >= end)
                    break;
                if ((rc = r->wait(slot, st)) != VTL_HIP_OK)
                    break;
            }
            Pieces::Piece &p = c.piece[pushed];
            char *const staged = r->at(slot);
            if (p.host)
                crew.push(staged + p.skew(), static_cast<const char *>(p.src), p.bytes, p.left, &p,
                          p.one ? nullptr : reinterpret_cast<float *>(staged + p.scales_at()), job_bytes(p.unit));
            else
                crew.push(staged + p.skew(), static_cast<const char *>(p.src), p.bytes, p.left);
            pushed++;
        }
        for (int i = issued; i < end && rc == VTL_HIP_OK; i++)
            crew.finish(c.piece[i].left);
        if (rc == VTL_HIP_OK)
            rc = launch(issued, end - issued, (s0 + issued) % kSlots, end == n);
        if (rc == VTL_HIP_OK)
            issued = end;
    }
    for (int i = 0; i < pushed; i++)   // after a failure: nothing may still write to the slots
        crew.finish(c.piece[i].left);
    if (rc != VTL_HIP_OK)
        r->give_up(st);
    r->slot = (s0 + n) % kSlots;
    return rc;
}

// A transfer that host threads share, for the length of a scope.
struct CrewWork {
    Crew &crew = Crew::instance();
    explicit CrewWork(bool more) { crew.begin(more); }
    ~CrewWork() { crew.end(); }
    CrewWork(const CrewWork &) = delete;
    CrewWork &operator=(const CrewWork &) = delete;
};

int upload_large(Ring *r, const Source *from, int count, hipStream_t st, bool host = false)
{
    Pieces c(from, count, host);
    const CrewWork work(host && from[count - 1].bytes >= kManyHelpersFrom);
    return send_pieces(r, c, st, [&](int first, int n, int slot, bool last) {
        Load load;
        size_t bytes = 0;
        for (int i = 0; i < n; i++) {
            const Pieces::Piece &p = c.piece[first + i];
            load.add(p, r->at((slot + i) % kSlots));
            bytes += p.link_bytes();
        }
        const unsigned blocks = copy_blocks(bytes < kSmall ? bytes : kSmall - 1);
        const int rc = load.launch(blocks, r->signals_for(slot, blocks, last, false), st);
        if (rc == VTL_HIP_OK)
            r->launched(slot, n, blocks, last);
        return rc;
    });
}

// A large transfer the other way: pieces of a MiB, then twice as large each up to a slot.
struct Chunks {
    struct Chunk {
        size_t at, bytes;
        std::atomic<int> left{0};
    };
    std::unique_ptr<Chunk[]> chunk;
    int count = 0;

    Chunks(size_t bytes, size_t first)
    {
        for (int pass = 0; pass < 2; pass++) {
            size_t at = 0, size = first;
            int n = 0;
            while (at < bytes) {
                const size_t take = bytes - at < size ? bytes - at : size;
                if (pass) {
                    chunk[n].at = at;
                    chunk[n].bytes = take;
                }
                n++;
                at += take;
                size = size * 2 < kSlotBytes ? size * 2 : kSlotBytes;
            }
            if (!pass)
                chunk.reset(new Chunk[(size_t)n]);
            count = n;
        }
    }
};

// The other way round, into memory that the device cannot write itself.
int download_large(Ring *r, char *dst, const char *src, size_t bytes, hipStream_t st)
{
    int rc = r->close(st);
    if (rc != VTL_HIP_OK)
        return rc;
    const size_t skew = reinterpret_cast<uintptr_t>(src) & 15;
    Chunks c(bytes, (size_t)1 << 20);
    const int n = c.count, s0 = r->slot;
    Crew &crew = Crew::instance();
    crew.begin();
    int issued = 0, pushed = 0, finished = 0;   // chunks under way, handed to the threads, done
    while (finished < n && rc == VTL_HIP_OK) {
        while (rc == VTL_HIP_OK && issued < n && issued - finished < kSlots) {
            const int slot = (s0 + issued) % kSlots;
            if ((rc = r->wait(slot, st)) == VTL_HIP_OK)
                rc = r->launch(slot, r->at(slot) + skew, src + c.chunk[issued].at, c.chunk[issued].bytes, true, st);
            if (rc == VTL_HIP_OK)
                issued++;
        }
        if (rc == VTL_HIP_OK && pushed < issued) {
            const int slot = (s0 + pushed) % kSlots;
            if ((rc = r->wait(slot, st)) == VTL_HIP_OK) {
                crew.push(dst + c.chunk[pushed].at, r->at(slot) + skew, c.chunk[pushed].bytes, c.chunk[pushed].left);
                pushed++;
            }
        }
        while (finished < pushed && (pushed == issued || c.chunk[finished].left.load(std::memory_order_acquire) == 0))
            crew.finish(c.chunk[finished++].left);
    }
    for (; finished < pushed; finished++)
        crew.finish(c.chunk[finished].left);
    crew.end();
    r->slot = (s0 + n) % kSlots;
    return rc;
}

}  // namespace

// The host makes codes of f32 rows, and the link carries those: 180 MB of weights with their scales and the forward behind them 3640 -> 1480 us, 4 MiB
// of activations through three layers 208 -> 157, 200 KB 28.7 -> 25.4 (16 processors).  Only above so many processors that the
// caller and its helpers are about half of them: with fewer, memory is what a copy and the codes wait for alike (8 processors, GB/s of f32 by 4
// threads: copied 35, quantized 32; what one thread makes, up to kSmall, was not timed on such machines).
constexpr int kQuantizeProcessors = 2 * Crew::kHelpers;

const HostQuantizer *quantizer_to_use()
{
    static const bool many = processors() > kQuantizeProcessors;
    const int asked = tuning().host_quantize;
    return (asked < 0 ? many : asked != 0) ? host_quantizer() : nullptr;
}

void HostInput::release()
{
    if (!ring_)
        return;
    // counted only now, when the kernels that read the bytes are enqueued: a download that waits
    // from here on waits for them too
    Ring *r = static_cast<Ring *>(ring_);
    r->uploads->enqueued.fetch_add(1, std::memory_order_acq_rel);
    r->lock.unlock();
    ring_ = nullptr;
    data = nullptr;
}

// The lock of the ring is held until then, so that no other transfer closes the slot before.
bool HostInput::stage(const void *src, size_t bytes)
try {
    if (!single_stream() || bytes > kSmall)
        return false;
    Ring *r = ring_of_current_device();
    if (!r)
        return false;
    r->lock.lock();
    if (open_small(r, small_room(bytes), current_stream()) != VTL_HIP_OK) {
        r->lock.unlock();
        return false;
    }
    ring_ = r;
    data = put_small(r, src, bytes, 0);
    return true;
} catch (const std::exception &) {
    return false;
}

bool HostInput::stage_codes(const float *src, int64_t rows, int64_t cols, int per_row, int64_t row)
try {
    const HostQuantizer *host = quantizer_to_use();
    const size_t codes = ((size_t)rows * (size_t)row + 15) & ~(size_t)15, room = small_room(codes + (size_t)rows * sizeof(float));
    if (!host || !single_stream() || rows < 1 || cols < 1 || row < cols || room > kSmall)
        return false;
    Ring *r = ring_of_current_device();
    if (!r)
        return false;
    r->lock.lock();
    if (open_small(r, room, current_stream()) != VTL_HIP_OK) {
        r->lock.unlock();
        return false;
    }
    ring_ = r;
    char *const staged = r->at(r->slot) + r->used;
    float *const s = reinterpret_cast<float *>(staged + codes);
    if (per_row) {
        host->rows(src, rows, cols, reinterpret_cast<int8_t *>(staged), row, s);
    } else {
        *s = host->scale(host->absmax(src, rows * cols));
        host->scaled(src, rows, cols, reinterpret_cast<int8_t *>(staged), row, *s);
    }
    r->used += room;
    data = staged;
    scales = s;
    return true;
} catch (const std::exception &) {
    return false;
}

bool upload_two(void *dst0, const void *src0, size_t bytes0, void *dst1, const void *src1, size_t bytes1, int &status)
try {
    if (!bytes0 || !bytes1 || !single_stream())
        return false;
    const OwnerDevice owner(dst0, dst1);
    Ring *r = owner.kernels() ? ring_of_current_device() : nullptr;
    if (!r)
        return false;
    const Source from[2] = {{dst0, src0, bytes0}, {dst1, src1, bytes1}};
    std::lock_guard<std::mutex> hold(r->lock);
    // One launch for both saves its 3 us while they are small; from there on the first is on the link while the host copies
    // the second, and what one host thread copies well needs no others (f32 products, together and in turn: 700 x 1024 x 200 129 and
    // 122 us, 512 x 512 x 300 87 and 83, 1024 x 1000 x 128 139 and 136; 1024 x 1001 x 64 115 and 117).
    // With little of one there is nothing to overlap (a bias behind its weights; of 512 x 512, 1 MiB exactly, 74.0 us together, 76.5 in turn).
    const size_t all = bytes0 + bytes1, less = bytes0 < bytes1 ? bytes0 : bytes1;
    if (all <= kUploadTogether || (all - less <= kSmall && less <= kWithAnother)) {
        status = upload_small(r, from, 2, current_stream());
    } else if (bytes0 <= kSmall && bytes1 <= kSmall) {
        status = upload_small(r, from, 1, current_stream());
        if (status == VTL_HIP_OK)
            status = upload_small(r, from + 1, 1, current_stream());
    } else {
        status = upload_large(r, from, 2, current_stream());
    }
    return true;
} catch (const std::exception &) {
    status = VTL_HIP_ERR_OUT_OF_MEMORY;
    return true;
}

bool upload_together(const HostUpload *uploads, int count, int &status)
try {
    if (count < 1 || count > kMaxSegments || !single_stream())
        return false;
    Source from[kMaxSegments];
    size_t bytes = 0;
    for (int i = 0; i < count; i++) {
        from[i] = {uploads[i].dst, uploads[i].src, uploads[i].bytes};
        bytes += uploads[i].bytes;
    }
    if (bytes > kUploadTogether)
        return false;
    const OwnerDevice owner(uploads[0].dst, uploads[count - 1].dst);
    Ring *r = owner.kernels() ? ring_of_current_device() : nullptr;
    if (!r)
        return false;
    std::lock_guard<std::mutex> hold(r->lock);
    status = upload_small(r, from, count, current_stream());
    return true;
} catch (const std::exception &) {
    status = VTL_HIP_ERR_OUT_OF_MEMORY;
    return true;
}

// Rows over the link as codes, and (extra_bytes of them) something copied with them; false: to be made in two steps.
bool upload_rows(const float *src, int64_t rows, int64_t cols, int8_t *q, float *scale, void *extra_dst, const void *extra_src,
                 size_t extra_bytes, int &status)
try {
    hipStream_t st = current_stream();
    const bool one_stream = single_stream();
    if (rows < 1 || rows > 0x7fffffff || cols < kRowsLeastCols || cols > kRowsMostCols || cols % 4 ||
        (size_t)rows * (size_t)cols * sizeof(float) < kRowsFrom || (reinterpret_cast<uintptr_t>(q) & 3) || (!one_stream && stream_is_capturing(st)))
        return false;
    const OwnerDevice owner(q, extra_bytes ? extra_dst : nullptr);
    Ring *r = owner.kernels() && owner.holds(scale) ? ring_of_current_device() : nullptr;
    if (!r)
        return false;
    const size_t unit = (size_t)cols * sizeof(float);
    const Quantized codes = {q, scale, unit};
    const Source from[2] = {{nullptr, src, (size_t)rows * unit, codes}, {extra_dst, extra_src, extra_bytes}};
    const int count = extra_bytes ? 2 : 1;
    std::lock_guard<std::mutex> hold(r->lock);
    status = upload_large(r, from, count, st);
    if (status == VTL_HIP_OK && !one_stream && hipStreamSynchronize(st) != hipSuccess)   // the ring's slots are shared by all streams
        status = record_hip_error(hipErrorUnknown, "upload_rows_kernel");
    return true;
} catch (const std::exception &) {
    status = VTL_HIP_ERR_OUT_OF_MEMORY;
    return true;
}

bool host_makes_codes(int64_t rows, int64_t cols, int64_t row)
{
    // (a slot has room for a row, and for the codes and scales of as many bytes of f32)
    return rows >= 1 && cols >= kCodesLeastCols && (size_t)cols * sizeof(float) <= kSlotBytes && row >= cols &&
           (size_t)row + sizeof(float) <= (size_t)cols * sizeof(float) && quantizer_to_use() &&
           (single_stream() || !stream_is_capturing(current_stream()));
}

// A row costs the host's units two divisions and two ends that are no whole vectors beside its values: up to kSmall, which one thread makes, that of short rows outweighs
// what the link saves, and that of rows of fewer than 32 values for several threads too.  A layer's weights and a small forward, parts of the time with the upload that was
// there before, by the device and by the host: scales per row, from 16 K codes on, 16 to 31 values 0.97 and 1.21 to 1.65, 32 to 63 0.97 and 1.05 to 1.40, 64 to 127 0.97 and
// 0.96 to 1.09, 128 to 191 0.96 and 0.99, whole steps of 64 of them 0.97 and 0.94, 192 to 255 0.96 and 0.95, 256 and more 0.96 and 0.93; one scale, 16 to 31 values 0.93 and
// 0.95, from 64 K codes on 0.96 and 1.03, 32 to 63 0.95 and 0.92.  Forward, scales per row: 178 x 160 26.9 us before, 30.3 by the host, 1770 x 48 33.3 and 40.7, 185 x 196 22.5
// and 24.0; beyond kSmall 16 to 31 values 1 and 1.06 to 1.19, 32 to 63 1 and 0.96.
bool rows_long_enough(int64_t rows, int64_t cols, int per_row)
{
    const size_t codes = (size_t)rows * (size_t)cols;
    if (tuning().host_quantize == 1 || codes <= (size_t)(per_row && cols < 32 ? 8 : 16) << 10)
        return true;
    if (!per_row || codes * sizeof(float) > kSmall)
        return cols >= 32;
    return cols >= 192 || (cols >= 128 && cols % 64 == 0);
}

bool upload_codes(const float *src, int64_t rows, int64_t cols, int per_row, int8_t *q, int64_t row, float *scale, void *extra_dst,
                  const void *extra_src, size_t extra_bytes, int &status)
try {
    if (!host_makes_codes(rows, cols, row) || extra_bytes > kWithAnother)
        return false;
    const HostQuantizer *host = quantizer_to_use();
    hipStream_t st = current_stream();
    const bool one_stream = single_stream();
    const size_t unit = (size_t)cols * sizeof(float), bytes = (size_t)rows * unit;
    const OwnerDevice owner(q, extra_bytes ? extra_dst : nullptr);
    Ring *r = owner.kernels() && owner.holds(scale) ? ring_of_current_device() : nullptr;
    if (!r)
        return false;
    Quantized codes = {q, scale, unit, host, (size_t)row, !per_row};
    std::lock_guard<std::mutex> hold(r->lock);
    std::unique_ptr<CrewWork> work;        // of the scale of all rows
    const char *const x = reinterpret_cast<const char *>(src);
    if (bytes > kSmall && !per_row)
        work.reset(new CrewWork(bytes >= kManyHelpersFrom));
    float most = 0.0f;
    if (!per_row) {
        if (work) {
            std::atomic<int> left{0};
            work->crew.push(nullptr, x, bytes, left, &codes, &most);
            work->crew.finish(left);
        } else {
            most = host->absmax(src, rows * cols);
        }
        codes.given = host->scale(most);
    }
    // the scale of all rows and the extra bytes in front: what the host makes last is then carried by a small launch
    Source from[3];
    int count = 0;
    if (extra_bytes)
        from[count++] = {extra_dst, extra_src, extra_bytes};
    if (!per_row)
        from[count++] = {scale, &codes.given, sizeof(float)};
    from[count++] = {nullptr, src, bytes, codes};
    status = bytes > kSmall ? upload_large(r, from, count, st, true) : upload_small(r, from, count, st);
    if (status == VTL_HIP_OK && !one_stream && hipStreamSynchronize(st) != hipSuccess)   // the ring's slots are shared by all streams
        status = record_hip_error(hipErrorUnknown, "host_copy_kernel");
    return true;
} catch (const std::exception &) {
    status = VTL_HIP_ERR_OUT_OF_MEMORY;
    return true;
}

void *HostResult::begin(void *dst, size_t bytes, size_t most)
{
    if (bytes == 0 || bytes > most || nafter_ == kParts || (!single_stream() && stream_is_capturing(current_stream())))
        return nullptr;
    const bool direct = (reinterpret_cast<uintptr_t>(dst) & 15) == 0 && bytes > 4096 && in_pinned_pool(dst, bytes);
    const size_t take = (bytes + 255) & ~(size_t)255;
    if (!direct && staged_ + take > kLaneStage)
        return nullptr;
    if (!lane_) {
        Lane *lane = nullptr;
        if (lease_lane(lane) != VTL_HIP_OK)
            return nullptr;
        lane_ = lane;
    }
    if (direct) {
        after_[nafter_++] = {dst, nullptr, bytes};
        return dst;
    }
    char *stage = static_cast<Lane *>(lane_)->stage + staged_;
    after_[nafter_++] = {dst, stage, bytes};
    staged_ += take;
    return stage;
}

void HostResult::attach(DoneSignal &signal, unsigned blocks)
{
    Lane *lane = static_cast<Lane *>(lane_);
    signal = lane->signal.next(blocks);
    lane->signal.launched(blocks);
    uploads_ = g_uploads[lane->device].enqueued.load(std::memory_order_acquire);
    attached_ = true;
}

int HostResult::finish()
{
    Lane *lane = static_cast<Lane *>(lane_);
    hipStream_t st = current_stream();
    const bool one_stream = single_stream();
    int rc = VTL_HIP_OK;
    if (!attached_ && one_stream) {
        CopyArgs g = {};
        attach(g.signals.done, 1);
        g.signals.to_host = 1;
        hipLaunchKernelGGL(host_copy_kernel, dim3(1), dim3(64), 0, st, g);
        rc = check_launch("host_copy_kernel");
    }
    if (rc == VTL_HIP_OK && attached_)
        rc = wait_behind(lane, uploads_, one_stream, st);
    else if (rc == VTL_HIP_OK)   // a release has waited for the device, or will: no launch more to raise a flag
        VTL_HIP_TRY(hipStreamSynchronize(st));
    if (rc != VTL_HIP_OK)
        return rc;
    for (int i = 0; i < nafter_; i++)
        if (after_[i].stage)
            memcpy(after_[i].dst, after_[i].stage, after_[i].bytes);
    return_lane(lane);
    lane_ = nullptr;
    return VTL_HIP_OK;
}

// After a failure launches may still write the results: they are waited for.  The lane goes back where its counter and flag are
// known, no launch having been given its signal, or that launch having raised it; else it is left alone.
HostResult::~HostResult()
{
    if (!lane_)
        return;
    Lane *lane = static_cast<Lane *>(lane_);
    const bool ended = hipStreamSynchronize(current_stream()) == hipSuccess;
    (void)hipGetLastError();
    if (!ended || (attached_ && !lane->signal.raised()))
        return;
    try {
        return_lane(lane);
    } catch (const std::exception &) {   // no room in the list
    }
}

void trim_pinned_pool()
{
    PinnedPool &p = pinned_pool();
    std::vector<void *> out;
    {
        std::lock_guard<std::mutex> hold(p.lock);
        for (auto &e : p.free_list)
            out.insert(out.end(), e.second.begin(), e.second.end());
        p.free_list.clear();
        p.idle_bytes = 0;
    }
    for (void *b : out)
        (void)hipHostFree(b);
    (void)hipGetLastError();
}

}  // namespace vtlhip

using namespace vtlhip;

extern "C" {

int vtl_hip_host_alloc(void **hptr, size_t bytes)
try {
    if (!hptr || bytes == 0)
        return VTL_HIP_ERR_INVALID_ARG;
    *hptr = nullptr;
    PinnedPool &p = pinned_pool();
    const size_t cls = size_class(bytes < 4096 ? 4096 : bytes);
    {
        std::lock_guard<std::mutex> hold(p.lock);
        if (p.live_bytes + cls > kPinnedLiveMost)
            return VTL_HIP_ERR_OUT_OF_MEMORY;
        p.live_bytes += cls;
        auto it = p.free_list.find(cls);
        if (it != p.free_list.end() && !it->second.empty()) {
            *hptr = it->second.back();
            it->second.pop_back();
            p.idle_bytes -= cls;
            p.live[reinterpret_cast<uintptr_t>(*hptr)] = cls;
            return VTL_HIP_OK;
        }
    }
    const hipError_t e = hipHostMalloc(hptr, cls, hipHostMallocDefault);
    std::lock_guard<std::mutex> hold(p.lock);
    if (e != hipSuccess) {
        p.live_bytes -= cls;
        *hptr = nullptr;
        return record_hip_error(e, "hipHostMalloc");
    }
    p.live[reinterpret_cast<uintptr_t>(*hptr)] = cls;
    return VTL_HIP_OK;
} catch (const std::exception &) {
    if (*hptr) {
        PinnedPool &p = pinned_pool();
        std::lock_guard<std::mutex> hold(p.lock);
        p.live_bytes -= size_class(bytes < 4096 ? 4096 : bytes);
        (void)hipHostFree(*hptr);
        *hptr = nullptr;
    }
    return VTL_HIP_ERR_OUT_OF_MEMORY;
}

int vtl_hip_host_free(void *hptr)
try {
    if (!hptr)
        return VTL_HIP_OK;
    PinnedPool &p = pinned_pool();
    {
        std::lock_guard<std::mutex> hold(p.lock);
        auto it = p.live.find(reinterpret_cast<uintptr_t>(hptr));
        if (it == p.live.end())
            return VTL_HIP_ERR_INVALID_ARG;
        const size_t cls = it->second;
        p.live.erase(it);
        p.live_bytes -= cls;
        if (p.idle_bytes + cls <= kPinnedIdleMost) {
            p.free_list[cls].push_back(hptr);
            p.idle_bytes += cls;
            return VTL_HIP_OK;
        }
    }
    VTL_HIP_TRY(hipHostFree(hptr));
    return VTL_HIP_OK;
} catch (const std::exception &) {
    return VTL_HIP_ERR_OUT_OF_MEMORY;
}

int vtl_hip_upload(void *dst_device, const void *src_host, size_t bytes)
try {
    if (bytes == 0)
        return VTL_HIP_OK;
    if (!dst_device || !src_host)
        return VTL_HIP_ERR_INVALID_ARG;
    hipStream_t st = current_stream();
    const OwnerDevice owner(dst_device);
    const bool one_stream = single_stream();
    if (owner.kernels() && (one_stream || !stream_is_capturing(st))) {
        Ring *r = ring_of_current_device();
        if (r) {
            std::lock_guard<std::mutex> hold(r->lock);
            const Source from = {dst_device, src_host, bytes};
            const int rc = bytes <= kSmall ? upload_small(r, &from, 1, st) : upload_large(r, &from, 1, st);
            if (rc != VTL_HIP_OK || one_stream)
                return rc;
            // the ring's slots are shared by all streams
            VTL_HIP_TRY(hipStreamSynchronize(st));
            return VTL_HIP_OK;
        }
    }
    VTL_HIP_TRY(hipMemcpyAsync(dst_device, src_host, bytes, hipMemcpyHostToDevice, st));
    VTL_HIP_TRY(hipStreamSynchronize(st));
    return VTL_HIP_OK;
} catch (const std::exception &) {
    return VTL_HIP_ERR_OUT_OF_MEMORY;
}

int vtl_hip_memcpy_h2d(void *dst_device, const void *src_host, size_t bytes)
try {
    if (bytes == 0)
        return VTL_HIP_OK;
    if (!dst_device || !src_host)
        return VTL_HIP_ERR_INVALID_ARG;
    hipStream_t st = current_stream();
    const size_t skew = reinterpret_cast<uintptr_t>(dst_device) & 15;
    const OwnerDevice owner(dst_device);
    if (!owner.kernels() || bytes + skew > kLaneStage || stream_is_capturing(st)) {
        const int rc = vtl_hip_upload(dst_device, src_host, bytes);
        if (rc != VTL_HIP_OK)
            return rc;
        VTL_HIP_TRY(hipStreamSynchronize(st));
        return VTL_HIP_OK;
    }
    Lane *lane = nullptr;
    int rc = lease_lane(lane);
    if (rc != VTL_HIP_OK)
        return rc;
    memcpy(lane->stage + skew, src_host, bytes);
    CopyArgs g = {};
    g.seg[0] = make_segment(dst_device, lane->stage + skew, bytes);
    g.count = 1;
    rc = copy_and_wait(g, bytes, lane, st);
    if (rc == VTL_HIP_OK)
        return_lane(lane);
    return rc;
} catch (const std::exception &) {
    return VTL_HIP_ERR_OUT_OF_MEMORY;
}

int vtl_hip_download(int count, void *const *dst_host, const void *const *src_device, const size_t *bytes)
try {
    if (count < 0 || (count > 0 && (!dst_host || !src_device || !bytes)))
        return VTL_HIP_ERR_INVALID_ARG;
    const void *first = nullptr;
    for (int i = 0; i < count; i++) {
        if (bytes[i] && (!dst_host[i] || !src_device[i]))
            return VTL_HIP_ERR_INVALID_ARG;
        if (!first && bytes[i])
            first = src_device[i];
    }
    if (!first)
        return VTL_HIP_OK;
    const OwnerDevice owner(first);
    for (int i = 0; i < count; i++)
        if (bytes[i] && src_device[i] != first && !owner.holds(src_device[i])) {   // of several devices: one by one
            int rc = VTL_HIP_OK;
            for (int k = 0; k < count && rc == VTL_HIP_OK; k++)
                rc = vtl_hip_download(1, dst_host + k, src_device + k, bytes + k);
            return rc;
        }
    hipStream_t st = current_stream();
    // What goes straight into pinned memory or fits a lane's staging buffer travels together, one
    // wait for all of it; anything else goes through the ring, one by one.
    CopyArgs g = {};
    struct { void *dst; const char *stage; size_t bytes; } after[kMaxSegments];
    int nafter = 0;
    size_t staged = 0, total = 0;
    Lane *lane = nullptr;
    const bool fast = owner.kernels() && (single_stream() || !stream_is_capturing(st));
    if (fast) {
        const int rc = lease_lane(lane);
        if (rc != VTL_HIP_OK)
            return rc;
    }
    int rc = VTL_HIP_OK;
    auto flush = [&] {
        if (g.count == 0)
            return;
        rc = copy_and_wait(g, total, lane, st);
        for (int k = 0; rc == VTL_HIP_OK && k < nafter; k++)
            memcpy(after[k].dst, after[k].stage, after[k].bytes);
        g.count = nafter = 0;
        staged = total = 0;
    };
    for (int i = 0; i < count && rc == VTL_HIP_OK; i++) {
        if (bytes[i] == 0)
            continue;
        const size_t skew = reinterpret_cast<uintptr_t>(src_device[i]) & 15;
        const bool direct = fast && (reinterpret_cast<uintptr_t>(dst_host[i]) & 15) == skew &&
                            bytes[i] > 4096 && in_pinned_pool(dst_host[i], bytes[i]);
        const size_t take = (bytes[i] + skew + 255) & ~(size_t)255;
        if (fast && (direct || take <= kLaneStage)) {
            if (g.count == kMaxSegments || (!direct && staged + take > kLaneStage)) {
                flush();
                if (rc != VTL_HIP_OK)
                    break;
            }
            char *to = direct ? static_cast<char *>(dst_host[i]) : lane->stage + staged + skew;
            g.seg[g.count++] = make_segment(to, src_device[i], bytes[i]);
            total += bytes[i];
            if (!direct) {
                after[nafter++] = {dst_host[i], to, bytes[i]};
                staged += take;
            }
        } else {
            Ring *r = fast ? ring_of_current_device() : nullptr;
            if (r) {
                std::lock_guard<std::mutex> hold(r->lock);
                rc = download_large(r, static_cast<char *>(dst_host[i]), static_cast<const char *>(src_device[i]),
                                    bytes[i], st);
            } else {
                hipError_t e = hipMemcpyAsync(dst_host[i], src_device[i], bytes[i], hipMemcpyDeviceToHost, st);
                if (e == hipSuccess)
                    e = hipStreamSynchronize(st);
                if (e != hipSuccess)
                    rc = record_hip_error(e, "hipMemcpyAsync(device to host)");
            }
        }
    }
    if (rc == VTL_HIP_OK)
        flush();
    if (lane) {
        if (rc == VTL_HIP_OK)
            return_lane(lane);   // after a failure its counter and flag are unknown: it is left alone
    }
    return rc;
} catch (const std::exception &) {
    return VTL_HIP_ERR_OUT_OF_MEMORY;
}

int vtl_hip_memcpy_d2h(void *dst_host, const void *src_device, size_t bytes)
{
    return vtl_hip_download(1, &dst_host, &src_device, &bytes);
}

}  // extern "C"
