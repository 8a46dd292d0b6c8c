// Shared declarations of libvtlhip.so (gfx950 only).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "vtl_hip.h"

namespace vtlhip {

// Stream every compute entry point enqueues on (nullptr = the null stream).
hipStream_t current_stream();

// True while no thread has named a stream of its own with vtl_hip_set_stream and memory of one
// device only has been asked for: all of the library's work is on one null stream and therefore in one order.
bool single_stream();

// Called with the device that memory is asked for on.
void note_device(int dev);

// The device whose memory a copy touches.  A copy takes memory of any device, whichever is current: on
// the null stream the owner is made current for the object's life, so that the copy comes behind the work
// enqueued there; a stream of the caller's stays where it is, and the copy is left to the runtime.
class OwnerDevice {
public:
    // Memory of two devices (`also` set and elsewhere) is left to the runtime too.
    explicit OwnerDevice(const void *memory, const void *also = nullptr);
    ~OwnerDevice();
    OwnerDevice(const OwnerDevice &) = delete;
    OwnerDevice &operator=(const OwnerDevice &) = delete;
    bool kernels() const { return kernels_; }         // whether kernels on the current stream can access the memory
    bool holds(const void *memory) const;             // whether this memory has the same owner

private:
    int owner_ = -1, back_ = -1;
    bool kernels_ = true;
};

// Whether memory of `a_bytes` from a and of `b_bytes` from b meet.
inline bool meet(const void *a, size_t a_bytes, const void *b, size_t b_bytes)
{
    const uintptr_t pa = reinterpret_cast<uintptr_t>(a), pb = reinterpret_cast<uintptr_t>(b);
    return a && b && pa < pb + b_bytes && pb < pa + a_bytes;
}

// Whether `st` is being captured into a graph (true also when that cannot be found out).
bool stream_is_capturing(hipStream_t st);

// hipMalloc; gives the idle blocks of vtl_hip_malloc's pool back to the driver and tries again
// when memory has run out.
hipError_t malloc_or_trim(void **ptr, size_t bytes);

// The size that a pooled block of `bytes` gets (memory.hip), and giving back the idle pinned
// blocks of vtl_hip_host_alloc (host_copy.hip).
size_t size_class(size_t bytes);
void trim_pinned_pool();

// Records a failed HIP runtime call for vtl_hip_last_error() and maps it to a
// status code of the C ABI.
int record_hip_error(hipError_t e, const char *what);

// Checks the launch that was just made.
int check_launch(const char *kernel_name);

// A small host array in pinned memory, for kernels that can take their input over the link themselves instead
// of behind a copy (the L2 keeps what comes over the link for the length of a launch, so workgroups that all read it
// share one transfer per XCD).  The bytes stay until release() and until the work enqueued before that is done.  No
// vtl_hip_upload in between on the same thread.
struct HostInput {
    const void *data = nullptr;
    // False when the bytes have to be uploaded instead: too many, or streams of the caller's.
    bool stage(const void *src, size_t bytes);
    // As codes and scales (data, scales), made by the host as upload_codes has them made.
    bool stage_codes(const float *src, int64_t rows, int64_t cols, int per_row, int64_t row);
    const float *scales = nullptr;
    void release();
    HostInput() = default;
    ~HostInput() { release(); }
    HostInput(const HostInput &) = delete;
    HostInput &operator=(const HostInput &) = delete;

private:
    void *ring_ = nullptr;
};

// Two uploads as vtl_hip_upload makes them, which share their launches; false: to be made one by one.
bool upload_two(void *dst0, const void *src0, size_t bytes0, void *dst1, const void *src1, size_t bytes1, int &status);

// Up to four small uploads, kUploadTogether bytes in all, to one device in one launch; false: to be made one by one.
constexpr size_t kUploadTogether = (size_t)640 << 10;
struct HostUpload {
    void *dst;
    const void *src;
    size_t bytes;   // not 0
};
bool upload_together(const HostUpload *uploads, int count, int &status);

// Rows that are quantized as they arrive, one scale each, and extra bytes copied with them; false: to be uploaded and quantized.
bool upload_rows(const float *src, int64_t rows, int64_t cols, int8_t *q, float *scale, void *extra_dst, const void *extra_src,
                 size_t extra_bytes, int &status);

// Rows that the host's threads quantize in front of the link, which then carries a quarter of their bytes: per_row, or with one
// scale; `row` bytes from one row of codes to the next (zeros behind the codes).  False: to be quantized by the device, as always
// where the host does not make codes of such rows.
bool host_makes_codes(int64_t rows, int64_t cols, int64_t row);
// Whether such rows are long enough for the host to be the faster.
bool rows_long_enough(int64_t rows, int64_t cols, int per_row);
bool upload_codes(const float *src, int64_t rows, int64_t cols, int per_row, int8_t *q, int64_t row, float *scale, void *extra_dst,
                  const void *extra_src, size_t extra_bytes, int &status);

// How a launch tells the host that its results are there: every workgroup counts itself when its stores are
// complete, and the one that reaches the target raises the flag.  No flag: nothing to tell.
struct DoneSignal {
    unsigned *counter;   // in device memory
    unsigned target;
    unsigned value;
    unsigned *flag;      // in pinned host memory
};

// The result of a whole host-to-host call, written over the link by the launch that computes it instead of by a
// copy behind it (64 x 256 f32: 0.8 us more than to device memory, where the copy is a launch of 4.3; 256 x 1024 f32 19 against
// 23, 512 x 512 f64 36 against 43).  Kernels that store whole cache lines, or a few pieces of lines, store them through
// to the host and raise the flag (attach): a part of a line crosses the link alone (512 x 512 doubles in
// halves of lines: 17 ms).  When none did, ordinary stores went to the host's memory by way of the caches and finish() lets a small
// launch raise the flag behind them; a fence in every workgroup instead would write the caches back each time (7.6 us with
// 256 of them).
class HostResult {
public:
    HostResult() = default;
    ~HostResult();
    HostResult(const HostResult &) = delete;
    HostResult &operator=(const HostResult &) = delete;
    // Pinned memory to write a result of `bytes` to that finish() leaves in dst (up to kParts of them); nullptr:
    // compute in device memory and download, as with more than `most`.
    void *begin(void *dst, size_t bytes, size_t most);
    // For the last launch of the call, right before it, with its number of workgroups.
    void attach(DoneSignal &signal, unsigned blocks);
    // After the release() of an input that the launch with the signal has read.
    bool attached() const { return attached_; }
    void input_released() { uploads_++; }
    // Waits for the results and hands them over.
    int finish();

private:
    struct Part {
        void *dst;
        const char *stage;
        size_t bytes;
    };
    static constexpr int kParts = 3;
    void *lane_ = nullptr;
    Part after_[kParts];
    int nafter_ = 0;
    size_t staged_ = 0;
    uint64_t uploads_ = 0;
    bool attached_ = false;
};

#ifdef __HIPCC__
// A result element: with a signal to raise it goes through the caches to where the host sees it.
template <typename T>
__device__ __forceinline__ void store_result(T *p, T v, const DoneSignal &done)
{
    if (done.flag)
        __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    else
        *p = v;
}

// 8 or 16 bytes of a result of less than 4 GiB, `off` bytes from its start and aligned as an element is: one store, through
// the caches.  (By way of a builtin and not of inline assembly: the compiler puts the wait states in that gfx950 wants
// between a wide store, or the MFMA before it, and the instructions that touch the same registers.  Behind a store of 16 bytes
// it does so only where the scalar offset is a constant, as here; store_run in matmul_f64acc.hip, where it is a register, adds them.)
typedef unsigned Words2 __attribute__((ext_vector_type(2)));
typedef unsigned Words4 __attribute__((ext_vector_type(4)));
constexpr int kThrough = 17;   // sc0 sc1
__device__ __forceinline__ __amdgpu_buffer_rsrc_t result_buffer(void *out)
{
    return __builtin_amdgcn_make_buffer_rsrc(out, 0, 0xffffffff, 0x00027000);
}
__device__ __forceinline__ void store_through(void *out, unsigned off, Words2 v)
{
    __builtin_amdgcn_raw_buffer_store_b64(v, result_buffer(out), off, 0, kThrough);
}
template <int HOW = kThrough>
__device__ __forceinline__ void store_through(void *out, unsigned off, Words4 v)
{
    __builtin_amdgcn_raw_buffer_store_b128(v, result_buffer(out), off, 0, HOW);
}

// Called by every thread of a workgroup after its last store_result.  Those are written through, so their
// acknowledgement is enough to count on; the fence of the last workgroup covers results of launches before.
__device__ __forceinline__ void raise_when_last(const DoneSignal &done)
{
    if (!done.flag)
        return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x != 0)
        return;
    const unsigned before = __hip_atomic_fetch_add(done.counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (before + 1 == done.target) {
        __threadfence_system();
        __hip_atomic_store(done.flag, done.value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}
#endif

// Streaming copy kernel (quant.hip); false when alignment or size do not qualify.
bool launch_copy(void *dst, const void *src, size_t bytes, hipStream_t st);

// Device scratch owned by the library: per device three independent buffers
// (slot 0: split-K partial sums and partial column sums; slot 1: quantized
// activations staged between the two launches of a dynamic-quantization call;
// slot 2: int8 operands repacked to a row length the fast kernels take),
// grown on demand and kept until the process ends.  Kernels enqueued on the
// current stream may use a slot until the next call that asks for it; nullptr
// when the allocation fails.  While the current stream records a graph a slot
// is handed out only if it is already large enough (growing would free and
// allocate), and a buffer handed out then is never freed afterwards, because
// replays of the graph keep using its address: a later, larger request gets a
// new buffer and the old one stays allocated.
void *library_workspace(size_t bytes, int slot = 0);
// Why the last library_workspace() call of this thread returned nullptr
// (VTL_HIP_ERR_OUT_OF_MEMORY, or VTL_HIP_ERR_UNSUPPORTED when the request does
// not fit the static scratch or would have to allocate during a stream capture).
int workspace_status();

// A small index (0 .. kStreamSlots - 1) that belongs to `st` on the current device, for code
// that keeps a little state in device memory between its launches and must not share it with
// work that may run at the same time: the first kStreamSlots streams that ask get one each, for
// as long as the process lives (a stream handle that is reused inherits its predecessor's
// index, which is as good).  -1 when none is left, when the stream is being captured into a
// graph (a replay would meet the state of another moment) or when that cannot be found out.
constexpr int kStreamSlots = 16;
int stream_slot(hipStream_t st);

// Static per-device scratch for the entry point that allocates nothing, and the
// scope during which library_workspace() serves from it.  static_scratch()
// returns the device address of the current device's array (nullptr on error).
constexpr size_t kStaticScratchBytes = size_t(32) << 20;
void *static_scratch();
struct ScratchArena {
    char *base;
    size_t capacity, used = 0;
    ScratchArena(void *base_, size_t capacity_);
    ~ScratchArena();
    ScratchArena(const ScratchArena &) = delete;
    ScratchArena &operator=(const ScratchArena &) = delete;
};

// While one is alive, library_workspace() hands this thread blocks of its own instead of the library's: whole host calls run in
// several threads at once, and between two launches of one that meet in a slot another's may write it.  A released block's next owner
// comes behind these launches on the null stream; once the process has named a stream a release would wait for the
// device, and the library's buffers are what there is.
class CallScratch {
public:
    CallScratch();
    ~CallScratch();
    CallScratch(const CallScratch &) = delete;
    CallScratch &operator=(const CallScratch &) = delete;
    // nullptr: no memory
    void *take(size_t bytes, int slot);

private:
    void *own_[3] = {};
    size_t bytes_[3] = {};
};

// Whether this thread's scratch is the static one just now.
bool scratch_is_static();

// Per-row quantization into rows of ldq codes, zeros past the end (quant.hip); false when the sizes do not qualify.
bool launch_quantize_rows_padded(const float *x, int64_t rows, int cols, int8_t *q, int ldq, float *scale_out,
                                 hipStream_t st, int &status);

// vtl_hip_matmul_* without a transposed b.  `result`: c is its memory, and this is the call's last launch.
int matmul_to(HostResult *result, const float *a, const float *b, float *c, int m, int n, int k, int trans_a);
int matmul_to(HostResult *result, const double *a, const double *b, double *c, int m, int n, int k, int trans_a);
// dW = grad^T . x and, unless it is null, db = the column sums of grad.
int weight_gradients_to(HostResult *result, const float *grad, const float *x, float *dw, float *db, int m, int n, int k);
int weight_gradients_to(HostResult *result, const double *grad, const double *x, double *dw, double *db, int m, int n, int k);
// Those, and dX = grad . W, in one launch, the call's last, whose results are `result`'s memory; false: launch by launch.
bool gradients_in_one(HostResult *result, const float *grad, const float *x, const float *w, float *dx, float *dw, float *db, int m, int n,
                      int k, int &status);
bool gradients_in_one(HostResult *result, const double *grad, const double *x, const double *w, double *dx, double *dw, double *db, int m,
                      int n, int k, int &status);

// vtl_hip_linear_i8_f32 and vtl_hip_linear_i8_requant with the parameters of a layer, whose weights may have padded rows.
// `result`: Y is its memory.  `padded`: so have the codes A.
int layer_linear_i8_f32(const vtl_hip_layer &l, const int8_t *A, const float *sa, float *Y, int M, int relu,
                        HostResult *result = nullptr, bool padded = false);
// vtl_hip_layer_f32; of one row with one scale for the weights too.  `x_on_host`: X is in pinned memory (HostInput).
int layer_f32(const vtl_hip_layer &l, const float *X, float *Y, int M, int relu, void *workspace, size_t workspace_bytes,
              HostResult *result = nullptr, bool x_on_host = false);
// Whether layer_f32 has rows in device memory, or of a host call's input, in one launch (more than eight of them).
bool layer_takes_rows(const vtl_hip_layer &l, int M);
bool layer_takes_input(const vtl_hip_layer &l, int M);
int layer_linear_i8_requant(const vtl_hip_layer &l, const int8_t *A, const float *sa, int8_t *Yq, float *sy, int M,
                            int relu, bool padded = false);

// Tuning and test switches, taken from the environment once (first use) and
// again only when vtl_hip_reload_env() is called: the dispatch path of a launch
// reads this struct, never the environment.
struct Tuning {
    bool no_gemv = false;           // VTL_HIP_NO_GEMV: keep M <= 8 off the matrix-vector kernels
    int gemv_rows = -1;             // VTL_HIP_GEMV_ROWS: 1 / 0 force the few-token kernel on / off
    int gemm_small = -1;            // VTL_HIP_GEMM_SMALL: 1 / 0 force the small-product kernel on / off
    int ragged = -1;                // VTL_HIP_RAGGED: 1 / 0 force the kernels that take rows of any length as they are on / off
    int gemm_config = -1;           // VTL_HIP_GEMM_CONFIG "<tile index>,<splits>"
    int gemm_splits = 1;
    bool no_fused_requant = false;  // VTL_HIP_NO_FUSED_REQUANT: linear, then the row quantizer
    int requant_wide = 0;           // VTL_HIP_REQUANT_WIDE: 1 row maxima in the tile kernel + wide quantizer, 0 one workgroup per row
    bool quant_four_launches = false;  // VTL_HIP_QUANT_FOUR_LAUNCHES: whole-tensor quantize as clear + absmax + scale + quantize (tests)
    int quant_groups = 0;           // VTL_HIP_QUANT_GROUPS: workgroups of a whole-tensor quantize launch whatever streams there are (tests)
    bool no_fused_decode = false;   // VTL_HIP_NO_FUSED_DECODE: quantizer launch in front of the linear
    int stage_spin = 4096;          // VTL_HIP_STAGE_SPIN: polls a workgroup of the decode launch waits for the quantized rows (0: none, tests)
    int stream_weights_mib = 48;    // VTL_HIP_STREAM_WEIGHTS_MIB: weight matrices of this many MiB and more are read with non-temporal loads by the kernels for 2 to 32 rows (0: always)
    int skinny_tiled = -1;          // VTL_HIP_SKINNY_TILED: 1 / 0 force the 32x32-block weight-streaming kernel for M > 32
    int skinny_waves = 4;           // VTL_HIP_SKINNY_WAVES: 2, 4 or 8 waves (K ranges) per workgroup there
    int matmul_tile = 0;            // VTL_HIP_MATMUL_TILE: which kernel and tile the f64-accumulating matmul takes (matmul_f64acc.hip)
    int host_quantize = -1;         // VTL_HIP_HOST_QUANTIZE: 1 / 0 force rows in host memory to be quantized by the host's / the device's units; 2: by
                                    // the host's where it is faster, with any number of processors
    int backward_group = -1;        // VTL_HIP_BACKWARD_GROUP: 1 / 0 force a backward's gradients in one launch on (where it can be) / off
    int matmul_splits = -1;         // VTL_HIP_MATMUL_SPLITS: K ranges of the f64-accumulating matmul
};
const Tuning &tuning();

constexpr int kWave = 64;

}  // namespace vtlhip

#define VTL_HIP_TRY(expr)                                                  \
    do {                                                                   \
        hipError_t vtl_e_ = (expr);                                        \
        if (vtl_e_ != hipSuccess)                                          \
            return ::vtlhip::record_hip_error(vtl_e_, #expr);              \
    } while (0)
