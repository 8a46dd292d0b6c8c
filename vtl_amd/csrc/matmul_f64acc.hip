// Dense matmul with f64 products and sums on the gfx950 f64 matrix cores, for
// f32 and f64 tensors: the device form of la.matmul (la/la.v:38-55) and
// gate_matmul (autograd/gates_blas.v:6-23), which widen every operand to f64,
// multiply with a f64 GEMM and round the result once to the tensor's type.
// Also the unquantized Linear forward (nn/layers/linear_forward_f32.v:16-18)
// and LinearGate.backward (nn/gates/layers/linear.v:69-79) built on it.
//
// matmul_f64acc_direct_kernel takes operands from global memory straight to registers; choose_plan() picks its
// shape by estimated time.
#include <stdlib.h>

#include <type_traits>

#include "common.hpp"

namespace {

using vtlhip::check_launch;
using vtlhip::current_stream;

typedef double double4_t __attribute__((ext_vector_type(4)));

struct MatmulArgs {
    const void *A;      // trans_a == 0: [M,K] row-major, else [K,M]
    const void *B;      // trans_b == 0: [K,N] row-major, else [N,K]
    void *C;            // [M,N] row-major
    const void *bias;   // N values added after rounding to the output type, or nullptr
    int M, N, K;
    int relu;
    int slice_steps;    // steps of 16 of K in one grid.y slice
    double *partial;    // launches that slice K: [slices][M][N] unrounded sums, or [tail tile][slice][tile]; else nullptr
    int whole_tiles;    // with tail_slices > 1 the tiles from here on, the last round's, have K in that many slices
    int tail_slices;
    int fold_slices;    // > 1: K in so many slices (grid.y), whose sums the last workgroup of each tile adds up; partial: [tile][slice][tile]
    int fold_slot;      // which counters
    vtlhip::DoneSignal done;     // C is the memory of a whole host call's result
    vtlhip::HostResult *result;  // host side only
};

template <typename T>
struct alignas(16) Vec4 {
    T v[4];
};

// ---- operands straight from global memory --------------------------------------------------
// A wave owns 16 * TM x 16 * TN of C.  An f64 MFMA wants two values a lane every 64 cycles, so operands
// need neither LDS nor barriers: the tiles are small, K is cut over the WK waves of a workgroup (partial
// tiles meet in LDS) and, with few tiles, over grid.y.  With 64 x 64 tiles staged in LDS a wave had four MFMAs for every 4
// of K, 7 us at K = 256 and 14 us at K = 512 whatever else the chip did, and ragged sizes loaded
// element by element: 512^3 22.4 -> 8.8 us, 64 x 784 x 256 16.4 -> 5.5, 64 x 256 x 784 44 -> 7.5,
// 255 x 11007 x 4095 447 -> 367, 333 x 517 x 701 47 -> 13 (f32; f64 alike).
//
// What bounds a large product: nothing of the vector unit runs beside an f64 MFMA.  An instruction between two of them
// costs 11 cycles and each further one 5 to 7 (measured, one and two waves on a SIMD, conversions, integer
// and f32 operations alike), against 64 for the MFMA.  So the loop has no vector instruction but the
// conversions of f32 operands, all of a step's at once, and those are fewer the larger a wave's tile is:
// loads take a lane's offset that never changes and scalars for the rest (buffer loads), and a pair of columns at
// the odd edge of a matrix is moved, not chosen from.
//
// Steps of 16 of K are dealt out to the WK waves in turn.  In a step lane l holds four k for TM / 2 pairs of
// rows 2 * (l % 16) + {0, 1} of A and for TN / 2 such pairs of columns of B: 16-byte loads where K runs
// along memory, pairs of 32 neighbouring columns where it does not.  MFMA j of a step takes the j-th of
// each lane's four: which k they are is free as long as both operands agree.
// Vector loads need no more than the elements' own alignment on gfx950, so ragged rows take them too.  What K has beyond whole
// steps is the first one: loaded like any other, and what belongs to the second cleared.  (As a last step with checked
// loads, waited for one after another, it was as long as several: f32 256 x 11008 x 300 44.3 -> 39.5 us, 101 x 720 x 394 8.0 -> 6.9; f64
// 105 x 653 x 361 7.7 -> 6.8.)  CHECKED: every load is (a single row or column of a matrix that has to give pairs, rows
// too long for a lane's 32-bit offset); so it is below K = 16.
template <typename T>
constexpr int kRun = 16 / (int)sizeof(T);   // elements of a 16-byte load; the lane's four are those of each run of 4 * kRun

// The longest rows that offsets of 32 bits reach over.  Where K runs along them a wave covers up to 64; where it runs across
// them, a step's 16.  Neither limits how many rows there are: their first is a scalar.
template <typename T>
constexpr int kLongest64 = (int)(0xffffffffu / (64 * sizeof(T)));
template <typename T>
constexpr int kLongest16 = (int)(0xffffffffu / (16 * sizeof(T)));

// N elements at `off` bytes (a lane's own) + `along` from base, one load.
template <typename T, int N>
__device__ __forceinline__ void load_run(T (&out)[N], __amdgpu_buffer_rsrc_t base, unsigned off, unsigned along)
{
    typedef unsigned Two __attribute__((ext_vector_type(2)));
    typedef unsigned Four __attribute__((ext_vector_type(4)));
    constexpr int bytes = N * (int)sizeof(T);
    static_assert(bytes == 8 || bytes == 16, "one load");
    if constexpr (bytes == 16) {
        const Four v = __builtin_amdgcn_raw_buffer_load_b128(base, off, along, 0);
        __builtin_memcpy(out, &v, bytes);
    } else {
        const Two v = __builtin_amdgcn_raw_buffer_load_b64(base, off, along, 0);
        __builtin_memcpy(out, &v, bytes);
    }
}

template <bool THROUGH>
__device__ __forceinline__ void store_run(__amdgpu_buffer_rsrc_t base, unsigned off, unsigned along, float a, float b)
{
    typedef unsigned Two __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(Two{__float_as_uint(a), __float_as_uint(b)}, base, off, along, THROUGH ? vtlhip::kThrough : 0);
}

template <bool THROUGH>
__device__ __forceinline__ void store_run(__amdgpu_buffer_rsrc_t base, unsigned off, unsigned along, double a, double b)
{
    typedef unsigned Four __attribute__((ext_vector_type(4)));
    const unsigned long long ua = (unsigned long long)__double_as_longlong(a), ub = (unsigned long long)__double_as_longlong(b);
    __builtin_amdgcn_raw_buffer_store_b128(Four{(unsigned)ua, (unsigned)(ua >> 32), (unsigned)ub, (unsigned)(ub >> 32)}, base, off,
                                           along, THROUGH ? vtlhip::kThrough : 0);
    // A store of more than 8 bytes reads its registers for two more instructions.  The compiler keeps instructions that write them
    // away only where the offset is no scalar register; left to it, the next pair's first word was moved in behind the store, and
    // now and then went out with this one (dW 2625 x 3136 x 16: elements in even columns off by 1e-7 of themselves).
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 1");
    __builtin_amdgcn_sched_barrier(0);
}

// One pair of rows or columns of an operand for the lanes of a wave.
template <typename T, bool KROWS>
struct DirectOperand {
    const char *base;      // of the wave's rows or columns
    int64_t k_stride;      // bytes from one k to the next
    unsigned off[2];       // a lane's bytes from there, at k = 0: of its two rows, or of its pair

    // [MN, K], its rows mn[0] and mn[1], or [K, MN], its columns mn[0] and mn[0] + 1
    __device__ __forceinline__ DirectOperand(const T *p, int mn_total, int k_total, int mn_first, const int (&mn)[2], int kq)
    {
        if constexpr (KROWS) {
            base = reinterpret_cast<const char *>(p + (int64_t)mn_first * k_total);
            k_stride = (int)sizeof(T);
#pragma unroll
            for (int i = 0; i < 2; ++i)
                off[i] = ((unsigned)(mn[i] - mn_first) * (unsigned)k_total + (unsigned)(kRun<T> * kq)) * (unsigned)sizeof(T);
        } else {
            base = reinterpret_cast<const char *>(p);
            k_stride = (int64_t)mn_total * (int)sizeof(T);
            off[0] = off[1] = ((unsigned)(kRun<T> * kq) * (unsigned)mn_total + (unsigned)mn[0]) * (unsigned)sizeof(T);
        }
    }
    __device__ __forceinline__ void fetch(T (&out)[2][4], int k0) const
    {
        constexpr int VK = kRun<T>;
        const __amdgpu_buffer_rsrc_t at =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(base + k0 * k_stride), 0, 0xffffffff, 0x00027000);
#pragma unroll
        for (int q = 0; q < 4; q += VK) {
            if constexpr (KROWS) {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    T run[VK];
                    load_run<T, VK>(run, at, off[i], (unsigned)(4 * q) * (unsigned)sizeof(T));
#pragma unroll
                    for (int j = 0; j < VK; ++j)
                        out[i][q + j] = run[j];
                }
            } else {
#pragma unroll
                for (int j = 0; j < VK; ++j) {
                    T pair[2];
                    load_run<T, 2>(pair, at, off[0], (unsigned)(4 * q + j) * (unsigned)k_stride);
                    out[0][q + j] = pair[0];
                    out[1][q + j] = pair[1];
                }
            }
        }
    }
};

// Steps of 16 that K is.
__host__ __device__ __forceinline__ int steps_of(int k) { return (k >> 4) + ((k & 15) != 0); }

// The same with every load checked and no vector loads, at any size.
template <typename T, bool KROWS>
__device__ __forceinline__ void checked_fetch(T (&out)[2][4], const T *__restrict__ base, int mn_total, int k_total,
                                              const int (&mn)[2], int k0, int kq)
{
    constexpr int VK = kRun<T>;
#pragma unroll
    for (int q = 0; q < 4; q += VK)
#pragma unroll
        for (int j = 0; j < VK; ++j) {
            const int k = k0 + 4 * q + VK * kq + j;
#pragma unroll
            for (int i = 0; i < 2; ++i)
                out[i][q + j] = k < k_total ? base[KROWS ? (int64_t)mn[i] * k_total + k : (int64_t)k * mn_total + mn[i]] : T(0);
        }
}

// Two neighbours of a row from element `at` of out, aligned as one element is (written through, to a host call's result: a
// few MiB).
template <typename T>
__device__ __forceinline__ void store_pair(T *out, int64_t at, T a, T b, const vtlhip::DoneSignal &done)
{
    typedef T Two __attribute__((ext_vector_type(2), aligned(sizeof(T))));
    using Words = std::conditional_t<sizeof(T) == 4, vtlhip::Words2, vtlhip::Words4>;
    const Two v = {a, b};
    if (done.flag)   // waited for in raise_when_last
        vtlhip::store_through(out, (unsigned)at * (unsigned)sizeof(T), __builtin_bit_cast(Words, v));
    else
        *reinterpret_cast<Two *>(out + at) = v;
}

__device__ __forceinline__ void tile_of_block(int block, int tiles_m, int tiles_n, int &tm, int &tn)
{
    const int total = tiles_m * tiles_n;
    const int xcd = block & 7, over = total & 7;
    const int pid = xcd * (total >> 3) + min(xcd, over) + (block >> 3);
    const int group = 8 * tiles_n, first_m = (pid / group) * 8, gm = min(tiles_m - first_m, 8);
    tm = first_m + (pid % group) % gm;
    tn = (pid % group) / gm;
}

// The partial tiles of a workgroup whose waves cut K.
template <int WM, int WN, int WK, int TM, int TN>
struct PartialTiles {
    double at[WK > 1 ? WM * WN * WK : 1][WK > 1 ? 4 * TM * TN : 1][64];
};

// Slices of K that meet within a launch.  Each workgroup writes its sums through to memory (16 bytes a thread, whole lines), waits until that is
// acknowledged and counts itself at its tile; who completes the count reads the slices back, past the caches, adds them up in
// their order and leaves the counter at 0 for the next launch.  Nobody waits for another, and no fence writes a cache back.  A launch that adds them up
// instead is 3.4 to 4.7 us on the device, a gap, and 3.4 us on the host (us, with one and so: f32 64 x 256 x 2000 12.2 -> 8.0, 32 x 1024 x 1024 8.3 -> 6.8, 128 x 1024 x 4096
// 27.2 -> 24.2, f64 64 x 64 x 4096 16.4 -> 10.9, 64 x 1024 x 1024 11.5 -> 8.5).  The counters belong to a stream, whose launches follow one another.
constexpr int kFoldTiles = 1024, kFoldStride = 16;
__device__ unsigned g_fold_count[vtlhip::kStreamSlots * kFoldTiles * kFoldStride];

// Whether this workgroup, whose sums are written, is the last of its tile's.
__device__ __forceinline__ bool last_of_tile(const MatmulArgs &g, int block)
{
    __shared__ int s_last;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();   // every thread's are
    if (threadIdx.x == 0) {
        unsigned *const count = g_fold_count + ((int64_t)g.fold_slot * kFoldTiles + block) * kFoldStride;
        const bool last = __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == (unsigned)g.fold_slices;
        if (last)
            __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_last = last;
    }
    __syncthreads();
    return s_last;
}

// One workgroup's part of a product: tile `block` and slice `slice` of K, of g.slice_steps steps.  `turn`: this workgroup's number in the launch.
// (The arguments by value: by reference the compiler lays the branches of the end out otherwise, 512^3 f64 to the host 48.4 -> 48.7 us.)
// The tiles of a workgroup are WM x WN wave tiles, K is cut over WK waves each.
// Blocks are renumbered so that each of the 8 XCDs (own L2) works on a compact patch of tiles, eight
// tile rows deep: with the plain order the rows that share a column panel of B run on different XCDs.
template <typename T, int WM, int WN, int WK, int TM, int TN, bool TA, bool TB, bool CHECKED, bool FOLD = false>
__device__ __forceinline__ void direct_tile(const MatmulArgs g, int block, int slice, unsigned turn,
                                            PartialTiles<WM, WN, WK, TM, TN> &red)
{
    constexpr int PA = TM / 2, PB = TN / 2;                // row and column pairs of a lane
    constexpr bool TAIL = TM == 4 && WK > 1;               // kSquare: choose_plan
    // Steps whose operands are in flight.  f64 with three: no faster in large products (11008 x 4096 x 256 349 and 345 us), and
    // up to 15 % slower in short ones, which have the registers for fewer waves and load steps that they have not; but where K runs
    // across the rows of B, in tiles of 32 x 32 with K over four waves, a last round that is not full is a round longer
    // with two (dW 408 x 3057 x 2373 95 -> 111 us, 396 x 2741 x 2398 94 -> 109, dX 1803 x 1248 x 3212 231 -> 250; K < 400 2 % ahead).
    constexpr int D = sizeof(T) == 4 ? (TM * TN <= 4 ? 4 : 2) : (TM * TN == 4 && WK == 4 && !TB ? 3 : 2);
    constexpr int V = 4 * TM * TN;                         // values of a lane
    const T *__restrict__ A = static_cast<const T *>(g.A);
    const T *__restrict__ B = static_cast<const T *>(g.B);
    constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN;
    const int tiles_m = (g.M + BM - 1) / BM, tiles_n = (g.N + BN - 1) / BN;
    int of_tail = -1;
    if (TAIL && g.tail_slices > 1 && block >= g.whole_tiles) {
        of_tail = block - g.whole_tiles;
        slice = of_tail % g.tail_slices;
        block = g.whole_tiles + of_tail / g.tail_slices;
    }
    int tm, tn;
    tile_of_block(block, tiles_m, tiles_n, tm, tn);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wk = wave % WK, tile = wave / WK;
    const int m0 = tm * BM + (tile / WN) * 16 * TM, n0 = tn * BN + (tile % WN) * 16 * TN;
    const int r16 = lane & 15, kq = lane >> 4;
    // this workgroup's steps of K (all of them, or a slice) and this wave's among them
    const int steps = steps_of(g.K), per = TAIL && g.tail_slices > 1 && of_tail < 0 ? steps : g.slice_steps;
    const int first = slice * per, last = min(first + per, steps) - 1;
    const int count = first + wk > last ? 0 : (last - first - wk) / WK + 1;
    // where K is no whole steps the first one has what is left, and loads some of the next one's that it clears
    const int beyond = CHECKED ? 0 : -g.K & 15;

    // Rows and columns past the edge repeat the last ones; what they give is not stored.  A pair that would
    // reach past the edge is moved back by one: its second is then the edge.
    int row[PA][2], col[PB][2];
    auto pair_at = [&](int (&mn)[2], int at, int total, bool along) {
        mn[0] = min(at, total - (along && !CHECKED ? 2 : 1));
        mn[1] = along && !CHECKED ? mn[0] + 1 : min(at + 1, total - 1);
    };
#pragma unroll
    for (int p = 0; p < PA; ++p)
        pair_at(row[p], m0 + 32 * p + 2 * r16, g.M, TA);
#pragma unroll
    for (int p = 0; p < PB; ++p)
        pair_at(col[p], n0 + 32 * p + 2 * r16, g.N, !TB);
    T fa[D][PA][2][4], fb[D][PB][2][4];
    auto checked = [&](int d, int k0) {
#pragma unroll
        for (int p = 0; p < PA; ++p)
            checked_fetch<T, !TA>(fa[d][p], A, g.M, g.K, row[p], k0, kq);
#pragma unroll
        for (int p = 0; p < PB; ++p)
            checked_fetch<T, TB>(fb[d][p], B, g.N, g.K, col[p], k0, kq);
    };
    // Two workgroups that share a compute unit should end one after the other: where they end at once, a last round that is not
    // full may find both places of one unit and none of the next.  f32 tiles of 32 x 64, K along the rows of B: the wait in the loop; K
    // across them, where that wait does not do it: every other 256 workgroups, one per compute unit, go first (dX 144 x 8720 x
    // 1072, 2.7 rounds, 68 to 75 us -> 61 to 62; dX and dW of 280 to 1800 tiles on average level).
    constexpr bool in_turn = !CHECKED && sizeof(T) == 4 && TM * TN == 8 && WK > 1;
    if constexpr (in_turn && !TB) {
        if ((turn >> 8 & 1) == 0)
            __builtin_amdgcn_s_setprio(1);
    }
    const int row_first = min(m0, g.M - 1), col_first = min(n0, g.N - 1);
    auto fetch = [&](int d, int i) {   // the wave's i-th step; past its end the last one again
        const int k0 = max(min(first + wk + i * WK, last) * 16 - beyond, 0);
        if constexpr (CHECKED) {
            checked(d, k0);
        } else {
#pragma unroll
            for (int p = 0; p < PA; ++p)
                DirectOperand<T, !TA>(A, g.M, g.K, row_first, row[p], kq).fetch(fa[d][p], k0);
#pragma unroll
            for (int p = 0; p < PB; ++p)
                DirectOperand<T, TB>(B, g.N, g.K, col_first, col[p], kq).fetch(fb[d][p], k0);
        }
    };
    double4_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
            acc[i][j] = double4_t{0.0, 0.0, 0.0, 0.0};
    // The products of step d, and behind its conversions (or, of f64, behind its MFMAs) the loads that take its place.
    auto step = [&](int d, auto &&refill) {
        double a[TM][4], b[TN][4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
                a[i][k] = (double)fa[d][i >> 1][i & 1][k];
#pragma unroll
            for (int j = 0; j < TN; ++j)
                b[j][k] = (double)fb[d][j >> 1][j & 1][k];
        }
        if constexpr (sizeof(T) == 4) {
            __builtin_amdgcn_sched_barrier(0);
            refill();
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i][k], b[j][k], acc[i][j], 0, 0, 0);
        if constexpr (sizeof(T) == 8) {
            __builtin_amdgcn_sched_barrier(0);
            refill();
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto clear_beyond = [&] {   // the first step's, once it is loaded
        if (CHECKED || beyond == 0 || first + wk != 0)
            return;
        constexpr int VK = kRun<T>;
#pragma unroll
        for (int q = 0; q < 4; q += VK)
#pragma unroll
            for (int j = 0; j < VK; ++j) {
                const bool mine = 4 * q + VK * kq + j < 16 - beyond;
#pragma unroll
                for (int i = 0; i < 2; ++i) {
#pragma unroll
                    for (int p = 0; p < PA; ++p)
                        fa[0][p][i][q + j] = mine ? fa[0][p][i][q + j] : T(0);
#pragma unroll
                    for (int p = 0; p < PB; ++p)
                        fb[0][p][i][q + j] = mine ? fb[0][p][i][q + j] : T(0);
                }
            }
    };
    // (What is expected here is where the compiler lays the loop: behind the other paths, tiles of one wave each, all of a chip's
    // workgroups reading the same code, took 4 to 12 % longer, f32 dW 4411 x 1344 x 192 42 -> 51 us, f64 4096 x 2496 x 128 46 -> 49.)
    if (!CHECKED && __builtin_expect(g.K < 16, 0)) {
        if (count > 0) {
            checked(0, 0);
            step(0, [] {});
        }
    } else if (TM * TN <= 8 && (WK > 1 ? count <= D : __builtin_expect(count <= D, 0))) {
        // No more steps than can be in flight: none is loaded twice, and each number of them has code of its own (60 x 500 in tiles
        // of 32 x 32, K over four waves, loaded twice and now: f32 K = 64 4.5 -> 3.6 us, 128 5.0 -> 4.2, 192 5.4 -> 4.7; f64 64 4.1 -> 4.0, 128 5.3 -> 4.8).
        // (Conditions on single loads have the compiler move them behind the products before, and wait in the loop for
        // all that are in flight: f64 256 x 11008 x 4096 368 -> 429.)
        auto all = [&](auto n) {
#pragma unroll
            for (int d = 0; d < n; ++d)
                fetch(d, d);
            clear_beyond();
#pragma unroll
            for (int d = 0; d < n; ++d)
                step(d, [] {});
        };
        if (count == 1)
            all(std::integral_constant<int, 1>());
        else if (count == 2)
            all(std::integral_constant<int, 2>());
        else if (D > 2 && count == 3)
            all(std::integral_constant<int, D < 3 ? D : 3>());
        else if (D > 3 && count == 4)
            all(std::integral_constant<int, D < 4 ? D : 4>());
    } else if (count > 0) {
#pragma unroll
        for (int d = 0; d < D; ++d)
            fetch(d, d);
        clear_beyond();
        int i = 0;
        for (; i + D <= count; i += D) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                // All of a step's f32 operands are waited for before the first is converted: conversions that wait one by one lie
                // between the MFMAs of the workgroup beside this one, and the two end at once instead of one after the other
                // (f32 229 x 5211 x 1251 in 2.5 rounds 62 us, waiting for each 80; 256 x 11008 x 4096 level).
                if constexpr (in_turn && TB) {
                    constexpr int later = ((TA ? 4 : 2) * PA + 2 * PB) * (D - 1);             // loads of the steps behind it
                    __builtin_amdgcn_s_waitcnt(0x0f70 | (later & 15) | (later >> 4) << 14);   // vmcnt
                    __builtin_amdgcn_sched_barrier(0);
                }
                step(d, [&] { fetch(d, i + d + D); });
            }
        }
#pragma unroll
        for (int d = 0; d < D - 1; ++d)
            if (i + d < count)
                step(d, [] {});
    }
    if constexpr (!CHECKED) {
        // the edge of an odd matrix is the second of its pair
        if (m0 + 16 * TM > g.M - 1)
#pragma unroll
            for (int i = 0; i < TM; i += 2)
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        acc[i][j][e] = m0 + 16 * i + 2 * (4 * e + kq) == g.M - 1 ? acc[i + 1][j][e] : acc[i][j][e];
        if (n0 + 16 * TN > g.N - 1)
#pragma unroll
            for (int j = 0; j < TN; j += 2)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        acc[i][j][e] = n0 + 16 * j + 2 * r16 == g.N - 1 ? acc[i][j + 1][e] : acc[i][j][e];
    }
    T *__restrict__ C = static_cast<T *>(g.C);
    const T *__restrict__ bias = static_cast<const T *>(g.bias);
    double *__restrict__ partial = nullptr;   // and the place of C's first element, were it there
    int64_t partial_row = g.N;
    if (TAIL && of_tail >= 0) {
        partial = g.partial + (int64_t)of_tail * (BM * BN) - ((int64_t)tm * BM * BN + (int64_t)tn * BN);
        partial_row = BN;
    } else if (!FOLD && g.partial && !(TAIL && g.tail_slices > 1)) {
        partial = g.partial + (int64_t)slice * g.M * g.N;
    }
    // Value v of a lane: i = v / (4 TN), j = v / 4 % TN, e = v % 4.  Values v and v + 4 of an even j are
    // neighbours in a row and stored together: whole lines of 16 lanes.
    // Inside the matrix a store's address is a scalar and a lane's offset too.
    const bool inside = !CHECKED && !partial && m0 + 16 * TM <= g.M && n0 + 16 * TN <= g.N && g.N <= kLongest64<T>;
    const __amdgpu_buffer_rsrc_t tile_out =
        __builtin_amdgcn_make_buffer_rsrc(C + (inside ? (int64_t)m0 * g.N + n0 : 0), 0, 0xffffffff, 0x00027000);
    const unsigned lane_out = (2u * kq * (unsigned)g.N + 2u * r16) * (unsigned)sizeof(T);
    auto store = [&](int v, double s0, double s1) {
        const int i = v / (4 * TN), j = (v >> 2) % TN;
        if (inside) {
            T y[2] = {(T)s0, (T)s1};
            if (bias) {
                const T *at = bias + n0 + 32 * (j >> 1) + 2 * r16;
                y[0] = y[0] + at[0];
                y[1] = y[1] + at[1];
            }
            if (g.relu) {
                y[0] = y[0] < T(0) ? T(0) : y[0];
                y[1] = y[1] < T(0) ? T(0) : y[1];
            }
            const unsigned along = ((unsigned)(32 * (i >> 1) + 8 * (v & 3) + (i & 1)) * (unsigned)g.N + 32u * (j >> 1)) * (unsigned)sizeof(T);
            if (g.done.flag)
                store_run<true>(tile_out, lane_out, along, y[0], y[1]);
            else
                store_run<false>(tile_out, lane_out, along, y[0], y[1]);
            return;
        }
        const int r = m0 + 32 * (i >> 1) + 2 * (4 * (v & 3) + kq) + (i & 1), c = n0 + 32 * (j >> 1) + 2 * r16;
        if (r >= g.M || c >= g.N)
            return;
        const bool both = c + 1 < g.N;
        if (partial) {
            partial[(int64_t)r * partial_row + c] = s0;
            if (both)
                partial[(int64_t)r * partial_row + c + 1] = s1;
            return;
        }
        T y[2] = {(T)s0, (T)s1};     // the one rounding to the tensor's type
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            if (bias)
                y[u] = y[u] + bias[u && both ? c + 1 : c];     // Tensor.add in the tensor's type
            if (g.relu && y[u] < T(0))
                y[u] = T(0);
        }
        const int64_t at = (int64_t)r * g.N + c;
        if (both)
            store_pair(C, at, y[0], y[1], g.done);
        else
            vtlhip::store_result(C + at, y[0], g.done);
    };
    if constexpr (WK == 1) {
        // Nothing but conversions and stores: what `store` asks of every pair is asked once for the tile.  No vector
        // instruction runs beside another wave's MFMAs, so with a short K this end of a tile is what a launch waits for:
        // f32 dW 8192 x 8192 x 64 168 -> 149 us, 11008 x 4096 x 128 197 -> 183, x 256 363 -> 347.
        if (inside && !bias && !g.relu && !g.done.flag) {
#pragma unroll
            for (int v = 0; v < V; ++v)
                if (!(v & 4)) {
                    const int i = v / (4 * TN), j = (v >> 2) % TN;
                    const unsigned along = ((unsigned)(32 * (i >> 1) + 8 * (v & 3) + (i & 1)) * (unsigned)g.N + 32u * (j >> 1)) * (unsigned)sizeof(T);
                    store_run<false>(tile_out, lane_out, along, (T)acc[i][j][v & 3], (T)acc[i][j + 1][v & 3]);
                }
            return;   // no signal to raise
        }
#pragma unroll
        for (int v = 0; v < V; ++v)
            if (!(v & 4))
                store(v, acc[v / (4 * TN)][(v >> 2) % TN][v & 3], acc[v / (4 * TN)][(v >> 2) % TN + 1][v & 3]);
    } else {
        static_assert(!FOLD || !(TAIL || CHECKED), "slices meet in the launch for the shapes that are cut most");
        typedef double Pair __attribute__((ext_vector_type(2)));
        constexpr int kDevice = 16;   // sc1: past the caches of the XCD
        double *const slices_of_tile = FOLD ? g.partial + (int64_t)block * g.fold_slices * (BM * BN) : nullptr;
        const auto pair_at_tile = [](int u) { return (unsigned)(u * (64 * WM * WN * WK) + (int)threadIdx.x) * 16u; };
        // partial tiles, in the order of the registers
#pragma unroll
        for (int v = 0; v < V; ++v)
            red.at[wave][v][lane] = acc[v / (4 * TN)][(v >> 2) % TN][v & 3];
        __syncthreads();
#pragma unroll
        for (int u = 0; u < V / 2 / WK; ++u) {
            const int pair = wk + WK * u, v = 8 * (pair >> 2) + (pair & 3);
            double s0 = red.at[tile * WK][v][lane], s1 = red.at[tile * WK][v + 4][lane];
#pragma unroll
            for (int w = 1; w < WK; ++w) {
                s0 += red.at[tile * WK + w][v][lane];
                s1 += red.at[tile * WK + w][v + 4][lane];
            }
            if constexpr (FOLD)
                vtlhip::store_through<kDevice>(slices_of_tile + (int64_t)slice * (BM * BN), pair_at_tile(u), __builtin_bit_cast(vtlhip::Words4, Pair{s0, s1}));
            else
                store(v, s0, s1);
        }
        if constexpr (FOLD) {
            if (!last_of_tile(g, block))
                return;
            // four slices' pairs on their way at a time
            const __amdgpu_buffer_rsrc_t from = vtlhip::result_buffer(slices_of_tile);
            constexpr int PAIRS = V / 2 / WK, AT_ONCE = 4;
            Pair sum[PAIRS] = {};
            for (int s = 0; s < g.fold_slices; s += AT_ONCE) {
                Pair p[AT_ONCE][PAIRS];
#pragma unroll
                for (int q = 0; q < AT_ONCE; ++q)
#pragma unroll
                    for (int u = 0; u < PAIRS; ++u) {
                        const unsigned slice_at = (unsigned)min(s + q, g.fold_slices - 1) * (BM * BN * 8u);   // (the last one again, not added)
                        p[q][u] = __builtin_bit_cast(Pair, __builtin_amdgcn_raw_buffer_load_b128(from, pair_at_tile(u) + slice_at, 0, kDevice));
                    }
#pragma unroll
                for (int q = 0; q < AT_ONCE; ++q)
                    if (s + q < g.fold_slices)
#pragma unroll
                        for (int u = 0; u < PAIRS; ++u)
                            sum[u] += p[q][u];
            }
#pragma unroll
            for (int u = 0; u < PAIRS; ++u) {
                const int pair = wk + WK * u;
                store(8 * (pair >> 2) + (pair & 3), sum[u].x, sum[u].y);
            }
        }
    }
    vtlhip::raise_when_last(g.done);   // (a launch that leaves partial sums has no signal)
}

template <typename T, int WM, int WN, int WK, int TM, int TN, bool TA, bool TB, bool CHECKED, bool FOLD = false>
__global__ __launch_bounds__(64 * WM * WN * WK) void matmul_f64acc_direct_kernel(const MatmulArgs g)
{
    __shared__ PartialTiles<WM, WN, WK, TM, TN> red;
    direct_tile<T, WM, WN, WK, TM, TN, TA, TB, CHECKED, FOLD>(g, (int)blockIdx.x, (int)blockIdx.y, blockIdx.x + gridDim.x * blockIdx.y, red);
}

// The sums of kSumCols columns by one workgroup of 256 threads: 16 phases of rows, added in order.  Rows start at any element.
constexpr int kSumCols = 64;

template <typename T>
struct ColumnSums {
    const T *x;
    int rows, cols;
    T *out;
};

template <typename T>
__device__ __forceinline__ void colsum_tile(const ColumnSums<T> &g, int block, const vtlhip::DoneSignal &done,
                                            double (&red)[16][kSumCols])
{
    struct alignas(sizeof(T)) Run {
        T v[4];
    };
    const int group = threadIdx.x & 15, phase = threadIdx.x >> 4, c = block * kSumCols + 4 * group;
    const int first = min(c, g.cols - 4);   // the last columns with some of those before them
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    if (first >= 0 && c < g.cols) {
        const T *at = g.x + first;
        int r = phase;
        for (; r + 48 < g.rows; r += 64) {   // four loads in flight
            Run v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                v[u] = *reinterpret_cast<const Run *>(at + (int64_t)(r + 16 * u) * g.cols);
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    acc[j] += (double)v[u].v[j];
        }
        for (; r < g.rows; r += 16) {
            const Run v = *reinterpret_cast<const Run *>(at + (int64_t)r * g.cols);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                acc[j] += (double)v.v[j];
        }
    } else if (c < g.cols) {   // fewer than four columns
        for (int r = phase; r < g.rows; r += 16)
#pragma unroll
            for (int j = 0; j < 3; ++j)
                if (j < g.cols)
                    acc[j] += (double)g.x[(int64_t)r * g.cols + j];
    }
    const int shift = first >= 0 ? c - first : 0;   // 0 but for the last columns
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (j >= shift)
            red[phase][4 * group + j - shift] = acc[j];
    __syncthreads();
    const int mine = block * kSumCols + (int)threadIdx.x;
    if (threadIdx.x < kSumCols && mine < g.cols) {
        double s = 0.0;
#pragma unroll
        for (int i = 0; i < 16; ++i)
            s += red[i][threadIdx.x];
        vtlhip::store_result(g.out + mine, (T)s, done);
    }
}

template <typename T>
__global__ __launch_bounds__(256) void colsum_short_kernel(const ColumnSums<T> g)
{
    __shared__ double red[16][kSumCols];
    colsum_tile(g, (int)blockIdx.x, vtlhip::DoneSignal{}, red);
}

// ---- a Linear layer's gradients in one launch -----------------------------------------------
// dX = grad . W, dW = grad^T . x and db need nothing of each other, and of a small layer each leaves most of the chip idle for the 3
// to 5 us that a launch takes at least: workgroups 0 .. dx_blocks - 1 have the tiles of dX (slice by slice of K; the longest first), the next
// dw_blocks those of dW, the others the column sums.  Fifty sets of gradients of 16 to 256 rows, 64 to 8716 x 64 to 3722 parameters, half f32 and half f64:
// 19.2 us launch by launch, 12.3 now (geometric mean); 64 x 256 x 640 10.9 -> 5.6, 192 x 832 x 832 22.5 -> 13.8, 192 x 4096 x 1600 123 -> 95; with the
// forward in front 33 -> 28.
template <typename T>
struct BackwardArgs {
    ColumnSums<T> db;
    MatmulArgs dx, dw;
    int dx_tiles, dx_blocks, dw_blocks;
};

template <typename T, int TNX, int TNW, bool FOLD>
__global__ __launch_bounds__(256) void linear_backward_kernel(const BackwardArgs<T> g)
{
    __shared__ union {
        PartialTiles<1, 1, 4, 2, TNX> dx;
        PartialTiles<1, 1, 4, 2, TNW> dw;
        double db[16][kSumCols];
    } red;
    int block = (int)blockIdx.x;
    if (block < g.dx_blocks) {
        direct_tile<T, 1, 1, 4, 2, TNX, false, false, false, FOLD>(g.dx, block % g.dx_tiles, block / g.dx_tiles, blockIdx.x, red.dx);
        return;
    }
    block -= g.dx_blocks;
    if (block < g.dw_blocks) {
        direct_tile<T, 1, 1, 4, 2, TNW, true, false, false>(g.dw, block, 0, blockIdx.x, red.dw);
        return;
    }
    colsum_tile(g.db, block - g.dw_blocks, g.dw.done, red.db);
    vtlhip::raise_when_last(g.dw.done);
}

// Column sums with f64 accumulation: la.matmul(ones[1,M], grad) of
// nn/gates/layers/linear.v:75-79.  Block = 64 column groups x 4 row phases;
// grid.y splits the rows, each split writing f64 partial sums when there is
// more than one.
template <typename T, int VEC>
__global__ __launch_bounds__(256) void colsum_kernel(const T *__restrict__ x, int64_t rows, int64_t cols,
                                                     int64_t rows_per_split, T *__restrict__ out,
                                                     double *__restrict__ partial)
{
    __shared__ double red[4][64 * VEC];
    const int cg = threadIdx.x & 63, ph = threadIdx.x >> 6;
    const int64_t c0 = ((int64_t)blockIdx.x * 64 + cg) * VEC;
    const int64_t r_begin = (int64_t)blockIdx.y * rows_per_split;
    const int64_t r_end = r_begin + rows_per_split < rows ? r_begin + rows_per_split : rows;
    double acc[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j)
        acc[j] = 0.0;
    if (c0 < cols) {
        int64_t r = r_begin + ph;
        for (; r + 12 < r_end; r += 16) {
            T v[4][VEC];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                if constexpr (VEC == 4) {
                    const Vec4<T> t4 = *reinterpret_cast<const Vec4<T> *>(x + (r + 4 * u) * cols + c0);
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        v[u][j] = t4.v[j];
                } else {
                    v[u][0] = x[(r + 4 * u) * cols + c0];
                }
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int j = 0; j < VEC; ++j)
                    acc[j] += (double)v[u][j];
        }
        for (; r < r_end; r += 4) {
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                acc[j] += (double)x[r * cols + c0 + j];
        }
    }
#pragma unroll
    for (int j = 0; j < VEC; ++j)
        red[ph][cg * VEC + j] = acc[j];
    __syncthreads();
    if (ph == 0 && c0 < cols) {
#pragma unroll
        for (int j = 0; j < VEC; ++j) {
            const double s = ((red[0][cg * VEC + j] + red[1][cg * VEC + j]) + red[2][cg * VEC + j]) +
                             red[3][cg * VEC + j];
            if (partial)
                partial[(int64_t)blockIdx.y * cols + c0 + j] = s;
            else
                out[c0 + j] = (T)s;
        }
    }
}

template <typename T>
__global__ __launch_bounds__(256) void colsum_finalize_kernel(const double *__restrict__ partial, int splits,
                                                              int64_t cols, T *__restrict__ out)
{
    const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (c >= cols)
        return;
    double s = 0.0;
    for (int i = 0; i < splits; ++i)
        s += partial[(int64_t)i * cols + c];
    out[c] = (T)s;
}

// Sums the K slices of a split launch in slice order, rounds once to T, then
// bias and ReLU as in the unsplit epilogue.
template <typename T>
__global__ __launch_bounds__(256) void matmul_splitk_finalize_kernel(const MatmulArgs g, int splits)
{
    const int64_t total = (int64_t)g.M * g.N;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx < total) {
        double s = 0.0;
        for (int i = 0; i < splits; ++i)
            s += g.partial[(int64_t)i * total + idx];
        T y = (T)s;
        const T *__restrict__ bias = static_cast<const T *>(g.bias);
        if (bias)
            y = y + bias[idx % g.N];
        if (g.relu && y < T(0))
            y = T(0);
        vtlhip::store_result(static_cast<T *>(g.C) + idx, y, g.done);
    }
    vtlhip::raise_when_last(g.done);
}

// The last round's tiles, 256 elements a workgroup (with a tile each 128 x 8704 x 2049 in eight slices took 117 us, now 86).
template <typename T>
__global__ __launch_bounds__(256) void matmul_tail_finalize_kernel(const MatmulArgs g, int bm, int bn)
{
    const int per_tile = bm * bn / 256, t = (int)blockIdx.x / per_tile, i = ((int)blockIdx.x % per_tile) * 256 + (int)threadIdx.x;
    int tm, tn;
    tile_of_block(g.whole_tiles + t, (g.M + bm - 1) / bm, (g.N + bn - 1) / bn, tm, tn);
    const int r = tm * bm + i / bn, c = tn * bn + i % bn;
    if (r >= g.M || c >= g.N)
        return;
    const double *__restrict__ partial = g.partial + (int64_t)t * g.tail_slices * (bm * bn) + i;
    double s = 0.0;
#pragma unroll 4
    for (int k = 0; k < g.tail_slices; ++k)
        s += partial[(int64_t)k * (bm * bn)];
    T y = (T)s;
    const T *__restrict__ bias = static_cast<const T *>(g.bias);
    if (bias)
        y = y + bias[c];
    if (g.relu && y < T(0))
        y = T(0);
    static_cast<T *>(g.C)[(int64_t)r * g.N + c] = y;
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

template <typename T>
int finalize_split(MatmulArgs g, int splits, hipStream_t st)
{
    const int64_t blocks = ((int64_t)g.M * g.N + 255) / 256;
    if (g.result)
        g.result->attach(g.done, (unsigned)blocks);
    hipLaunchKernelGGL((matmul_splitk_finalize_kernel<T>), dim3((unsigned)blocks), dim3(256), 0, st, g, splits);
    return check_launch("matmul_splitk_finalize_kernel");
}

// The kernel's shapes, and K in `slices` over the grid.
enum Shape { kK8, kK4, kWide, kLarge, kSquare, kBlock, kShapes };
struct Plan {
    Shape shape;
    int slices;
    int tail_slices;   // of the last round's tiles alone
    double us;         // estimated
};

// Three kinds of product differ in what a shape costs: f32, f64, and f64 with K along both operands' rows (the
// Linear forward), where a 16-byte load is two k of one row and a small tile waits for its loads.
enum Kind { kF32, kF64, kF64Rows, kKinds };

// Wave tiles and waves per tile.  kLarge is one wave of 32 x 64 for f32 (level with 64 x 128 of four waves in large
// products, up to 3 % ahead with a short K) and that workgroup for f64 (2 % ahead of single waves at 4096^3).
// kSquare (a 64 x 64 wave tile, K over four) and kBlock (one such wave) are for kF64Rows: against kWide
// 256 x 11008 x 4096 523 -> 366 us, 64 x 10979 x 3840 169 -> 119, 4096^3 2760 -> 1865.
constexpr int kTileM[kKinds][kShapes] = {{32, 32, 32, 32, 0, 0}, {32, 32, 32, 64, 0, 0}, {32, 32, 32, 0, 64, 64}};
constexpr int kTileN[kKinds][kShapes] = {{32, 32, 64, 64, 0, 0}, {32, 32, 64, 128, 0, 0}, {32, 32, 64, 0, 64, 64}};
constexpr int kPerUnit[kKinds][kShapes] = {{1, 1, 1, 4, 0, 0}, {1, 1, 1, 1, 0, 0}, {1, 1, 1, 0, 1, 4}};   // workgroups that fill a compute unit's SIMDs once

// Estimated microseconds: start + rounds * (per_tile + work / rate), where `rounds` is how many times the busiest
// compute unit is filled and `work` the time its matrix cores need for that at
// 2.3 GHz; slicing K adds a launch and its partial sums (per MB).  Fitted to products drawn over m, n up to 11008 and k up to
// 4096, half of them with k below 300, whole and ragged, the layouts of forward and backward, every shape timed alternately: kF32 and kF64
// to 1200 of the forms before this one's for a short K, kF64Rows to 470 of these.  On 700 each the choice is on average 3.6, 2.8 and
// 1.3 % (kF32, kF64, kF64Rows) behind the fastest, at most 65, 29 and 26 %, the worst with k below 300.  (kF32 and kF64 refitted the same
// way come to 0.9 % there, but over 160 products with K from 200 to 4000 and rounds that are not full to 0 to 1 % more time than now and up to 15 %
// in single ones: kept as they were.)
struct Cost {
    double start, per_tile, inverse_rate, slice_start, slice_mb;
};
constexpr Cost kCost[kKinds][kShapes] = {
    {{1.59, 2.57, 1.18, 4.24, 0.42}, {3.22, 0.88, 1.13, 4.10, 0.43}, {2.89, 1.65, 1.05, 4.71, 0.45}, {2.52, 2.71, 1.08, 4.06, 0.53}, {}, {}},
    {{1.64, 2.07, 1.22, 4.27, 0.49}, {2.87, 0.83, 1.14, 4.01, 0.55}, {2.81, 1.65, 1.06, 4.57, 0.53}, {2.41, 3.48, 0.97, 5.23, 0.30}, {}, {}},
    {{1.51, 2.26, 2.08, 3.78, 0.67}, {1.59, 0.45, 1.97, 2.65, 0.74}, {2.10, 1.82, 1.42, 3.92, 0.52}, {}, {1.44, 6.76, 0.96, 4.19, 0.42},
     {0.02, 7.80, 1.07, 3.19, 0.42}},
};

// What a second launch has to be worth beyond its time on the device: it takes the host 3.4 us, which a chain of small products
// waits for.  Steps whose forward is cut for an estimated 0.04 and 0.46 us (16 x 2496 x 572 and 204 x 149 x 539, f64): 39.4 and
// 39.5 us, and 35.9 and 36.2 in one piece; 64 x 256 x 784, 0.84, is 8.9 cut and 10.9 in one piece.  Not in whole host
// calls, where the link is behind the host (242 x 78 x 765: 60.5 cut, 62.5 in one piece).
constexpr double kLaunch = 0.6;

Kind kind_of(bool f64, bool ta, bool tb) { return !f64 ? kF32 : (!ta && tb ? kF64Rows : kF64); }

// may_slice: whether K may be cut (matmul_impl).
Plan choose_plan(Kind kind, int m, int n, int k, bool may_slice, bool may_tail, double launch, unsigned shapes = ~0u)
{
    Plan best = {kK4, 1, 1, 1e30};
    const int most_slices = k / 96;
    for (int s = 0; s < kShapes; s++) {
        const int bm = kTileM[kind][s], bn = kTileN[kind][s], unit = kPerUnit[kind][s];
        if (bm == 0 || !(shapes >> s & 1))
            continue;
        const Cost &c = kCost[kind][s];
        // (tile sides are powers of two, and so is what fills the chip: no divisions where a small product spends its time)
        const int fill = unit == 4 ? 10 : 8;
        const int64_t tiles = (((int64_t)m + bm - 1) >> __builtin_ctz(bm)) * (((int64_t)n + bn - 1) >> __builtin_ctz(bn));
        // no slices, one workgroup per compute unit in all, or two where K is long
        int64_t want[3] = {1, 0, 0};
        if (may_slice && k >= 512 && tiles < 256) {
            want[1] = 256 / (int)tiles;
            want[2] = k >= 2048 ? 2 * want[1] : 0;
        }
        for (int64_t slices : want) {
            if (slices == 0)
                break;
            if (slices > most_slices)
                slices = most_slices;
            if (slices > 32)
                slices = 32;
            if (slices < 1)
                slices = 1;
            const double rounds = (double)((tiles * slices + (1 << fill) - 1) >> fill);
            const double work = (double)bm * bn * unit * ((double)k / (double)slices) / (64.0 * 2300.0);
            double us = c.start + rounds * (c.per_tile + work * c.inverse_rate);
            if (slices > 1)
                us += c.slice_start + launch + c.slice_mb * 8e-6 * (double)slices * (double)m * (double)n;
            if (us < best.us)
                best = {(Shape)s, (int)slices, 1, us};
        }
        // The last round with few tiles: K cut until they fill the chip.  For kSquare alone: its sums take 128 KiB of LDS, one
        // workgroup is all a compute unit holds, and a round is as long as its last (f64 forward, us: 256 x 4352 x 4096
        // 261 -> 145, 128 x 10240 x 2560 168 -> 110, 100 x 11008 x 4096 262 -> 191, 250 x 5000 x 640 50 -> 44).  The others have
        // two that share a unit's matrix cores and level that out: f32 256 x 11008 x 4096 came to 343 from 348.
        const int64_t whole = tiles >> fill, left = tiles & ((1 << fill) - 1);
        if (s == kSquare && may_tail && whole > 0 && left > 0) {
            const int64_t most = most_slices < 8 ? most_slices : 8;
            const int64_t slices = 256 * unit / left < most ? 256 * unit / left : most;
            if (slices > 1) {
                const double work = (double)bm * bn * unit * k / (64.0 * 2300.0);
                const double us = c.start + (double)whole * (c.per_tile + work * c.inverse_rate) + c.per_tile +
                                  work / (double)slices * c.inverse_rate + c.slice_start +
                                  c.slice_mb * 8e-6 * (double)(slices * left) * bm * bn;
                if (us < best.us)
                    best = {(Shape)s, 1, (int)slices, us};
            }
        }
    }
    return best;
}

// ROWS_ONLY: the layout of kF64Rows, no other.
template <typename T, int WM, int WN, int WK, int TM, int TN, bool CHECKED = false, bool ROWS_ONLY = false>
int launch_direct_shape(MatmulArgs g, bool ta, bool tb, int slices, hipStream_t st)
{
    constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN;
    const int64_t tiles = (int64_t)((g.M + BM - 1) / BM) * ((g.N + BN - 1) / BN);
    if (tiles > 0x7fffffff)
        return VTL_HIP_ERR_UNSUPPORTED;
    // (whole_tiles + the tail's slices: a few workgroups more than tiles)
    const int64_t blocks = g.tail_slices > 1 ? g.whole_tiles + (tiles - g.whole_tiles) * g.tail_slices : tiles;
    if (blocks > 0x7fffffff)
        return VTL_HIP_ERR_UNSUPPORTED;
    const dim3 grid((unsigned)blocks, (unsigned)slices), block(64 * WM * WN * WK);
    if (g.result && (slices == 1 || g.fold_slices > 1))
        g.result->attach(g.done, grid.x);
    constexpr bool FOLDS = WK > 1 && TM == 2 && !CHECKED;   // (fold_slices asks for no other)
#define VTL_DIRECT(TA, TB)                                                                                                                 \
    if (FOLDS && g.fold_slices > 1)                                                                                                        \
        hipLaunchKernelGGL((matmul_f64acc_direct_kernel<T, WM, WN, WK, TM, TN, TA, TB, CHECKED, FOLDS>), grid, block, 0, st, g);           \
    else                                                                                                                                   \
        hipLaunchKernelGGL((matmul_f64acc_direct_kernel<T, WM, WN, WK, TM, TN, TA, TB, CHECKED>), grid, block, 0, st, g)
    if constexpr (ROWS_ONLY) {
        VTL_DIRECT(false, true);
    } else {
        if (!ta && !tb) {
            VTL_DIRECT(false, false);
        } else if (!ta && tb) {
            VTL_DIRECT(false, true);
        } else if (ta && !tb) {
            VTL_DIRECT(true, false);
        } else {
            VTL_DIRECT(true, true);
        }
    }
#undef VTL_DIRECT
    return check_launch("matmul_f64acc_direct_kernel");
}

MatmulArgs arguments(const void *a, const void *b, void *c, int m, int n, int k)
{
    MatmulArgs g = {};
    g.A = a;
    g.B = b;
    g.C = c;
    g.M = m;
    g.N = n;
    g.K = k;
    g.tail_slices = 1;
    return g;
}

// Pairs of a row or column index that runs along memory need two of them.
template <typename T>
bool needs_checks(int m, int n, int k, bool ta, bool tb)
{
    return (ta && (m < 2 || m > kLongest16<T>)) || (!tb && (n < 2 || n > kLongest16<T>)) || ((!ta || tb) && k > kLongest64<T>);
}

// Memory for the slices' partial sums.  While the process uses the null stream alone (`alone`) it is a block
// of the call's own, released when the launches that use it are enqueued: the next owner's work comes
// behind them, and calls of several threads never meet in it.  Once a stream has been named a release would
// wait for the device, and the library's scratch, one per device, is what there is.
struct Partial {
    void *own = nullptr;
    ~Partial()
    {
        if (own)
            (void)vtl_hip_free(own);
    }
    Partial() = default;
    Partial(const Partial &) = delete;
    Partial &operator=(const Partial &) = delete;
    double *take(size_t bytes, bool alone)
    {
        if (alone)
            return vtl_hip_malloc(&own, bytes) == VTL_HIP_OK ? static_cast<double *>(own) : nullptr;
        return static_cast<double *>(vtlhip::library_workspace(bytes));
    }
};

// From how long a K on slices meet within their launch: shorter ones are level with a launch that adds them up (64 x 256 x 784 f32 7.4 and 7.2 us a
// call, f64 7.6 and 7.5).
constexpr int kFoldFrom = 800;

// The slices of a launch with tiles of bm x bn (kK8, kK4 or kWide) meet within it, where the stream has counters (not while it is being captured: replays of two graphs
// may meet) and the memory is there; else g is left as it is.  Nor where C lies over A or B: a tile is stored while others still read them.
template <typename T>
void fold_slices(MatmulArgs &g, int bm, int bn, int slices, Partial &partial, bool alone, hipStream_t st)
{
    const int64_t tiles = (int64_t)((g.M + bm - 1) / bm) * ((g.N + bn - 1) / bn);
    const size_t m = (size_t)g.M, n = (size_t)g.N, k = (size_t)g.K, c_bytes = m * n * sizeof(T);
    const bool over = vtlhip::meet(g.C, c_bytes, g.A, m * k * sizeof(T)) || vtlhip::meet(g.C, c_bytes, g.B, n * k * sizeof(T));
    const int slot = tiles <= kFoldTiles && g.K >= kFoldFrom && !over ? vtlhip::stream_slot(st) : -1;
    if (slot < 0 || !(g.partial = partial.take((size_t)tiles * (size_t)slices * (size_t)(bm * bn) * sizeof(double), alone)))
        return;
    g.fold_slices = slices;
    g.fold_slot = slot;
}

template <typename T>
int launch_direct(MatmulArgs g, Kind kind, bool ta, bool tb, Plan plan, bool alone, hipStream_t st)
{
    const bool checked = needs_checks<T>(g.M, g.N, g.K, ta, tb);
    const int steps = steps_of(g.K);
    int per = (steps + plan.slices - 1) / plan.slices;
    int slices = per > 0 ? (steps + per - 1) / per : 1;
    Partial partial;
    if (slices > 1) {
        if (!checked && (plan.shape == kK8 || plan.shape == kK4 || plan.shape == kWide))
            fold_slices<T>(g, kTileM[kind][plan.shape], kTileN[kind][plan.shape], slices, partial, alone, st);
        if (!g.partial)
            g.partial = partial.take((size_t)slices * (size_t)g.M * (size_t)g.N * sizeof(double), alone);
        if (!g.partial) {   // no memory, or a capture that may not allocate: K in one piece
            per = steps;
            slices = 1;
        }
    }
    constexpr int bm = 64, bn = 64;   // kSquare
    int64_t left = 0;
    if (plan.tail_slices > 1 && plan.shape == kSquare && slices == 1 && !checked && !g.result) {
        const int64_t tiles = (int64_t)((g.M + bm - 1) / bm) * ((g.N + bn - 1) / bn);
        left = tiles < 0x7fffffff ? tiles % 256 : 0;
        const int tail_per = (steps + plan.tail_slices - 1) / plan.tail_slices;
        const int tail = tail_per > 0 ? (steps + tail_per - 1) / tail_per : 1;
        if (left > 0 && tail > 1 && (g.partial = partial.take((size_t)left * (size_t)tail * (size_t)(bm * bn) * sizeof(double), alone))) {
            g.tail_slices = tail;
            g.whole_tiles = (int)(tiles - left);
            per = tail_per;
        }
    }
    g.slice_steps = per;
    int rc = VTL_HIP_ERR_UNSUPPORTED;
    if (checked)
        rc = launch_direct_shape<T, 1, 1, 8, 2, 2, true>(g, ta, tb, slices, st);
    else if (plan.shape == kK8)
        rc = launch_direct_shape<T, 1, 1, 8, 2, 2>(g, ta, tb, slices, st);
    else if (plan.shape == kK4)
        rc = launch_direct_shape<T, 1, 1, 4, 2, 2>(g, ta, tb, slices, st);
    else if (plan.shape == kWide)
        rc = launch_direct_shape<T, 1, 1, 4, 2, 4>(g, ta, tb, slices, st);
    else if constexpr (sizeof(T) == 4)
        rc = launch_direct_shape<T, 1, 1, 1, 2, 4>(g, ta, tb, slices, st);
    else if (plan.shape == kLarge)
        rc = launch_direct_shape<T, 2, 2, 1, 2, 4>(g, ta, tb, slices, st);
    else if (plan.shape == kSquare)
        rc = launch_direct_shape<T, 1, 1, 4, 4, 4, false, true>(g, ta, tb, slices, st);
    else
        rc = launch_direct_shape<T, 1, 1, 1, 4, 4, false, true>(g, ta, tb, slices, st);
    if (rc != VTL_HIP_OK)
        return rc;
    if (g.tail_slices > 1) {
        hipLaunchKernelGGL((matmul_tail_finalize_kernel<T>), dim3((unsigned)(left * (bm * bn / 256))), dim3(256), 0, st, g, bm, bn);
        return check_launch("matmul_tail_finalize_kernel");
    }
    return slices == 1 || g.fold_slices > 1 ? rc : finalize_split<T>(g, slices, st);
}

template <typename T>
int matmul_impl(const T *a, const T *b, T *c, const T *bias, int m, int n, int k, int trans_a, int trans_b,
                int relu, vtlhip::HostResult *result = nullptr)
{
    if (m < 0 || n < 0 || k < 0)
        return VTL_HIP_ERR_INVALID_ARG;
    if (m == 0 || n == 0)
        return VTL_HIP_OK;
    if (!c || (k > 0 && (!a || !b)))
        return VTL_HIP_ERR_INVALID_ARG;
    MatmulArgs g = arguments(a, b, c, m, n, k);
    g.result = result;
    g.bias = bias;
    g.relu = relu;
    // Where streams have been named, K is cut from 2048 on only: there the header asks callers to order
    // calls of different streams, which then share scratch; shorter products stay independent of each other
    // (64 x 256 x 784 f32: 8.9 us sliced, 10.9 in one piece; 64 x 256 x 2000: 9.3 and 21.9).
    const bool alone = vtlhip::single_stream();
    const Kind kind = kind_of(sizeof(T) == 8, trans_a != 0, trans_b != 0);
    Plan plan = choose_plan(kind, m, n, k, alone || k >= 2048, !result && (alone || k >= 2048), result ? 0.0 : kLaunch);
    // Tuning and tests: VTL_HIP_MATMUL_TILE 1 .. 6 forces a shape (one that the kind of product does not have gives its
    // largest), 64 and 128 the larger ones; VTL_HIP_MATMUL_SPLITS the slices of K, from -2 down those of the last round.
    const int tile = vtlhip::tuning().matmul_tile, splits = vtlhip::tuning().matmul_splits;
    if (tile > 0) {
        const int shape = tile == 64 ? (int)kSquare : (tile <= kShapes ? tile - 1 : (int)kBlock);
        plan.shape = kTileM[kind][shape] ? (Shape)shape : (kind == kF64Rows ? kBlock : kLarge);
    }
    if (splits >= 0 || splits < -1) {
        plan.slices = splits > 1 && k >= 32 * splits ? splits : 1;
        plan.tail_slices = splits < -1 ? -splits : 1;
    }
    return launch_direct<T>(g, kind, trans_a != 0, trans_b != 0, plan, alone, current_stream());
}

// Where one launch has the column sums, a workgroup all rows of its columns; elsewhere the rows are split from 128 on and a second
// launch adds up (us, split and in one: f32 256 x 11008 6.5 and 3.4, 128 x 300 6.3 and 3.6, 512 x 4097 6.7 and 4.4, 1024 x 4097 10.2
// and 11.1; f64 512 x 11008 11.4 and 7.9, 512 x 32768 24.6 and 20.0, 1024 x 4097 13.2 and 21.0).  Of wider rows a wave reads four times
// as much of one at a time in the split form, or, where they start anywhere, a word a lane: f64 127 x 65536 11.2 and 16.8, 96 x 65536 8.9
// and 12.2, 256 x 65536 23.5 and 25.4, 192 x 100003 27.6 and 28.7, f32 127 x 100003 12.4 and 12.9; but f32 320 x 65536 17.1 and 13.8.
constexpr int64_t kShortSums = 512, kShortSumsWidth = 32768;

template <typename T>
bool sums_in_one(const T *x, int64_t rows, int64_t cols)
{
    return rows <= kShortSums &&
           (cols <= kShortSumsWidth || (sizeof(T) == 4 && cols % 4 == 0 && aligned16(x) && cols <= 0x7fffffff - kSumCols));
}

template <typename T>
int colsum_impl(const T *x, int64_t rows, int64_t cols, T *out)
{
    if (rows < 0 || cols < 0)
        return VTL_HIP_ERR_INVALID_ARG;
    if (cols == 0)
        return VTL_HIP_OK;
    if (!out || (rows > 0 && !x))
        return VTL_HIP_ERR_INVALID_ARG;
    hipStream_t st = current_stream();
    const size_t out_bytes = (size_t)cols * sizeof(T);
    // (Not where the sums lie within x: a workgroup would write over columns that another still reads.)
    if (sums_in_one(x, rows, cols) && !vtlhip::meet(x, (size_t)rows * out_bytes, out, out_bytes)) {
        const ColumnSums<T> g = {x, (int)rows, (int)cols, out};
        hipLaunchKernelGGL((colsum_short_kernel<T>), dim3((unsigned)((cols + kSumCols - 1) / kSumCols)), dim3(256), 0, st, g);
        return check_launch("colsum_short_kernel");
    }
    const bool vec = aligned16(x) && cols % 4 == 0;
    const int per_block = vec ? 256 : 64;
    const int64_t col_blocks = (cols + per_block - 1) / per_block;
    if (col_blocks > 0x7fffffff)
        return VTL_HIP_ERR_UNSUPPORTED;
    // enough workgroups to fill the chip, but at least 64 rows per split
    int64_t splits = 1;
    if (col_blocks < 1024 && rows >= 128) {
        splits = 1024 / col_blocks;
        if (splits > rows / 64)
            splits = rows / 64;
        if (splits > 1024)
            splits = 1024;
        if (splits < 1)
            splits = 1;
    }
    const int64_t rows_per_split = splits > 1 ? (rows + splits - 1) / splits : rows;
    if (splits > 1)
        splits = (rows + rows_per_split - 1) / rows_per_split;
    double *partial = nullptr;
    if (splits > 1) {
        partial = static_cast<double *>(
            vtlhip::library_workspace((size_t)splits * (size_t)cols * sizeof(double)));
        if (!partial)
            return vtlhip::workspace_status();
    }
    const dim3 grid((unsigned)col_blocks, (unsigned)splits);
    if (vec)
        hipLaunchKernelGGL((colsum_kernel<T, 4>), grid, dim3(256), 0, st, x, rows, cols, rows_per_split, out,
                           partial);
    else
        hipLaunchKernelGGL((colsum_kernel<T, 1>), grid, dim3(256), 0, st, x, rows, cols, rows_per_split, out,
                           partial);
    int rc = check_launch("colsum_kernel");
    if (rc != VTL_HIP_OK || splits == 1)
        return rc;
    hipLaunchKernelGGL((colsum_finalize_kernel<T>), dim3((unsigned)((cols + 255) / 256)), dim3(256), 0, st,
                       partial, (int)splits, cols, out);
    return check_launch("colsum_finalize_kernel");
}

// dW and what else is asked for (not null) in one launch; false: launch by launch.  `result`: dw and db are its memory, and this is
// the call's last launch.
template <typename T>
bool backward_in_one(vtlhip::HostResult *result, const T *grad, const T *x, const T *w, T *dx, T *dw, T *db, int m, int n, int k,
                     int &status)
{
    const int forced = vtlhip::tuning().backward_group;
    if (!dw || !(dx || db) || m < 1 || n < 1 || k < 1 || (db && m > kShortSums) || forced == 0 || vtlhip::tuning().matmul_tile > 0 ||
        vtlhip::tuning().matmul_splits != -1 || needs_checks<T>(n, k, m, true, false) || (dx && needs_checks<T>(m, k, n, false, false)))
        return false;
    // launch by launch a gradient may take the place of what those before it were made from
    const size_t e = sizeof(T), grad_bytes = (size_t)m * n * e, x_bytes = (size_t)m * k * e, w_bytes = (size_t)n * k * e, b_bytes = (size_t)n * e;
    const struct { const void *at; size_t bytes; } all[6] = {{grad, grad_bytes}, {x, x_bytes}, {dx ? w : nullptr, w_bytes},
                                                             {dx, x_bytes}, {dw, w_bytes}, {db, b_bytes}};
    for (int i = 3; i < 6; i++)
        for (int j = 0; j < i; j++)
            if (vtlhip::meet(all[i].at, all[i].bytes, all[j].at, all[j].bytes))
                return false;

    const bool alone = vtlhip::single_stream();
    const Kind kind = sizeof(T) == 8 ? kF64 : kF32;
    constexpr unsigned shapes = 1u << kK4 | 1u << kWide;   // workgroups of four waves
    const Plan pw = choose_plan(kind, n, k, m, false, false, kLaunch, shapes);
    const bool may_slice = !(result && dx) && (alone || n >= 2048);   // (sums of slices would come behind the call's last launch)
    const Plan px = dx ? choose_plan(kind, m, k, n, may_slice, false, kLaunch, shapes) : Plan{kK4, 1, 1, 0.0};
    const auto tiles = [&](Shape s, int rows, int cols) {
        return (int64_t)((rows + 31) / 32) * ((cols + kTileN[kind][s] - 1) / kTileN[kind][s]);
    };
    const auto tile_us = [&](Shape s, double depth) {
        const Cost &c = kCost[kind][s];
        return c.per_tile + 32.0 * kTileN[kind][s] * depth / (64.0 * 2300.0) * c.inverse_rate;
    };
    const int64_t tiles_w = tiles(pw.shape, n, k), tiles_x = dx ? tiles(px.shape, m, k) : 0;
    const int64_t sums = db ? (n + kSumCols - 1) / kSumCols : 0;
    const int steps = steps_of(n), per = (steps + px.slices - 1) / px.slices, slices = dx ? (steps + per - 1) / per : 1;
    if (tiles_w + tiles_x * slices + sums > 0x7fffffff)
        return false;
    if (forced < 0) {
        // As choose_plan estimates, the tiles of both products dealt out over the chip.  Five hundred sets of gradients of 2 to 600 rows, n and k
        // of 2 to 6000, half f32 and half f64, in one launch and one by one: up to 0.8 of `apart` 0.34 to 0.97 of the time, up to 0.9 0.74 to 0.99, up to
        // 1.05 0.77 to 1.03; above 1.2, where large weight tiles have shapes of their own, 1.21 to 1.85.  Less sure are tiles that are mostly
        // stores or partial sums: from 0.85 on f32 9 x 1899 x 2356 27.0 and 33.1 us, 31 x 1870 x 1608 23.0 and 23.9, f64 7 x 927 x 4509 15.3 and 17.4, 442 x 6 x 3774
        // 15.0 and 15.9, without dX f32 88 x 1150 x 4098 31.7 and 34.4, f64 15 x 1993 x 769 8.8 and 9.6.
        const double each_x = tile_us(px.shape, (double)n / px.slices), each_w = tile_us(pw.shape, m);
        const double longest = dx && each_x > each_w ? each_x : each_w;
        double us = 2.9 + ((double)(tiles_x * px.slices) * each_x + (double)tiles_w * each_w) / 256.0 + 0.5 * longest;
        if (px.slices > 1)
            us += kCost[kind][px.shape].slice_start + kLaunch + kCost[kind][px.shape].slice_mb * 8e-6 * px.slices * (double)m * (double)k;
        double apart = choose_plan(kind, n, k, m, alone || m >= 2048, false, kLaunch).us + (db ? 4.0 : 0.0);
        if (dx)
            apart += choose_plan(kind, m, k, n, alone || n >= 2048, false, kLaunch).us;
        const bool slim = n < 32 || (m < 32 && (!dx || px.slices > 1)) || (m < 128 && w_bytes > (size_t)16 << 20);
        if (us > (slim ? 0.85 : 1.05) * apart)
            return false;
    }
    BackwardArgs<T> g = {};
    g.dw = arguments(grad, x, dw, n, k, m);
    g.dw.slice_steps = steps_of(m);
    g.dw_blocks = (int)tiles_w;
    g.dx = arguments(grad, w, dx, m, k, n);
    g.dx.slice_steps = per;
    g.db = {grad, m, n, db};
    Partial partial;
    int cut = slices;
    if (cut > 1)
        fold_slices<T>(g.dx, 32, kTileN[kind][px.shape], cut, partial, alone, current_stream());
    if (cut > 1 && !g.dx.partial && !(g.dx.partial = partial.take((size_t)cut * (size_t)m * (size_t)k * sizeof(double), alone))) {
        g.dx.slice_steps = steps;   // no memory, or a capture that may not allocate: K in one piece
        cut = 1;
    }
    g.dx_tiles = (int)(tiles_x > 0 ? tiles_x : 1);
    g.dx_blocks = (int)tiles_x * cut;
    const dim3 grid((unsigned)(g.dx_blocks + tiles_w + sums));
    if (result) {
        result->attach(g.dw.done, grid.x);
        g.dx.done = g.dw.done;
    }
    hipStream_t st = current_stream();
#define VTL_BACKWARD(TNX, TNW)                                                                        \
    if (g.dx.fold_slices > 1)                                                                         \
        hipLaunchKernelGGL((linear_backward_kernel<T, TNX, TNW, true>), grid, dim3(256), 0, st, g);   \
    else                                                                                              \
        hipLaunchKernelGGL((linear_backward_kernel<T, TNX, TNW, false>), grid, dim3(256), 0, st, g)
    if (px.shape == kK4 && pw.shape == kK4) {
        VTL_BACKWARD(2, 2);
    } else if (px.shape == kK4) {
        VTL_BACKWARD(2, 4);
    } else if (pw.shape == kK4) {
        VTL_BACKWARD(4, 2);
    } else {
        VTL_BACKWARD(4, 4);
    }
#undef VTL_BACKWARD
    status = check_launch("linear_backward_kernel");
    if (status == VTL_HIP_OK && cut > 1 && g.dx.fold_slices <= 1)
        status = finalize_split<T>(g.dx, cut, st);
    return true;
}

template <typename T>
int linear_backward_impl(const T *grad, const T *x, const T *w, T *dx, T *dw, T *db, int m, int n, int k)
{
    if (m < 0 || n < 0 || k < 0 || !grad)
        return VTL_HIP_ERR_INVALID_ARG;
    if ((dx && !w) || (dw && !x))
        return VTL_HIP_ERR_INVALID_ARG;
    int rc = VTL_HIP_OK;
    if (backward_in_one<T>(nullptr, grad, x, w, dx, dw, db, m, n, k, rc))
        return rc;
    if (dx)   // [M,K] = grad[M,N] . W[N,K]
        rc = matmul_impl<T>(grad, w, dx, nullptr, m, k, n, 0, 0, 0);
    if (rc == VTL_HIP_OK && dw)   // [N,K] = grad^T[N,M] . x[M,K]
        rc = matmul_impl<T>(grad, x, dw, nullptr, n, k, m, 1, 0, 0);
    if (rc == VTL_HIP_OK && db)   // [1,N] = ones[1,M] . grad[M,N]
        rc = colsum_impl<T>(grad, m, n, db);
    return rc;
}

// dW and, unless it is null, db.
template <typename T>
int weight_gradients(vtlhip::HostResult *result, const T *grad, const T *x, T *dw, T *db, int m, int n, int k)
{
    int rc = VTL_HIP_OK;
    if (backward_in_one<T>(result, grad, x, nullptr, nullptr, dw, db, m, n, k, rc))
        return rc;
    if (db)
        rc = colsum_impl<T>(grad, m, n, db);
    return rc == VTL_HIP_OK ? matmul_impl<T>(grad, x, dw, nullptr, n, k, m, 1, 0, 0, result) : rc;
}

}  // namespace

namespace vtlhip {

int matmul_to(HostResult *result, const float *a, const float *b, float *c, int m, int n, int k, int trans_a)
{
    return matmul_impl<float>(a, b, c, nullptr, m, n, k, trans_a, 0, 0, result);
}

int matmul_to(HostResult *result, const double *a, const double *b, double *c, int m, int n, int k, int trans_a)
{
    return matmul_impl<double>(a, b, c, nullptr, m, n, k, trans_a, 0, 0, result);
}

bool gradients_in_one(HostResult *result, const float *grad, const float *x, const float *w, float *dx, float *dw, float *db, int m, int n,
                      int k, int &status)
{
    return backward_in_one<float>(result, grad, x, w, dx, dw, db, m, n, k, status);
}

bool gradients_in_one(HostResult *result, const double *grad, const double *x, const double *w, double *dx, double *dw, double *db, int m,
                      int n, int k, int &status)
{
    return backward_in_one<double>(result, grad, x, w, dx, dw, db, m, n, k, status);
}

int weight_gradients_to(HostResult *result, const float *grad, const float *x, float *dw, float *db, int m, int n, int k)
{
    return weight_gradients<float>(result, grad, x, dw, db, m, n, k);
}

int weight_gradients_to(HostResult *result, const double *grad, const double *x, double *dw, double *db, int m, int n, int k)
{
    return weight_gradients<double>(result, grad, x, dw, db, m, n, k);
}

}  // namespace vtlhip

extern "C" {

int vtl_hip_matmul_f32(const float *a, const float *b, float *c, int m, int n, int k, int trans_a,
                       int trans_b)
{
    return matmul_impl<float>(a, b, c, nullptr, m, n, k, trans_a, trans_b, 0);
}

int vtl_hip_matmul_f64(const double *a, const double *b, double *c, int m, int n, int k, int trans_a,
                       int trans_b)
{
    return matmul_impl<double>(a, b, c, nullptr, m, n, k, trans_a, trans_b, 0);
}

int vtl_hip_linear_f32(const float *x, const float *w, const float *bias, float *y, int m, int n, int k,
                       int relu)
{
    return matmul_impl<float>(x, w, y, bias, m, n, k, 0, 1, relu);
}

int vtl_hip_linear_f64(const double *x, const double *w, const double *bias, double *y, int m, int n, int k,
                       int relu)
{
    return matmul_impl<double>(x, w, y, bias, m, n, k, 0, 1, relu);
}

int vtl_hip_colsum_f32(const float *x, int64_t rows, int64_t cols, float *out)
{
    return colsum_impl<float>(x, rows, cols, out);
}

int vtl_hip_colsum_f64(const double *x, int64_t rows, int64_t cols, double *out)
{
    return colsum_impl<double>(x, rows, cols, out);
}

int vtl_hip_linear_backward_f32(const float *grad, const float *x, const float *w, float *dx, float *dw,
                                float *db, int m, int n, int k)
{
    return linear_backward_impl<float>(grad, x, w, dx, dw, db, m, n, k);
}

int vtl_hip_linear_backward_f64(const double *grad, const double *x, const double *w, double *dx,
                                double *dw, double *db, int m, int n, int k)
{
    return linear_backward_impl<double>(grad, x, w, dx, dw, db, m, n, k);
}

}  // extern "C"
