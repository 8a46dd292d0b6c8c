// Dense matmul with f64 products and sums on the gfx950 f64 matrix cores, for
// f32 and f64 tensors: the device form of la.matmul (la/la.v:38-55) and
// gate_matmul (autograd/gates_blas.v:6-23), which widen every operand to f64,
// multiply with a f64 GEMM and round the result once to the tensor's type.
// Also the unquantized Linear forward (nn/layers/linear_forward_f32.v:16-18)
// and LinearGate.backward (nn/gates/layers/linear.v:69-79) built on it.
//
// Two kernels.  matmul_f64acc_kernel stages 128 x 128 tiles through LDS for large products of whole
// tiles; matmul_f64acc_direct_kernel, for everything else, takes operands from global memory
// straight to registers.  choose_plan() picks by estimated time.
//
// The staged kernel: one workgroup of WR x WC waves owns a BM x BN tile of C.  Both operands go
// through LDS in k-major form (As[k][m], Bs[k][n]) whatever their
// layout in memory, so that one 16- or 32-byte LDS read hands a lane the
// operands of all its 16x16x4 MFMA tiles for one k.  MFMA tile i of a wave
// holds the rows {TM * r + i : r = 0..15} of the wave's rows (and likewise for
// columns), which makes those reads and the final stores contiguous per lane.
#include "common.hpp"

#include <stdlib.h>

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
    int k_per_split;    // k range of one grid.y slice (multiple of 16)
    double *partial;    // launches that slice K: [slices][M][N] unrounded sums, else nullptr
    vtlhip::DoneSignal done;     // C is the memory of a whole host call's result
    vtlhip::HostResult *result;  // host side only
};

template <typename T>
struct alignas(16) Vec4 {
    T v[4];
};

// NT consecutive LDS elements (NT = 2 or 4, naturally aligned) widened to f64.
template <typename T, int NT>
__device__ __forceinline__ void read_operands(const T *__restrict__ p, double (&out)[NT])
{
    struct alignas(NT * sizeof(T) > 16 ? 16 : NT * sizeof(T)) Pack {
        T v[NT];
    };
    const Pack pk = *reinterpret_cast<const Pack *>(p);
#pragma unroll
    for (int i = 0; i < NT; ++i)
        out[i] = (double)pk.v[i];
}

// One operand tile of BK x BMN elements (k-major in LDS, row stride LDW).
// KMAJOR: the matrix is stored with the tile's m/n index contiguous ([K, MN]);
// otherwise it is stored [MN, K] and is transposed on the way into LDS.
template <typename T, int BK, int BMN, int LDW, int NT, bool KMAJOR>
struct OperandTile {
    static constexpr int kGroups = BK * BMN / 4;       // 4-element groups per tile
    static constexpr int kPerThread = (kGroups + NT - 1) / NT;   // NT threads in the workgroup
    typedef T Group __attribute__((ext_vector_type(4)));   // (a struct of four stays in scratch memory)
    Group regs[kPerThread];

    __device__ __forceinline__ void fetch(const T *__restrict__ base, int mn_total, int k_total, int mn0, int k0)
    {
        const int t = threadIdx.x;
#pragma unroll
        for (int i = 0; i < kPerThread; ++i) {
            const int g = t + NT * i;
            if (kGroups % NT != 0 && g >= kGroups)
                break;
            const T *__restrict__ p;
            if constexpr (KMAJOR)
                p = base + (int64_t)(k0 + g / (BMN / 4)) * mn_total + mn0 + 4 * (g % (BMN / 4));
            else
                p = base + (int64_t)(mn0 + g % BMN) * k_total + k0 + 4 * (g / BMN);
            regs[i] = *reinterpret_cast<const Group *>(p);
        }
    }

    __device__ __forceinline__ void stash(T *__restrict__ lds) const
    {
        const int t = threadIdx.x;
#pragma unroll
        for (int i = 0; i < kPerThread; ++i) {
            const int g = t + NT * i;
            if (kGroups % NT != 0 && g >= kGroups)
                break;
            if constexpr (KMAJOR) {
                const int krow = g / (BMN / 4), c4 = g % (BMN / 4);
                *reinterpret_cast<Group *>(lds + krow * LDW + 4 * c4) = regs[i];
            } else {
                const int mn = g % BMN, kc = g / BMN;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    lds[(4 * kc + j) * LDW + mn] = regs[i][j];
            }
        }
    }
};

// Workgroup barrier that orders LDS traffic only: unlike __syncthreads() it does
// not wait for outstanding global loads, so the operand loads issued two
// k-tiles ahead stay in flight across it.
__device__ __forceinline__ void lds_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// M, N, K are whole tiles and every row is 16-byte aligned.
// Workgroup = WR x WC waves, each with TM x TN MFMA tiles of 16x16:
// BM = 16 * TM * WR, BN = 16 * TN * WC.
template <typename T, int TM, int TN, int WR, int WC, bool TA, bool TB>
__global__ __launch_bounds__(64 * WR * WC) void matmul_f64acc_kernel(const MatmulArgs g)
{
    constexpr int BM = 16 * TM * WR, BN = 16 * TN * WC, NT = 64 * WR * WC;
    constexpr int BK = 64 / (int)sizeof(T);   // bytes of k per tile row: 64 (16 f32 / 8 f64)
    constexpr int LDA = BM + 4, LDB = BN + 4;
    static_assert(TM == 2 || TM == 4, "wave tile is 32 or 64 rows");
    static_assert(TN == 4, "wave tile is 64 columns");

    // Three LDS buffers per operand: while tile kt is multiplied, tile kt+1 is
    // written at the start of the step (its global loads were issued a step
    // earlier) and the one barrier per step sits before the last k-group, so
    // that the first operands of tile kt+1 are read from LDS under the last
    // MFMAs of tile kt and no MFMA waits for a barrier followed by an LDS read.
    __shared__ __attribute__((aligned(16))) T As[3][BK * LDA];
    __shared__ __attribute__((aligned(16))) T Bs[3][BK * LDB];

    const T *__restrict__ A = static_cast<const T *>(g.A);
    const T *__restrict__ B = static_cast<const T *>(g.B);
    const int tiles_n = g.N / BN;
    const int m0 = (int)(blockIdx.x / tiles_n) * BM;
    const int n0 = (int)(blockIdx.x % tiles_n) * BN;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = (wave / WC) * (16 * TM), wn = (wave % WC) * (16 * TN);
    const int r16 = lane & 15, kq = lane >> 4;

    // A as op(A)[M,K]: stored [K,M] when transposed (k-major already)
    OperandTile<T, BK, BM, LDA, NT, TA> ta;
    // B as op(B)[K,N]: stored [K,N] when not transposed (k-major already)
    OperandTile<T, BK, BN, LDB, NT, !TB> tb;

    double4_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
            acc[i][j] = double4_t{0.0, 0.0, 0.0, 0.0};

    const int ktiles = g.K / BK;
    constexpr int S = BK / 4;   // k-groups (one MFMA step each) per tile
    const int aoff = wm + TM * r16 + kq * LDA, boff = wn + TN * r16 + kq * LDB;

    ta.fetch(A, g.M, g.K, m0, 0);
    tb.fetch(B, g.N, g.K, n0, 0);
    ta.stash(As[0]);
    tb.stash(Bs[0]);
    if (ktiles > 1) {
        ta.fetch(A, g.M, g.K, m0, BK);
        tb.fetch(B, g.N, g.K, n0, BK);
    }
    __syncthreads();
    double a[TM], b[TN];
    read_operands<T, TM>(As[0] + aoff, a);
    read_operands<T, TN>(Bs[0] + boff, b);

    int cur = 0;
    for (int kt = 0; kt < ktiles; ++kt) {
        const int nxt = cur == 2 ? 0 : cur + 1;
        if (kt + 1 < ktiles) {
            // buffer nxt was last read two steps ago; every wave has passed a barrier since
            ta.stash(As[nxt]);
            tb.stash(Bs[nxt]);
        }
        if (kt + 2 < ktiles) {
            ta.fetch(A, g.M, g.K, m0, (kt + 2) * BK);
            tb.fetch(B, g.N, g.K, n0, (kt + 2) * BK);
        }
#pragma unroll
        for (int s = 0; s < S; ++s) {
            double an[TM], bn[TN];
            if (s + 1 < S) {
                read_operands<T, TM>(As[cur] + aoff + 4 * (s + 1) * LDA, an);
                read_operands<T, TN>(Bs[cur] + boff + 4 * (s + 1) * LDB, bn);
            } else {
                lds_barrier();   // tile kt+1 is in LDS for every wave; global loads stay in flight
                read_operands<T, TM>(As[nxt] + aoff, an);
                read_operands<T, TN>(Bs[nxt] + boff, bn);
            }
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < TM; ++i)
                a[i] = an[i];
#pragma unroll
            for (int j = 0; j < TN; ++j)
                b[j] = bn[j];
        }
        cur = nxt;
    }

    T *__restrict__ C = static_cast<T *>(g.C);
    const T *__restrict__ bias = static_cast<const T *>(g.bias);
    const int col0 = n0 + wn + TN * r16;
    T bv[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j)
        bv[j] = bias ? bias[col0 + j] : T(0);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int row = m0 + wm + TM * (4 * e + kq) + i;
            Vec4<T> out;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                T y = (T)acc[i][j][e];   // the one rounding to the tensor's type
                if (bias)
                    y = y + bv[j];       // Tensor.add in the tensor's type
                if (g.relu && y < T(0))
                    y = T(0);
                out.v[j] = y;
            }
            *reinterpret_cast<Vec4<T> *>(C + (int64_t)row * g.N + col0) = out;
        }
    }
}

// ---- operands straight from global memory --------------------------------------------------
// A wave owns 32 x 16 * TN of C.  An f64 MFMA wants two values a lane every 64 cycles, so operands
// need neither LDS nor barriers, and what bounds a launch is how evenly its MFMAs spread over the
// SIMDs: the tiles are small, K is cut over the WK waves of a workgroup (partial tiles meet in LDS)
// and, with few tiles, over grid.y.  With 64 x 64 tiles staged in LDS a wave had four MFMAs for every 4
// of K, 7 us at K = 256 and 14 us at K = 512 whatever else the chip did, and ragged sizes loaded
// element by element: 512^3 22.4 -> 8.8 us, 64 x 784 x 256 16.4 -> 5.5, 64 x 256 x 784 44 -> 7.5,
// 255 x 11007 x 4095 447 -> 367, 333 x 517 x 701 47 -> 13 (f32; f64 alike).
//
// Steps of 16 of K are dealt out to the WK waves in turn.  In a step lane l holds four k for the two
// rows 2 * (l % 16) + {0, 1} of A and for TN / 2 such pairs of columns of B: 16-byte loads where K runs
// along memory, pairs of 32 neighbouring columns where it does not.  MFMA j of a step takes the j-th of
// each lane's four: which k they are is free as long as both operands agree.
// Vector loads need no more than the elements' own alignment on gfx950, so ragged rows take them too;
// what is left of K after whole steps is a step of its own with checked loads.  CHECKED: every
// load is (a single row or column of a matrix that has to give pairs).
template <typename T, bool KROWS, bool CHECKED>
__device__ __forceinline__ void direct_fetch(T (&out)[2][4], const T *__restrict__ base, int mn_total, int k_total,
                                            const int (&mn)[2], bool second_only, int k0, int kq)
{
    // a 16-byte load holds VK elements; the lane's four are those VK of each run of 4 * VK
    constexpr int VK = 16 / (int)sizeof(T);
    struct alignas(sizeof(T)) Run {
        T v[VK];
    };
    struct alignas(sizeof(T)) Pair {
        T v[2];
    };
#pragma unroll
    for (int q = 0; q < 4; q += VK) {
        const int k = k0 + 4 * q + VK * kq;
        if constexpr (KROWS) {   // [MN, K]
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const T *__restrict__ p = base + (int64_t)mn[i] * k_total + k;
                if constexpr (!CHECKED) {
                    const Run v = *reinterpret_cast<const Run *>(p);
#pragma unroll
                    for (int j = 0; j < VK; ++j)
                        out[i][q + j] = v.v[j];
                } else {
#pragma unroll
                    for (int j = 0; j < VK; ++j)
                        out[i][q + j] = k + j < k_total ? p[j] : T(0);
                }
            }
        } else {                 // [K, MN]
#pragma unroll
            for (int j = 0; j < VK; ++j) {
                if constexpr (!CHECKED) {
                    // second_only: the pair was moved back by one to stay inside, its second is mn[0]
                    const Pair v = *reinterpret_cast<const Pair *>(base + (int64_t)(k + j) * mn_total + mn[0] -
                                                                   (second_only ? 1 : 0));
                    out[0][q + j] = second_only ? v.v[1] : v.v[0];
                    out[1][q + j] = v.v[1];
                } else {
#pragma unroll
                    for (int i = 0; i < 2; ++i)
                        out[i][q + j] = k + j < k_total ? base[(int64_t)(k + j) * mn_total + mn[i]] : T(0);
                }
            }
        }
    }
}

// Two neighbours of a row, aligned as one element is.
__device__ __forceinline__ void store_pair(float *p, float a, float b, const vtlhip::DoneSignal &done)
{
    typedef float Two __attribute__((ext_vector_type(2), aligned(4)));
    const Two v = {a, b};
    if (done.flag)   // waited for in raise_when_last
        asm volatile("global_store_dwordx2 %0, %1, off sc0 sc1" ::"v"(p), "v"(v) : "memory");
    else
        *reinterpret_cast<Two *>(p) = v;
}

__device__ __forceinline__ void store_pair(double *p, double a, double b, const vtlhip::DoneSignal &done)
{
    typedef double Two __attribute__((ext_vector_type(2), aligned(8)));
    const Two v = {a, b};
    if (done.flag)
        asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1" ::"v"(p), "v"(v) : "memory");
    else
        *reinterpret_cast<Two *>(p) = v;
}

// The tiles of a workgroup are WM x WN wave tiles of 32 x 16 * TN, K is cut over WK waves each.
// Blocks are renumbered so that each of the 8 XCDs (own L2) works on a compact patch of tiles, eight
// tile rows deep: with the plain order the rows that share a column panel of B run on different XCDs.
template <typename T, int WM, int WN, int WK, int TN, bool TA, bool TB, bool CHECKED>
__global__ __launch_bounds__(64 * WM * WN * WK) void matmul_f64acc_direct_kernel(const MatmulArgs g)
{
    constexpr int D = sizeof(T) == 4 && TN == 2 ? 4 : 2;   // steps whose operands are in flight
    constexpr int P = TN / 2;                              // column pairs of a lane
    constexpr int V = 8 * TN;                              // values of a lane
    __shared__ double red[WK > 1 ? WM * WN * WK : 1][WK > 1 ? V : 1][64];
    const T *__restrict__ A = static_cast<const T *>(g.A);
    const T *__restrict__ B = static_cast<const T *>(g.B);
    constexpr int BM = 32 * WM, BN = 16 * TN * WN;
    const int tiles_m = (g.M + BM - 1) / BM, tiles_n = (g.N + BN - 1) / BN;
    int tm, tn;
    {
        const int total = tiles_m * tiles_n, block = (int)blockIdx.x;
        const int xcd = block & 7, over = total & 7;
        const int pid = xcd * (total >> 3) + min(xcd, over) + (block >> 3);
        const int group = 8 * tiles_n, first_m = (pid / group) * 8, gm = min(tiles_m - first_m, 8);
        tm = first_m + (pid % group) % gm;
        tn = (pid % group) / gm;
    }
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wk = wave % WK, tile = wave / WK;
    const int m0 = tm * BM + (tile / WN) * 32, n0 = tn * BN + (tile % WN) * 16 * TN;
    const int r16 = lane & 15, kq = lane >> 4;
    // this workgroup's whole steps of K (all of them, or one of grid.y slices), this wave's among
    // them, and whether this wave does the part of a step at the end of K
    const int steps = CHECKED ? (g.K + 15) / 16 : g.K / 16, per = g.k_per_split / 16;
    const int first = (int)blockIdx.y * per, last = min(first + per, steps) - 1;
    const int count = first + wk > last ? 0 : (last - first - wk) / WK + 1;
    const bool rest = !CHECKED && steps * 16 < g.K && blockIdx.y == gridDim.y - 1 && wk == WK - 1;

    // rows and columns past the edge repeat the last ones; what they give is not stored
    const int row[2] = {min(m0 + 2 * r16, g.M - 1), min(m0 + 2 * r16 + 1, g.M - 1)};
    const bool row_alone = row[0] == g.M - 1;
    int col[P][2];
    bool col_alone[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        col[p][0] = min(n0 + 32 * p + 2 * r16, g.N - 1);
        col[p][1] = min(n0 + 32 * p + 2 * r16 + 1, g.N - 1);
        col_alone[p] = col[p][0] == g.N - 1;
    }
    T fa[D][2][4], fb[D][P][2][4];
    auto fetch = [&](int d, int i) {   // the wave's i-th step; past its end the last one again
        const int k0 = min(first + wk + i * WK, last) * 16;
        direct_fetch<T, !TA, CHECKED>(fa[d], A, g.M, g.K, row, row_alone, k0, kq);
#pragma unroll
        for (int p = 0; p < P; ++p)
            direct_fetch<T, TB, CHECKED>(fb[d][p], B, g.N, g.K, col[p], col_alone[p], k0, kq);
    };
    double4_t acc[2][TN];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
            acc[i][j] = double4_t{0.0, 0.0, 0.0, 0.0};
    auto multiply = [&](int d) {
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                        (double)fa[d][i][k], (double)fb[d][j >> 1][j & 1][k], acc[i][j], 0, 0, 0);
    };
    if (count > 0) {
#pragma unroll
        for (int d = 0; d < D; ++d)
            fetch(d, d);
        int i = 0;
        for (; i + D <= count; i += D) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                multiply(d);
                fetch(d, i + d + D);
            }
        }
#pragma unroll
        for (int d = 0; d < D - 1; ++d)
            if (i + d < count)
                multiply(d);
    }
    if (rest) {
        const int k0 = steps * 16;
        direct_fetch<T, !TA, true>(fa[0], A, g.M, g.K, row, false, k0, kq);
#pragma unroll
        for (int p = 0; p < P; ++p)
            direct_fetch<T, TB, true>(fb[0][p], B, g.N, g.K, col[p], false, k0, kq);
        multiply(0);
    }
    T *__restrict__ C = static_cast<T *>(g.C);
    const T *__restrict__ bias = static_cast<const T *>(g.bias);
    double *__restrict__ partial = g.partial ? g.partial + (int64_t)blockIdx.y * g.M * g.N : nullptr;
    // Value v of a lane: i = v / (4 TN), j = v / 4 % TN, e = v % 4.  Values v and v + 4 of an even j are
    // neighbours in a row and stored together: whole lines of 16 lanes.
    auto store = [&](int v, double s0, double s1) {
        const int j = (v >> 2) & (TN - 1);
        const int r = m0 + 2 * (4 * (v & 3) + kq) + v / (4 * TN), c = n0 + 32 * (j >> 1) + 2 * r16;
        if (r >= g.M || c >= g.N)
            return;
        const bool both = c + 1 < g.N;
        if (partial) {
            partial[(int64_t)r * g.N + c] = s0;
            if (both)
                partial[(int64_t)r * g.N + c + 1] = s1;
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
        T *to = C + ((int64_t)r * g.N + c);
        if (both)
            store_pair(to, y[0], y[1], g.done);
        else
            vtlhip::store_result(to, y[0], g.done);
    };
    if constexpr (WK == 1) {
#pragma unroll
        for (int v = 0; v < V; ++v)
            if (!(v & 4))
                store(v, acc[v / (4 * TN)][(v >> 2) & (TN - 1)][v & 3], acc[v / (4 * TN)][((v >> 2) & (TN - 1)) + 1][v & 3]);
    } else {
        // partial tiles, in the order of the registers
#pragma unroll
        for (int v = 0; v < V; ++v)
            red[wave][v][lane] = acc[v / (4 * TN)][(v >> 2) & (TN - 1)][v & 3];
        __syncthreads();
#pragma unroll
        for (int u = 0; u < V / 2 / WK; ++u) {
            const int pair = wk + WK * u, v = 8 * (pair >> 2) + (pair & 3);
            double s0 = red[tile * WK][v][lane], s1 = red[tile * WK][v + 4][lane];
#pragma unroll
            for (int w = 1; w < WK; ++w) {
                s0 += red[tile * WK + w][v][lane];
                s1 += red[tile * WK + w][v + 4][lane];
            }
            store(v, s0, s1);
        }
    }
    vtlhip::raise_when_last(g.done);   // (a launch that leaves partial sums has no signal)
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

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

template <typename T>
int launch_staged(const MatmulArgs &g, bool ta, bool tb, hipStream_t st)
{
    // eight waves of 32x64 per 128x128 tile measured a few percent above four waves of 64x64
    const int64_t tiles = (int64_t)(g.M / 128) * (g.N / 128);
    if (tiles > 0x7fffffff)
        return VTL_HIP_ERR_UNSUPPORTED;
    const dim3 grid((unsigned)tiles), block(512);
    if (!ta && !tb)
        hipLaunchKernelGGL((matmul_f64acc_kernel<T, 2, 4, 4, 2, false, false>), grid, block, 0, st, g);
    else if (!ta && tb)
        hipLaunchKernelGGL((matmul_f64acc_kernel<T, 2, 4, 4, 2, false, true>), grid, block, 0, st, g);
    else if (ta && !tb)
        hipLaunchKernelGGL((matmul_f64acc_kernel<T, 2, 4, 4, 2, true, false>), grid, block, 0, st, g);
    else
        hipLaunchKernelGGL((matmul_f64acc_kernel<T, 2, 4, 4, 2, true, true>), grid, block, 0, st, g);
    return check_launch("matmul_f64acc_kernel");
}

template <typename T>
int finalize_split(MatmulArgs g, int splits, hipStream_t st)
{
    const int64_t blocks = ((int64_t)g.M * g.N + 255) / 256;
    if (g.result)
        g.result->attach(g.done, (unsigned)blocks);
    hipLaunchKernelGGL((matmul_splitk_finalize_kernel<T>), dim3((unsigned)blocks), dim3(256), 0, st, g, splits);
    return check_launch("matmul_splitk_finalize_kernel");
}

// How a product runs: the staged kernel, or one of the direct kernel's shapes with K in `slices`.
enum Shape { kStaged, kK8, kK4, kWide, kPairK2, kPanel, kShapes };
struct Plan {
    Shape shape;
    int slices;
};

// Wave tiles and waves per tile: what the names above stand for.
constexpr int kTileM[kShapes] = {128, 32, 32, 32, 64, 64};
constexpr int kTileN[kShapes] = {128, 32, 32, 64, 64, 128};

// Estimated microseconds: start + rounds * (per_tile + work / rate), where `rounds` is how many
// workgroups the busiest compute unit gets and `work` the time its matrix cores need for one tile at
// 2.3 GHz; slicing K adds a launch and its partial sums (per MB).  Fitted to 240 products drawn over
// m, n up to 11008 and k up to 4096, whole and ragged, all four layouts, every shape timed alternately:
// the choice is on average 2.6 % and at most 30 % behind the fastest.
struct Cost {
    double start, per_tile, inverse_rate, slice_start, slice_mb;
};
constexpr Cost kCost[2][kShapes] = {
    // f32
    {{2.9, 0.0, 1.12, 0, 0}, {2.8, 1.27, 1.27, 3.5, 0.68}, {3.3, 0.56, 1.31, 3.9, 0.55}, {2.9, 1.61, 1.13, 3.7, 0.60},
     {3.1, 2.20, 1.13, 4.0, 0.35}, {3.2, 2.85, 1.19, 4.0, 0.35}},
    // f64
    {{2.5, 2.5, 1.14, 0, 0}, {1.9, 1.71, 1.41, 3.1, 1.39}, {3.1, 0.68, 1.44, 3.6, 0.73}, {2.8, 1.68, 1.23, 4.0, 0.58},
     {3.3, 2.21, 1.18, 4.0, 0.27}, {2.5, 3.40, 1.19, 4.0, 0.27}},
};

// may_slice: whether K may be cut (matmul_impl).
Plan choose_plan(bool f64, int m, int n, int k, bool whole, bool may_slice)
{
    Plan best = {kK4, 1};
    double best_us = 1e30;
    for (int s = whole ? kStaged : kK8; s < kShapes; s++) {
        const Cost &c = kCost[f64 ? 1 : 0][s];
        const int64_t tiles = (int64_t)((m + kTileM[s] - 1) / kTileM[s]) * ((n + kTileN[s] - 1) / kTileN[s]);
        // no slices, one workgroup per compute unit in all, or two where K is long
        int64_t want[3] = {1, 0, 0};
        if (may_slice && s != kStaged && k >= 512 && tiles < 256) {
            want[1] = 256 / tiles;
            want[2] = k >= 2048 ? 2 * want[1] : 0;
        }
        for (int64_t slices : want) {
            if (slices > k / 96)
                slices = k / 96;
            if (slices > 32)
                slices = 32;
            if (slices < 1)
                slices = 1;
            const double rounds = (double)((tiles * slices + 255) / 256);
            const double work = (double)kTileM[s] * kTileN[s] * ((double)k / (double)slices) / (64.0 * 2300.0);
            double us = c.start + rounds * (c.per_tile + work * c.inverse_rate);
            if (slices > 1)
                us += c.slice_start + c.slice_mb * 8e-6 * (double)slices * (double)m * (double)n;
            if (us < best_us) {
                best_us = us;
                best = {(Shape)s, (int)slices};
            }
        }
    }
    return best;
}

template <typename T, int WM, int WN, int WK, int TN, bool CHECKED = false>
int launch_direct_shape(MatmulArgs g, bool ta, bool tb, int slices, hipStream_t st)
{
    constexpr int BM = 32 * WM, BN = 16 * TN * WN;
    const int64_t tiles = (int64_t)((g.M + BM - 1) / BM) * ((g.N + BN - 1) / BN);
    if (tiles > 0x7fffffff)
        return VTL_HIP_ERR_UNSUPPORTED;
    const dim3 grid((unsigned)tiles, (unsigned)slices), block(64 * WM * WN * WK);
    if (g.result && slices == 1)
        g.result->attach(g.done, grid.x);
    if (!ta && !tb)
        hipLaunchKernelGGL((matmul_f64acc_direct_kernel<T, WM, WN, WK, TN, false, false, CHECKED>), grid, block, 0, st, g);
    else if (!ta && tb)
        hipLaunchKernelGGL((matmul_f64acc_direct_kernel<T, WM, WN, WK, TN, false, true, CHECKED>), grid, block, 0, st, g);
    else if (ta && !tb)
        hipLaunchKernelGGL((matmul_f64acc_direct_kernel<T, WM, WN, WK, TN, true, false, CHECKED>), grid, block, 0, st, g);
    else
        hipLaunchKernelGGL((matmul_f64acc_direct_kernel<T, WM, WN, WK, TN, true, true, CHECKED>), grid, block, 0, st, g);
    return check_launch("matmul_f64acc_direct_kernel");
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

template <typename T>
int launch_direct(MatmulArgs g, bool ta, bool tb, Plan plan, bool alone, hipStream_t st)
{
    // pairs of a row or column index that runs along memory need two of them
    const bool checked = (ta && g.M < 2) || (!tb && g.N < 2);
    const int steps = checked ? (g.K + 15) / 16 : g.K / 16;
    int per = (steps + plan.slices - 1) / plan.slices;
    int slices = per > 0 ? (steps + per - 1) / per : 1;
    Partial partial;
    if (slices > 1) {
        g.partial = partial.take((size_t)slices * (size_t)g.M * (size_t)g.N * sizeof(double), alone);
        if (!g.partial) {   // no memory, or a capture that may not allocate: K in one piece
            per = steps;
            slices = 1;
        }
    }
    g.k_per_split = 16 * per;
    int rc;
    if (checked)
        rc = launch_direct_shape<T, 1, 1, 8, 2, true>(g, ta, tb, slices, st);
    else if (plan.shape == kK8)
        rc = launch_direct_shape<T, 1, 1, 8, 2>(g, ta, tb, slices, st);
    else if (plan.shape == kWide)
        rc = launch_direct_shape<T, 1, 1, 4, 4>(g, ta, tb, slices, st);
    else if (plan.shape == kPairK2)
        rc = launch_direct_shape<T, 2, 1, 2, 4>(g, ta, tb, slices, st);
    else if (plan.shape == kPanel)
        rc = launch_direct_shape<T, 2, 2, 1, 4>(g, ta, tb, slices, st);
    else
        rc = launch_direct_shape<T, 1, 1, 4, 2>(g, ta, tb, slices, st);
    return rc != VTL_HIP_OK || slices == 1 ? rc : finalize_split<T>(g, slices, st);
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
    MatmulArgs g = {};
    g.result = result;
    g.A = a;
    g.B = b;
    g.C = c;
    g.bias = bias;
    g.M = m;
    g.N = n;
    g.K = k;
    g.relu = relu;
    // the staged kernel's loads and stores carry no bounds checks
    const bool whole = m % 128 == 0 && n % 128 == 0 && k % 32 == 0 && k > 0 && aligned16(a) && aligned16(b) &&
                       aligned16(c);
    // Where streams have been named, K is cut from 2048 on only: there the header asks callers to order
    // calls of different streams, which then share scratch; shorter products stay independent of each other
    // (64 x 256 x 784 f32: 8.9 us sliced, 10.9 in one piece; 64 x 256 x 2000: 9.3 and 21.9).
    const bool alone = vtlhip::single_stream();
    Plan plan = choose_plan(sizeof(T) == 8, m, n, k, whole, alone || k >= 2048);
    // Tuning and tests: VTL_HIP_MATMUL_TILE 128 forces the staged kernel where it can run, 64 the
    // 64 x 64 tiles, 1 .. 5 a shape of the direct kernel; VTL_HIP_MATMUL_SPLITS the slices of K.
    const int tile = vtlhip::tuning().matmul_tile, splits = vtlhip::tuning().matmul_splits;
    if (tile == 128 && whole)
        plan.shape = kStaged;
    else if (tile == 64)
        plan.shape = kPairK2;
    else if (tile >= kK8 && tile < kShapes)
        plan.shape = (Shape)tile;
    if (splits >= 0) {
        plan.slices = splits > 1 && k >= 32 * splits ? splits : 1;
        if (plan.shape == kStaged && plan.slices > 1)
            plan.shape = kK4;
    } else if (plan.shape == kStaged) {
        plan.slices = 1;
    }
    return plan.shape == kStaged ? launch_staged<T>(g, trans_a != 0, trans_b != 0, current_stream())
                                 : launch_direct<T>(g, trans_a != 0, trans_b != 0, plan, alone, current_stream());
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

template <typename T>
int linear_backward_impl(const T *grad, const T *x, const T *w, T *dx, T *dw, T *db, int m, int n, int k)
{
    if (m < 0 || n < 0 || k < 0 || !grad)
        return VTL_HIP_ERR_INVALID_ARG;
    if ((dx && !w) || (dw && !x))
        return VTL_HIP_ERR_INVALID_ARG;
    int rc = VTL_HIP_OK;
    if (dx)   // [M,K] = grad[M,N] . W[N,K]
        rc = matmul_impl<T>(grad, w, dx, nullptr, m, k, n, 0, 0, 0);
    if (rc == VTL_HIP_OK && dw)   // [N,K] = grad^T[N,M] . x[M,K]
        rc = matmul_impl<T>(grad, x, dw, nullptr, n, k, m, 1, 0, 0);
    if (rc == VTL_HIP_OK && db)   // [1,N] = ones[1,M] . grad[M,N]
        rc = colsum_impl<T>(grad, m, n, db);
    return rc;
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
