// Device-side pieces of the symmetric INT8 quantizer shared by the streaming
// kernels and the fused decode kernel: wave / workgroup max, the correctly
// rounded code of one element, packing.  Arithmetic contract in quant.hip.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace vtlhip {
namespace qdev {

typedef float float4_t __attribute__((ext_vector_type(4)));
typedef int int4_t __attribute__((ext_vector_type(4)));

// Max over the 64 lanes of a wave, returned to every lane: cross-lane moves
// inside the VALU (DPP) - quads, half rows and rows by mirroring, then lane 15
// of each row into the next row and lane 31 into the upper half; lane 63 holds
// the result.  Lanes a move does not reach see 0, the identity for the
// non-negative values this is used on.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_max_step(float v)
{
    const int t = __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROW_MASK, 0xF, false);
    return fmaxf(v, __int_as_float(t));
}

__device__ __forceinline__ float wave_max(float v)
{
    v = dpp_max_step<0xB1, 0xF>(v);   // quad_perm [1,0,3,2]
    v = dpp_max_step<0x4E, 0xF>(v);   // quad_perm [2,3,0,1]
    v = dpp_max_step<0x141, 0xF>(v);  // row_half_mirror
    v = dpp_max_step<0x140, 0xF>(v);  // row_mirror
    v = dpp_max_step<0x142, 0xA>(v);  // row_bcast:15 into rows 1 and 3
    v = dpp_max_step<0x143, 0xC>(v);  // row_bcast:31 into rows 2 and 3
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// Workgroup barrier that orders LDS traffic only: unlike __syncthreads() it does
// not wait for outstanding global loads, so direct-to-LDS weight loads issued
// earlier stay in flight across it.
__device__ __forceinline__ void lds_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Max over each group of SEG = 16, 32 or 64 consecutive lanes (a DPP row, two, or the wave),
// returned to every lane of the group.
template <int SEG>
__device__ __forceinline__ float segment_max(float v)
{
    static_assert(SEG == 16 || SEG == 32 || SEG == 64, "a DPP row, two, or the wave");
    if constexpr (SEG == 64)
        return wave_max(v);
    v = dpp_max_step<0xB1, 0xF>(v);
    v = dpp_max_step<0x4E, 0xF>(v);
    v = dpp_max_step<0x141, 0xF>(v);
    v = dpp_max_step<0x140, 0xF>(v);
    if constexpr (SEG == 32)
        v = fmaxf(v, __shfl_xor(v, 16));
    return v;
}

// Max over the workgroup; every thread gets the result.  smem holds T/64
// floats and is used once per kernel.
template <int T>
__device__ __forceinline__ float block_max(float v, float *smem)
{
    v = wave_max(v);
    if constexpr (T > 64) {
        const int w = threadIdx.x >> 6;
        if ((threadIdx.x & 63) == 0)
            smem[w] = v;
        __syncthreads();
        float r = smem[0];
#pragma unroll
        for (int i = 1; i < T / 64; i++)
            r = fmaxf(r, smem[i]);
        v = r;
    }
    return v;
}

__device__ __forceinline__ float absmax4(float m, float4_t v)
{
    m = fmaxf(m, fabsf(v.x));
    m = fmaxf(m, fabsf(v.y));
    m = fmaxf(m, fabsf(v.z));
    m = fmaxf(m, fabsf(v.w));
    return m;
}

// Saturating f32 -> i32 conversion; NaN converts to 0 in hardware.
__device__ __forceinline__ int cvt_i32_sat(float r)
{
    int i;
    asm("v_cvt_i32_f32 %0, %1" : "=v"(i) : "v"(r));
    return i;
}

struct QuantScale {
    float scale;
    float rinv;  // 1/scale when `fast`
    bool fast;   // scale and 1/scale are normal numbers with headroom
};

__device__ __forceinline__ QuantScale make_quant_scale(float scale)
{
    QuantScale p;
    p.scale = scale;
    p.fast = (scale >= 0x1p-100f) && (scale <= 0x1p100f);
    p.rinv = p.fast ? (1.0f / scale) : 0.0f;
    return p;
}

// Half-width of the band around k + 0.5 inside which the estimated quotient
// cannot decide the rounding.  For |x/scale| <= 128 the estimate
// fl(x * fl(1/scale)) is within 2^-16 of the true quotient and the correctly
// rounded quotient within 2^-18, so 2^-14 leaves a factor of three.  Larger
// quotients clamp to +-127 whichever way they round.
constexpr float kTieBand = 0x1p-14f;

__device__ __forceinline__ int quant_code(float x, const QuantScale &p)
{
    float r;
    if (p.fast) {
        const float t = x * p.rinv;
        r = rintf(t);
        if (__builtin_expect(fabsf(t - r) >= 0.5f - kTieBand, 0))
            r = rintf(x / p.scale);
    } else {
        r = rintf(x / p.scale);  // 0/0, x/Inf, subnormal scales: exact path
    }
    const int i = cvt_i32_sat(r);
    return min(max(i, -127), 127);
}

__device__ __forceinline__ unsigned pack4(int a, int b, int c, int d)
{
    return (unsigned)(a & 0xff) | ((unsigned)(b & 0xff) << 8) | ((unsigned)(c & 0xff) << 16) |
           ((unsigned)d << 24);
}

// Four codes at once: a quotient's rounding is what is left of it beside a number whose last place is one, the code its low
// byte, and one test sees whether any of the four is too close to a tie, or no number (v_maximum3 keeps a NaN): then the
// codes are made one by one.  6 vector instructions an element instead of 14, which the kernels that quantize a row in every workgroup, or hold
// a tensor in registers until its scale is known, have nothing to hide behind (us, one at a time before: linear on f32 rows 1 x 4096 x 11008 8.3 -> 7.75,
// 1 x 14336 x 4096 10.0 -> 8.8, 2 x 11.45 -> 10.2, 8 x 12.7 -> 11.5; 128 rows, in a launch of their own, level; 3001 x 4099 quantized with one scale and
// back 27.15 -> 26.5, 16384 x 16384 per row and back 425 -> 422).
// GIVEN: the scale is not that of the values' own maximum, so quotients may be out of range.
template <bool GIVEN = false>
__device__ __forceinline__ unsigned quant4(float4_t v, const QuantScale &p)
{
    constexpr float kOnes = 0x1.8p23f;
    float n[4], off[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float t = v[i] * p.rinv;
        n[i] = t + kOnes;
        const float r = n[i] - kOnes;
        off[i] = fabsf(t - r);
        if (GIVEN)
            n[i] = __builtin_amdgcn_fmed3f(r, -127.0f, 127.0f) + kOnes;
    }
    const float most = __builtin_elementwise_maximum(__builtin_elementwise_maximum(off[0], off[1]), __builtin_elementwise_maximum(off[2], off[3]));
    if (__builtin_expect(p.fast && most < 0.5f - kTieBand, 1)) {
        const unsigned lo = __builtin_amdgcn_perm(__float_as_uint(n[1]), __float_as_uint(n[0]), 0x0c0c0400);
        const unsigned hi = __builtin_amdgcn_perm(__float_as_uint(n[3]), __float_as_uint(n[2]), 0x04000c0c);
        return lo | hi;
    }
    return pack4(quant_code(v.x, p), quant_code(v.y, p), quant_code(v.z, p), quant_code(v.w, p));
}

}  // namespace qdev
}  // namespace vtlhip
