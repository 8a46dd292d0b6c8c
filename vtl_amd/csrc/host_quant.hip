// Quantization on the host's vector units, for f32 rows on their way to the device.
//
// Rows in host memory cross the link as codes, a quarter of their bytes.  The host touches the rows either way, to copy them into
// pinned memory; making codes instead reads the same bytes and writes a quarter of them.  Bound by memory, as the copy is (180 MB on a
// 16-processor EPYC, GB/s of f32 with 1 / 4 / 8 threads: quantized 31 / 95 / 156, AVX2 27 / 83 / 151, copied 34 / 99 / 138; the link takes 57).
// Codes and scales are those of the device's quantizer bit for bit (quant_device.hpp has the arithmetic): f32 operations
// that are correctly rounded on both, and where an estimated quotient is near a tie the division itself.
#include <string.h>

#include "host_quant.hpp"

#if defined(__x86_64__) && !defined(__HIP_DEVICE_COMPILE__)
#include <immintrin.h>
#define VTL_HOST_VECTORS 1
#endif

namespace vtlhip {

#ifdef VTL_HOST_VECTORS
namespace {

constexpr float kTie = 0.5f - 0x1p-14f;   // from here on an estimated quotient's distance from its rounding cannot decide

// Rounding to nearest, subnormals as they are, whatever the calling thread is set to.  (The compiler does not see that arithmetic
// depends on this: what is computed in between is read from memory and written there, which does not move past the barriers.)
struct DefaultFloats {
    unsigned before = _mm_getcsr();
    DefaultFloats()
    {
        _mm_setcsr(0x1f80);
        asm volatile("" ::: "memory");
    }
    ~DefaultFloats()
    {
        asm volatile("" ::: "memory");
        _mm_setcsr(before);
    }
};

// By division: NaN has code 0, what is out of range clamps.
int8_t code(float x, float scale)
{
    const float r = __builtin_rintf(x / scale);
    return (int8_t)(!(r == r) ? 0.0f : r < -127.0f ? -127.0f : r > 127.0f ? 127.0f : r);
}

// Whether scale and 1 / scale are normal numbers with headroom.
bool by_estimate(float scale) { return scale >= 0x1p-100f && scale <= 0x1p100f; }

#define VTL_AVX512 __attribute__((target("avx512f,avx512bw,avx512vl,avx512dq")))
#define VTL_AVX2 __attribute__((target("avx2")))

// The largest magnitude of n values (NaNs are passed over: of a NaN and a number the maximum is the second operand), and their codes
// where an estimated quotient decides; the others are made again.
struct Avx512 {
    VTL_AVX512 static __mmask16 lanes(int64_t left) { return left >= 16 ? (__mmask16)0xffff : (__mmask16)((1u << left) - 1); }
    VTL_AVX512 static float absmax(const float *x, int64_t n)
    {
        __m512 m[4] = {_mm512_setzero_ps(), _mm512_setzero_ps(), _mm512_setzero_ps(), _mm512_setzero_ps()};
        int64_t i = 0;
        for (; i + 64 <= n; i += 64)
            for (int j = 0; j < 4; j++)
                m[j] = _mm512_max_ps(_mm512_abs_ps(_mm512_loadu_ps(x + i + 16 * j)), m[j]);
        for (; i < n; i += 16)
            m[0] = _mm512_max_ps(_mm512_abs_ps(_mm512_maskz_loadu_ps(lanes(n - i), x + i)), m[0]);
        return _mm512_reduce_max_ps(_mm512_max_ps(_mm512_max_ps(m[0], m[1]), _mm512_max_ps(m[2], m[3])));
    }
    VTL_AVX512 static void codes(const float *x, int64_t n, int8_t *q, float scale)
    {
        const __m512 inv = _mm512_set1_ps(1.0f / scale), tie = _mm512_set1_ps(kTie);
        int64_t i = 0;
        for (; i + 64 <= n; i += 64) {
            uint64_t near = 0;
            for (int j = 0; j < 4; j++) {
                const __m512 t = _mm512_mul_ps(_mm512_loadu_ps(x + i + 16 * j), inv);
                const __m512 r = _mm512_roundscale_ps(t, _MM_FROUND_TO_NEAREST_INT | _MM_FROUND_NO_EXC);
                near |= (uint64_t)_mm512_cmp_ps_mask(_mm512_abs_ps(_mm512_sub_ps(t, r)), tie, _CMP_NLT_UQ) << (16 * j);   // (a NaN too)
                _mm_storeu_si128(reinterpret_cast<__m128i *>(q + i + 16 * j), _mm512_cvtsepi32_epi8(_mm512_cvtps_epi32(r)));
            }
            again(x + i, q + i, near, scale);
        }
        for (; i < n; i += 16) {
            const __mmask16 in = lanes(n - i);
            const __m512 t = _mm512_mul_ps(_mm512_maskz_loadu_ps(in, x + i), inv);
            const __m512 r = _mm512_roundscale_ps(t, _MM_FROUND_TO_NEAREST_INT | _MM_FROUND_NO_EXC);
            _mm_mask_storeu_epi8(q + i, in, _mm512_cvtsepi32_epi8(_mm512_cvtps_epi32(r)));
            again(x + i, q + i, _mm512_mask_cmp_ps_mask(in, _mm512_abs_ps(_mm512_sub_ps(t, r)), tie, _CMP_NLT_UQ), scale);
        }
    }
    static void again(const float *x, int8_t *q, uint64_t which, float scale)
    {
        for (; __builtin_expect(which != 0, 0); which &= which - 1)
            q[__builtin_ctzll(which)] = code(x[__builtin_ctzll(which)], scale);
    }
};

// What is beyond whole steps of 32 is a step that ends with the row; rows shorter than one are made value by value.
struct Avx2 {
    VTL_AVX2 static float absmax(const float *x, int64_t n)
    {
        float most = 0.0f;
        if (n < 32) {
            for (int64_t i = 0; i < n; i++)
                most = __builtin_fabsf(x[i]) > most ? __builtin_fabsf(x[i]) : most;
            return most;
        }
        const __m256 magnitude = _mm256_castsi256_ps(_mm256_set1_epi32(0x7fffffff));
        __m256 m[4] = {_mm256_setzero_ps(), _mm256_setzero_ps(), _mm256_setzero_ps(), _mm256_setzero_ps()};
        for (int64_t i = 0; i < n; i += 32) {
            const float *at = x + (i + 32 <= n ? i : n - 32);
            for (int j = 0; j < 4; j++)
                m[j] = _mm256_max_ps(_mm256_and_ps(_mm256_loadu_ps(at + 8 * j), magnitude), m[j]);
        }
        float lane[8];
        _mm256_storeu_ps(lane, _mm256_max_ps(_mm256_max_ps(m[0], m[1]), _mm256_max_ps(m[2], m[3])));
        for (float v : lane)
            most = v > most ? v : most;
        return most;
    }
    VTL_AVX2 static void codes(const float *x, int64_t n, int8_t *q, float scale)
    {
        if (n < 32) {
            for (int64_t i = 0; i < n; i++)
                q[i] = code(x[i], scale);
            return;
        }
        const __m256 magnitude = _mm256_castsi256_ps(_mm256_set1_epi32(0x7fffffff));
        const __m256 inv = _mm256_set1_ps(1.0f / scale), tie = _mm256_set1_ps(kTie);
        const __m256i order = _mm256_setr_epi32(0, 4, 1, 5, 2, 6, 3, 7);
        for (int64_t i = 0; i < n; i += 32) {
            const int64_t at = i + 32 <= n ? i : n - 32;
            __m256i c[4];
            unsigned near = 0;
            for (int j = 0; j < 4; j++) {
                const __m256 t = _mm256_mul_ps(_mm256_loadu_ps(x + at + 8 * j), inv);
                const __m256 r = _mm256_round_ps(t, _MM_FROUND_TO_NEAREST_INT | _MM_FROUND_NO_EXC);
                near |= (unsigned)_mm256_movemask_ps(_mm256_cmp_ps(_mm256_and_ps(_mm256_sub_ps(t, r), magnitude), tie, _CMP_NLT_UQ)) << (8 * j);
                c[j] = _mm256_cvtps_epi32(r);
            }
            const __m256i all = _mm256_packs_epi16(_mm256_packs_epi32(c[0], c[1]), _mm256_packs_epi32(c[2], c[3]));
            _mm256_storeu_si256(reinterpret_cast<__m256i *>(q + at), _mm256_permutevar8x32_epi32(all, order));
            for (; __builtin_expect(near != 0, 0); near &= near - 1)
                q[at + __builtin_ctz(near)] = code(x[at + __builtin_ctz(near)], scale);
        }
    }
};

template <typename V>
void codes_of(const float *x, int64_t n, int8_t *q, float scale)
{
    if (by_estimate(scale)) {
        V::codes(x, n, q, scale);
        return;
    }
    for (int64_t i = 0; i < n; i++)
        q[i] = code(x[i], scale);
}

template <typename V>
void scaled(const float *x, int64_t rows, int64_t cols, int8_t *q, int64_t row, float scale)
{
    const DefaultFloats mode;
    asm volatile("" : "+m"(scale));
    for (int64_t r = 0; r < rows; r++, x += cols, q += row) {
        codes_of<V>(x, cols, q, scale);
        memset(q + cols, 0, (size_t)(row - cols));
    }
}

template <typename V>
void rows_of(const float *x, int64_t rows, int64_t cols, int8_t *q, int64_t row, float *scales)
{
    const DefaultFloats mode;
    for (int64_t r = 0; r < rows; r++, x += cols, q += row) {
        scales[r] = V::absmax(x, cols) / 127.0f;
        codes_of<V>(x, cols, q, scales[r]);
        memset(q + cols, 0, (size_t)(row - cols));
    }
}

template <typename V>
float absmax(const float *x, int64_t count)
{
    float m;
    {
        const DefaultFloats mode;
        m = V::absmax(x, count);
        asm volatile("" : "+m"(m));
    }
    return m;
}

float scale_of(float absmax)
{
    float scale;
    {
        const DefaultFloats mode;
        asm volatile("" : "+m"(absmax));
        scale = absmax / 127.0f;
        asm volatile("" : "+m"(scale));
    }
    return scale;
}

constexpr HostQuantizer kAvx512 = {rows_of<Avx512>, scaled<Avx512>, absmax<Avx512>, scale_of};
constexpr HostQuantizer kAvx2 = {rows_of<Avx2>, scaled<Avx2>, absmax<Avx2>, scale_of};

}  // namespace

const HostQuantizer *host_quantizer()
{
    static const bool wide = __builtin_cpu_supports("avx512f") && __builtin_cpu_supports("avx512bw") &&
                             __builtin_cpu_supports("avx512vl") && __builtin_cpu_supports("avx512dq");
    static const bool any = __builtin_cpu_supports("avx2");
    return wide ? &kAvx512 : any ? &kAvx2 : nullptr;
}
#else
const HostQuantizer *host_quantizer() { return nullptr; }
#endif

}  // namespace vtlhip
