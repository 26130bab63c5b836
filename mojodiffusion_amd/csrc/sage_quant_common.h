// sage_quant_common.h — the quantizers' arithmetic that more than one kernel needs: element conversions, which keys count,
// and what turns a channel's sum, minimum and maximum into its mean and balancing factor.
#pragma once

#include "sage_internal.h"

#include <hip/hip_fp16.h>

namespace sage {

typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

// Running maximum of the magnitudes of bf16 pairs, as 16-bit integers: of one order with the values
// themselves, infinities and NaNs on top (>= 0x7F80).  One packed instruction per pair.
__device__ __forceinline__ uint32_t bf16_mag_max(uint32_t acc, uint32_t pair) {
    const u16x2 m = __builtin_elementwise_max(__builtin_bit_cast(u16x2, acc), __builtin_bit_cast(u16x2, pair & 0x7FFF7FFFu));
    return __builtin_bit_cast(uint32_t, m);
}
__device__ __forceinline__ bool bf16_mag_finite(uint32_t acc) { return (acc & 0xFFFFu) < 0x7F80u && (acc >> 16) < 0x7F80u; }

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xFFFF0000u); }

__device__ __forceinline__ void unpack8(const u32x4& w, float* x) {
    x[0] = bf16_lo(w.x); x[1] = bf16_hi(w.x);
    x[2] = bf16_lo(w.y); x[3] = bf16_hi(w.y);
    x[4] = bf16_lo(w.z); x[5] = bf16_hi(w.z);
    x[6] = bf16_lo(w.w); x[7] = bf16_hi(w.w);
}

__device__ __forceinline__ void load8(const float* p, float* x) {
    const float4 a = *reinterpret_cast<const float4*>(p);
    const float4 b = *reinterpret_cast<const float4*>(p + 4);
    x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
    x[4] = b.x; x[5] = b.y; x[6] = b.z; x[7] = b.w;
}

__device__ __forceinline__ bool key_kept(int s, int N, const KeyMask& m) { return s < N && !(s >= m.lo && s < m.hi); }

// Two values -> fp16, rounded to nearest even, finite overflow and infinities to +-65504, NaN to -65504 (the median of a NaN
// and two numbers is the lesser of those).  One operation and a half per element.
__device__ __forceinline__ uint32_t f16_pair_sat(float a, float b) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const h2 h = {(_Float16)__builtin_amdgcn_fmed3f(a, -65504.0f, 65504.0f), (_Float16)__builtin_amdgcn_fmed3f(b, -65504.0f, 65504.0f)};
    return __builtin_bit_cast(uint32_t, h);
}

// fp32 -> e4m3fn, round-to-nearest-even, saturating at +-448, NaN -> +-0.
__device__ __forceinline__ uint32_t f32_to_e4m3(float x) {
    const uint32_t u = __float_as_uint(x);
    const uint32_t sign = (u >> 24) & 0x80u;
    float a = fabsf(x);
    if (!(a == a)) return sign;
    a = fminf(a, 448.0f);
    uint32_t byte;
    if (a < 0.015625f) {                                   // below 2^-6: quantum 2^-9
        byte = (uint32_t)(int)rintf(a * 512.0f);           // 0..8; 8 is exactly code 0x08
    } else {
        const uint32_t au = __float_as_uint(a);
        // keep 3 mantissa bits, round half to even on the 20 dropped bits
        uint32_t r = au + 0x7FFFFu + ((au >> 20) & 1u);
        r >>= 20;                                          // (biased exp << 3) | mant3, carry included
        byte = r - ((127u - 7u) << 3);
        if (byte > 0x7Eu) byte = 0x7Eu;
    }
    return byte | sign;
}

__device__ __forceinline__ void k_final(double sum, float mn, float mx, int kept, int flags, float& mean, float& s) {
    mean = 0.0f;
    s = 1.0f;
    if (flags & 1) mean = (float)(sum / (double)kept);
    if (flags & 2) {
        const float amax = fmaxf(fabsf(mx - mean), fabsf(mn - mean));
        if (amax > 0.0f) s = sqrtf(amax);
    }
}

// the channel whose results thread t < D adds up
template <int D> __device__ __forceinline__ int leaf_channel(int t) { return t % (D / 8) * 8 + t / (D / 8); }

}  // namespace sage
