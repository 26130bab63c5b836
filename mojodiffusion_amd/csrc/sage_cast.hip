// sage_cast.hip — F32 <-> bf16 of up to four tensors in one launch (gfx950): callers with F32 activations
// cast q, k and v at the boundary and O on the way out (dO and the gradients: sage_bwd.hip), and a launch per tensor costs more than
// the copy itself at a trainer's sizes ([1,2304,12,64]: 4.5 us each for 10.6 MB).  Bound by memory: 16-byte
// loads and stores, eight elements per thread.
#include "sage_internal.h"

namespace sage {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t pack_rne(float a, float b) {
    const v2f f = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, v2bf));
}

constexpr int kPerBlock = 256 * 8;

template <bool TO_BF16>
__global__ __launch_bounds__(256) void cast_kernel(CastArgs a) {
    unsigned blk = blockIdx.x;
    int t = 0;
    while (t < a.count - 1 && blk >= a.blocks[t]) blk -= a.blocks[t++];
    const int64_t i = (int64_t)blk * kPerBlock + threadIdx.x * 8, n = a.n[t];
    if (i >= n) return;
    if (TO_BF16) {
        const float* src = static_cast<const float*>(a.src[t]) + i;
        uint16_t* dst = static_cast<uint16_t*>(a.dst[t]) + i;
        if (i + 8 <= n) {
            const v4f x = *reinterpret_cast<const v4f*>(src), y = *reinterpret_cast<const v4f*>(src + 4);
            *reinterpret_cast<u32x4*>(dst) = u32x4{pack_rne(x[0], x[1]), pack_rne(x[2], x[3]), pack_rne(y[0], y[1]), pack_rne(y[2], y[3])};
        } else {
            for (int64_t e = 0; i + e < n; e++) dst[e] = (uint16_t)pack_rne(src[e], 0.0f);
        }
    } else {
        const uint16_t* src = static_cast<const uint16_t*>(a.src[t]) + i;
        float* dst = static_cast<float*>(a.dst[t]) + i;
        if (i + 8 <= n) {
            const u32x4 w = *reinterpret_cast<const u32x4*>(src);
            v4f x, y;
#pragma unroll
            for (int e = 0; e < 2; e++) {
                x[2 * e] = __uint_as_float(w[e] << 16); x[2 * e + 1] = __uint_as_float(w[e] & 0xFFFF0000u);
                y[2 * e] = __uint_as_float(w[2 + e] << 16); y[2 * e + 1] = __uint_as_float(w[2 + e] & 0xFFFF0000u);
            }
            *reinterpret_cast<v4f*>(dst) = x;
            *reinterpret_cast<v4f*>(dst + 4) = y;
        } else {
            for (int64_t e = 0; i + e < n; e++) dst[e] = __uint_as_float((uint32_t)src[e] << 16);
        }
    }
}

hipError_t launch_cast(const CastArgs& a_in, bool to_bf16, hipStream_t st) {
    CastArgs a = a_in;
    int64_t total = 0;
    for (int t = 0; t < a.count; t++) {
        const int64_t b = (a.n[t] + kPerBlock - 1) / kPerBlock;
        total += b;
        if (total > 0x7FFFFFFF) return hipErrorInvalidValue;
        a.blocks[t] = (unsigned)b;
    }
    if (total == 0) return hipSuccess;
    if (to_bf16) hipLaunchKernelGGL(cast_kernel<true>, dim3((unsigned)total), dim3(256), 0, st, a);
    else hipLaunchKernelGGL(cast_kernel<false>, dim3((unsigned)total), dim3(256), 0, st, a);
    return hipGetLastError();
}

}  // namespace sage
