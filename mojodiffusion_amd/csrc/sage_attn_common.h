// sage_attn_common.h — what the attention kernels share: vector types, the biased score accumulators, the
// reference-maximum rule and the bf16 rounding of their outputs.
#pragma once

#include "sage_internal.h"

namespace sage {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));

// Byte offset of 16-byte chunk L of a tile.  Chunks are grouped into 128-byte super-rows
// (8 chunks); the chunk position inside a super-row is XORed with bits of the index of
// the PAIR of super-rows it belongs to, so that the 16 lanes the 64-bank LDS serves per
// cycle (16 consecutive rows, one logical column) land in 16 different 16-byte bank groups.
__device__ __forceinline__ int swz(int L) { return (((L >> 3) << 3) | ((L & 7) ^ ((L >> 4) & 7))) << 4; }

// 16 bytes per lane from global memory straight into LDS: lane l of the wave lands at
// lds_base + 16*l.  Written as assembly on purpose: the compiler then keeps no record of
// an outstanding LDS write and does not put a full vector-memory wait in front of every
// later LDS read; completion is awaited explicitly (dma_wait) before the workgroup
// barrier that publishes the tile.
__device__ __forceinline__ void dma16(const void* gbase_uniform, uint32_t goff, uint32_t lds_base_uniform) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(lds_base_uniform), "v"(goff), "s"(gbase_uniform)
                 : "memory");      // (m0 cannot be named as a clobber: to this compiler it is a reserved register — it
                                   // warns that "clobbering them may lead to undefined behaviour" — which it never
                                   // keeps a value in across statements; its own uses set m0 right before the use)
}
// Wait until at most N of this wave's copies are still in flight (they complete in order).
template <int N> __device__ __forceinline__ void dma_wait() {
    static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

__device__ __forceinline__ uint32_t lds_addr(const void* p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}

// Two floats -> packed bf16, round to nearest even.
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    const v2f f = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, v2bf));
}

// The int32 score accumulators start at the bit pattern of the float 1/(2*pi) instead of 0.
// That pattern is 2^-3 * (1 + 2292099 * 2^-23), so adding an integer dot with
// |dot| < 2292099 (the largest possible |dot| is 128*127*127 = 2064512) changes only the
// mantissa: a finished accumulator, read as fp32, IS the float 1/(2*pi) + dot * 2^-26.  No
// int->float conversion is needed and dequantisation, max subtraction and the exponent
// argument collapse into one FMA per score (the scale carries the factor 2^26).
constexpr int kMagicI = 0x3E22F983;
constexpr float kMagicF = 0.15915494309189532f;        // the same 32 bits
constexpr float kMagicUnit = 67108864.0f;               // 2^26: accumulator-as-float steps per integer
// With 256 channels |dot| can reach 256*127*127 = 4129024, more than the mantissa of 1/(2*pi) has
// room for below it.  0.1875 = 2^-3 * (1 + 2^22 * 2^-23) leaves 2^22 = 4194304 either way at the
// same step of 2^-26.
constexpr int kMagicWideI = 0x3E400000;
constexpr float kMagicWideF = 0.1875f;
// e4m3 variant: a wave whose bias * f can exceed this takes the bias off its accumulators (see exact_bias).
constexpr float kExactBias = 4096.0f;
template <int D> struct Magic {
    static constexpr int I = D > 128 ? kMagicWideI : kMagicI;
    static constexpr float F = D > 128 ? kMagicWideF : kMagicF;
};

// The score scale of a step that holds masked scores: at least the smallest normal number, because -inf times a scale
// that has underflowed to zero is NaN.  (A real score times a scale below it is 0 in the exponent either way; a NaN
// scale stays one.)
static __device__ __forceinline__ float masked_scale(float f) { return f < 0x1p-126f ? 0x1p-126f : f; }

// First matrix instruction of a score chain: accumulator input = the constant above, held in 16
// registers for the whole kernel (behind an empty statement, or the compiler re-creates the 16
// copies for every chain).  The instruction could take 1/(2*pi) as an inline operand, but only
// written as assembly, and then the compiler does not know that a matrix instruction is writing
// those registers: it neither keeps the wait states before the first other instruction that
// touches them — a spill store two instructions later wrote the old contents — nor can it be told.
template <int D>
__device__ __forceinline__ v16i magic_splat() {
    constexpr int M = Magic<D>::I;
    v16i c = {M, M, M, M, M, M, M, M, M, M, M, M, M, M, M, M};
    asm volatile("" : "+v"(c));
    return c;
}

// A row's reference maximum is only refreshed (and the accumulators rescaled) when a tile
// exceeds it by more than tau powers of two; until then p = exp2(s - m_used) may reach
// 2^tau.  fp16 P holds 2^8 without loss.  The e4m3 variant maps p = 2^tau to the format
// maximum 448, i.e. it stores e4m3(p * 448 / 2^tau); the factor cancels against the
// normaliser, which sums the same scaled values.  Its reference is always a whole number
// (the maximum rounded up): a probability's e4m3 significand then depends on the fractional
// part of its score only, not on which whole number the reference happens to be, so the
// stored probabilities are those of a softmax taken against ceil(row maximum) up to a power
// of two, and the rescale factors are exact.
template <int VARIANT> struct Lazy {
    static constexpr float tau = VARIANT == 0 ? 8.0f : 1.0f;
    static constexpr float log2_pscale = VARIANT == 0 ? 0.0f : 7.807354922057604f;     // log2(448 / 2)
    static constexpr bool integer_ref = VARIANT == 1;
};

// Eight scaled values of a row -> int8 codes: the quantizer's arithmetic (quant_i8_block in
// sage_quant.hip: one fused multiply-add with a magic addend per code, the true quotient where some lane
// comes close to a rounding tie).  The whole wave calls it.
__device__ __forceinline__ u32x2 encode8_i8(const float (&x)[8], float sc, float rinv, bool fast) {
    float kRound = 12582912.0f, rv = rinv;
    asm volatile("" : "+v"(rv), "+v"(kRound));
    uint32_t tb[8], wd[2];
    float dm = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
        const float t0 = fmaf(x[e], rv, kRound), t1 = fmaf(x[e + 1], rv, kRound);
        const float d0 = fmaf(x[e], rv, -(t0 - kRound)), d1 = fmaf(x[e + 1], rv, -(t1 - kRound));
        dm = fmaxf(fmaxf(dm, fabsf(d0)), fabsf(d1));
        tb[e] = __float_as_uint(t0);
        tb[e + 1] = __float_as_uint(t1);
    }
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const uint32_t lo = __builtin_amdgcn_perm(tb[4 * j + 1], tb[4 * j], 0x0c0c0400u);
        const uint32_t hi = __builtin_amdgcn_perm(tb[4 * j + 3], tb[4 * j + 2], 0x0c0c0400u);
        wd[j] = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
    }
    if (__builtin_expect(!fast || __any(!(dm <= 0.5f - 0x1p-16f)), 0)) {
        asm volatile("" ::: "memory");
        wd[0] = wd[1] = 0u;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            float r = rint_quotient(x[e], sc, rinv, fast);
            r = r > 127.0f ? 127.0f : r;
            r = r < -127.0f ? -127.0f : r;
            wd[e >> 2] |= ((uint32_t)((int)r) & 0xFFu) << ((e & 3) * 8);
        }
    }
    return u32x2{wd[0], wd[1]};
}

// The same in two parts, for loops over several chunks: the common case, which says whether some lane of the wave comes close to a
// tie, and the true quotient, in a loop over the chunks that did (redo_chunks).  Inside the unrolled loop the true quotient's eight divides
// are two kilobytes of code to jump over per chunk.
__device__ __forceinline__ u32x2 encode8_common(const float (&x)[8], float rinv, bool& near) {
    float kRound = 12582912.0f, rv = rinv;
    asm volatile("" : "+v"(rv), "+v"(kRound));
    uint32_t tb[8], wd[2];
    float dm = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
        const float t0 = fmaf(x[e], rv, kRound), t1 = fmaf(x[e + 1], rv, kRound);
        const float d0 = fmaf(x[e], rv, -(t0 - kRound)), d1 = fmaf(x[e + 1], rv, -(t1 - kRound));
        dm = fmaxf(fmaxf(dm, fabsf(d0)), fabsf(d1));
        tb[e] = __float_as_uint(t0);
        tb[e + 1] = __float_as_uint(t1);
    }
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const uint32_t lo = __builtin_amdgcn_perm(tb[4 * j + 1], tb[4 * j], 0x0c0c0400u);
        const uint32_t hi = __builtin_amdgcn_perm(tb[4 * j + 3], tb[4 * j + 2], 0x0c0c0400u);
        wd[j] = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
    }
    near = __any(!(dm <= 0.5f - 0x1p-16f));
    return u32x2{wd[0], wd[1]};
}
__device__ __forceinline__ u32x2 encode8_quotient(const float (&x)[8], float sc, float rinv, bool fast) {
    uint32_t wd[2] = {0u, 0u};
#pragma unroll
    for (int e = 0; e < 8; e++) {
        float r = rint_quotient(x[e], sc, rinv, fast);
        r = r > 127.0f ? 127.0f : r;
        r = r < -127.0f ? -127.0f : r;
        wd[e >> 2] |= ((uint32_t)((int)r) & 0xFFu) << ((e & 3) * 8);
    }
    return u32x2{wd[0], wd[1]};
}
// redo(i) for the set bits of a wave's mask.
template <typename F> __device__ __forceinline__ void redo_chunks(uint32_t mask, F redo) {
    mask = __builtin_amdgcn_readfirstlane(mask);
#pragma unroll 1
    while (__builtin_expect(mask != 0u, 0)) {
        redo(__builtin_ctz(mask));
        mask &= mask - 1u;
    }
}

// ---- additive bias: 32 rows x 32 keys of a wave ------------------------------------------------------
// Loaded 16 bytes per lane, whole rows next to each other (a lane's own four keys of its own row, the layout
// the scores have, are 64 separate pieces per instruction: 4 to 8 of them per step took longer than the
// step's arithmetic, and twice as long where odd key counts start the rows anywhere), turned into the scores'
// layout through LDS.  16-byte chunks of a row are XORed with the row, so that both sides touch every bank.
struct BiasStage {
    static constexpr int CPR = 4, RPI = 64 / CPR, NI = 32 / RPI;                 // chunks per row, rows per load, loads
    static constexpr int BYTES = 32 * 64;
    u32x4 w[NI];

    static __device__ __forceinline__ int at(int row, int chunk) { return row * 64 + ((chunk ^ ((row >> 2) & 3)) << 4); }
    // the lane's rows of row0 .. row0 + 31 (rows past the last repeat it)
    struct Rows { const uint16_t* p[NI]; };
    static __device__ __forceinline__ Rows rows(const uint16_t* head, int64_t row_stride, int row0, int last_row, int lane) {
        Rows r;
#pragma unroll
        for (int i = 0; i < NI; i++) r.p[i] = head + (int64_t)min(row0 + i * RPI + lane / CPR, last_row) * row_stride;
        return r;
    }
    // Keys key0 .. key0 + 31 of those rows, n of which there are.  Rows start at any even byte address: the access is as
    // wide as the hardware takes it unaligned.  A chunk that reaches past its row's end is loaded as the row's last eight
    // keys and shifted on its way to LDS: one load for all lanes, nothing past a row's end is read.  (Rows of fewer than
    // eight keys are taken key by key.)
    __device__ __forceinline__ void load(const Rows& r, int key0, int n, int lane) {
        const int key = key0 + (lane % CPR) * 8;
        if (__builtin_expect(n >= 8, 1)) {
#pragma unroll
            for (int i = 0; i < NI; i++) __builtin_memcpy(&w[i], r.p[i] + min(key, n - 8), 16);
        } else {
#pragma unroll
            for (int i = 0; i < NI; i++) {
                uint32_t v[4] = {0u, 0u, 0u, 0u};
#pragma unroll
                for (int e = 0; e < 8; e++)
                    if (key + e < n) v[e >> 1] |= (uint32_t)r.p[i][key + e] << ((e & 1) * 16);
                w[i] = u32x4{v[0], v[1], v[2], v[3]};
            }
        }
    }
    // (keys at and past n are 0)
    __device__ __forceinline__ void put(uint8_t* lds, int lane, int key0, int n) const {
#pragma unroll
        for (int i = 0; i < NI; i++) {
            u32x4 x = w[i];
            if (__builtin_expect(key0 + 32 > n && n >= 8, 0)) {
                const int d = key0 + (lane % CPR) * 8 - (n - 8);        // keys to shift out
                if (d & 4) x = u32x4{x.z, x.w, 0u, 0u};
                if (d & 2) x = u32x4{x.y, x.z, x.w, 0u};
                if (d & 1) x = u32x4{(x.x >> 16) | (x.y << 16), (x.y >> 16) | (x.z << 16), (x.z >> 16) | (x.w << 16), x.w >> 16};
                if (d >= 8) x = u32x4{0u, 0u, 0u, 0u};
                if (d <= 0) x = w[i];
            }
            *reinterpret_cast<u32x4*>(lds + at(i * RPI + lane / CPR, lane % CPR)) = x;
        }
    }
    // keys g * 8 + half * 4 .. + 3 of row l32
    static __device__ __forceinline__ u32x2 get_packed(const uint8_t* lds, int l32, int half, int g) {
        return *reinterpret_cast<const u32x2*>(lds + at(l32, g) + half * 8);
    }
    static __device__ __forceinline__ v4f get(const uint8_t* lds, int l32, int half, int g) {
        const u32x2 v = get_packed(lds, l32, half, g);
        return v4f{__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xFFFF0000u), __uint_as_float(v.y << 16), __uint_as_float(v.y & 0xFFFF0000u)};
    }
};

}  // namespace sage
