// sage_quant.hip — HBM-bound kernels of the quantized-SDPA path (gfx950), one launch for short key sequences
// (quant_short_kernel) and, in one-shot calls, for those of up to 8192 keys (quant_once_kernel); three otherwise, two for up to ten groups of
// 256 keys (quant_adds_up):
//
//   prep_kernel         per (b,h), workgroup roles:  V repack to tiled fp16  |  V channel
//                       maxima per 256-token group (e4m3 variant)  |  K channel sums (fp64),
//                       minima and maxima per 256-token group
//   stats_final_kernel  per (b,h,channel): K mean, balancing factor -> kmean, qmul, kmul;
//                       V maxima -> vscale
//   quant_kernel        per (b,h), workgroup roles:  Q blocks -> int8 + scale  |  K blocks ->
//                       int8 + scale  |  V tiles -> e4m3 (e4m3 variant)
//
// Every fp32 step that decides a code is a single IEEE operation (true divide, IEEE sqrt,
// round-half-to-even) and every reduction either has a fixed order (the fp64 sums) or is
// order-free (max / min), so codes, scales and statistics are reproducible bit for bit.
// All kernels read bf16 rows with 16-byte loads (8 channels per lane).
#include "sage_attn_common.h"
#include "sage_grid.h"
#include "sage_quant_common.h"

namespace sage {

// A lane exchange inside rows of 16 lanes that goes with the vector instruction, not through the LDS pipe.
template <int CTRL> __device__ __forceinline__ float dpp(float x) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(x), CTRL, 0xF, 0xF, false));
}
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppXor3 = 0x1B, kDppXor7 = 0x141, kDppRor = 0x120;      // quad_perm, row_half_mirror, row_ror
__device__ __forceinline__ float xor4(float x) { return dpp<kDppXor7>(dpp<kDppXor3>(x)); }
__device__ __forceinline__ float xor8(float x) { return dpp<kDppRor + 8>(x); }

// RMSNorm (+ RoPE) of rows spread over the D/8 consecutive lanes that hold their 16-byte chunks: x[0..7] are
// channels col..col+7.  Every lane of the group must call these (they exchange partial sums).
// Arithmetic, step for step (all fp32, no fused multiply-add):
//   the squares are added in the order of serenitymojo/ops/norm.mojo:56-72 — a 256-slot array
//   folded in halves, far pairs first: channel t with t+64 (D = 128), then strides 32, 16 and
//   8, which pair lanes of the row, then 4, 2, 1 inside the lane;
//   inv = 1/sqrt(sum/D + eps); y = bf16((x*inv)*gain); rotation of (y[2i], y[2i+1]) by
//   the table angle with both products rounded before the subtract / add; result bf16.
//   (p.halfsplit: the pairs are (y[i], y[i + D/2]) instead.)
// What bounds the kernels that use them is vector instructions, so: the exchanges are DPP modifiers of the adds
// (as LDS permutes they were 32 of them per 16-byte chunk), a row's square root and reciprocal are taken by one
// lane of its group instead of by all (row_inverses), and both roundings are the conversion instruction
// (half an operation per element instead of six).  Behind that it is latency: table entries are requested ahead
// (see RopeTab).  [2,4352,30,128], us: K statistics 89 -> 47, encoders (with the V repack) 174 -> 111.  Dealing the
// workgroups so that Q, K and the batch items share table rows in an XCD's L2 measured slower (K statistics 69).
template <int D>
__device__ __forceinline__ float row_square_sum(const float* x) {
    constexpr int CPR = D / 8;
    static_assert(CPR == 8 || CPR == 16, "rows of 8 or 16 lanes");
    float sq[8];
#pragma unroll
    for (int e = 0; e < 8; e++) sq[e] = x[e] * x[e];
    if constexpr (CPR == 16) {
        // (after the first step lanes l and l + 8 agree, after the second l and l + 4, ...: a rotation then
        // reaches the same value as the exclusive-or)
#pragma unroll
        for (int e = 0; e < 8; e++) sq[e] = sq[e] + xor8(sq[e]);
#pragma unroll
        for (int e = 0; e < 8; e++) sq[e] = sq[e] + dpp<kDppRor + 4>(sq[e]);
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++) sq[e] = sq[e] + xor4(sq[e]);
    }
#pragma unroll
    for (int e = 0; e < 8; e++) sq[e] = sq[e] + dpp<kDppXor2>(sq[e]);
#pragma unroll
    for (int e = 0; e < 8; e++) sq[e] = sq[e] + dpp<kDppXor1>(sq[e]);
#pragma unroll
    for (int e = 0; e < 4; e++) sq[e] = sq[e] + sq[e + 4];
    sq[0] = sq[0] + sq[2];
    sq[1] = sq[1] + sq[3];
    return sq[0] + sq[1];
}

// inv[i] = 1/sqrt(mean square of row i + eps) for the N rows of a lane group whose chunks are w[0..N-1]: lane j
// of the group takes the root of row j.
template <int D, int N>
__device__ __forceinline__ void row_inverses(float eps, const u32x4 (&w)[N], float (&inv)[N]) {
    constexpr int CPR = D / 8;
    const int lane = threadIdx.x & 63, j = lane % CPR;
#pragma unroll
    for (int i0 = 0; i0 < N; i0 += CPR) {
        float mine = 0.0f;
#pragma unroll
        for (int i = 0; i < CPR && i0 + i < N; i++) {
            float x[8];
            unpack8(w[i0 + i], x);
            const float sum = row_square_sum<D>(x);
            mine = j == i ? sum : mine;
            asm volatile("" : "+v"(mine));          // (or the compiler gathers the sums in an array in memory and indexes it)
        }
        const float mean = mine / (float)D;
        const float r = 1.0f / sqrtf(mean + eps);
#pragma unroll
        for (int i = 0; i < CPR && i0 + i < N; i++) inv[i0 + i] = __shfl(r, (lane & ~(CPR - 1)) + i, 64);
    }
}

__device__ __forceinline__ void round8_to_bf16(float* x) {
    typedef float v2f __attribute__((ext_vector_type(2)));
    typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
        const v2f f = {x[e], x[e + 1]};
        const uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector(f, v2bf));     // round to nearest even
        x[e] = bf16_lo(w);
        x[e + 1] = bf16_hi(w);
    }
}

// gains of the thread's channels (with a statistic of the whole token: H*D of them)
__device__ __forceinline__ void pre_gains(const PreOp& p, int h, int D, int col, float* g) {
    unpack8(*reinterpret_cast<const u32x4*>(p.gain + (p.row_inv != nullptr ? h * D : 0) + col), g);
}

// Table entries of one chunk, requested AHEAD chunks ahead.  PRE 1: 16 bytes of cosines and of sines, whatever
// the layout (bf16 tables of interleaved pairs: the 16 bytes around the 8 that are needed; no tables: the
// gains, which are not looked at) — the same loads in every case, because behind a branch around a load the compiler
// has to wait for every load in flight.  PRE 2: half-split pairs with fp32 tables, 32 bytes of each.
template <int PRE> struct RopeTab { u32x4 c[PRE > 0 ? PRE : 1], s[PRE > 0 ? PRE : 1]; };
struct RopeAt { const uint8_t *c, *s; int64_t row_bytes; };
template <int D>
__device__ __forceinline__ RopeAt rope_at(const PreOp& p, int b, int h, int H, int col) {
    const uint8_t* gain = reinterpret_cast<const uint8_t*>(p.gain + col);
    if (p.cos == nullptr) return RopeAt{gain, gain, 0};
    const int esz = p.tables_bf16 ? 2 : 4;
    const int at = ((p.halfsplit ? col & (D / 2 - 1) : col / 2) * esz) & ~15;
    const int64_t off = ((int64_t)b * p.batch_rows + h) * (D / 2) * esz + at;
    return RopeAt{reinterpret_cast<const uint8_t*>(p.cos) + off, reinterpret_cast<const uint8_t*>(p.sin) + off, (int64_t)H * (D / 2) * esz};
}
template <int PRE>
__device__ __forceinline__ void rope_load(const RopeAt& r, int row, RopeTab<PRE>& t) {
#pragma unroll
    for (int i = 0; i < PRE; i++) {
        t.c[i] = *reinterpret_cast<const u32x4*>(r.c + (int64_t)row * r.row_bytes + i * 16);
        t.s[i] = *reinterpret_cast<const u32x4*>(r.s + (int64_t)row * r.row_bytes + i * 16);
    }
}

// The rest of the pre-op for one row: normalise with `inv`, rotate; `valid` false = a padding row, which stays zero.
template <int D, int PRE>
__device__ __forceinline__ void pre_apply(const PreOp& p, int col, bool valid, float inv, const float* g, const RopeTab<PRE>& tab, float* x) {
    constexpr int CPR = D / 8;
    float y[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const float t = x[e] * inv;
        y[e] = t * g[e];
    }
    round8_to_bf16(y);
    if (PRE == 2 || (p.cos != nullptr && p.halfsplit)) {
        // pairs (i, i + D/2): the partner channel sits in the lane CPR/2 further on (or back) among
        // the CPR lanes of this row; both lanes of a pair use table entries (col mod D/2) .. +7
        float yp[8];
#pragma unroll
        for (int e = 0; e < 8; e++) yp[e] = CPR == 16 ? xor8(y[e]) : xor4(y[e]);
        const bool upper = col >= D / 2;
        float cv[8], sv[8];
        if constexpr (PRE == 2) {
#pragma unroll
            for (int e = 0; e < 8; e++) cv[e] = __uint_as_float(tab.c[e >> 2][e & 3]), sv[e] = __uint_as_float(tab.s[e >> 2][e & 3]);
        } else {
            unpack8(tab.c[0], cv);
            unpack8(tab.s[0], sv);
        }
#pragma unroll
        for (int e = 0; e < 8; e++) {
            // lower half: x0*c - x1*s with x0 = own, x1 = partner; upper half: x1*c + x0*s with x1 = own
            const float own = y[e] * cv[e], oth = yp[e] * sv[e];
            x[e] = upper ? own + oth : own - oth;
        }
        round8_to_bf16(x);
    } else if (p.cos != nullptr) {
        float cv[4], sv[4];
        if (p.tables_bf16) {
            const bool hi = (col >> 3) & 1;
            const u32x2 c = hi ? u32x2{tab.c[0].z, tab.c[0].w} : u32x2{tab.c[0].x, tab.c[0].y};
            const u32x2 s = hi ? u32x2{tab.s[0].z, tab.s[0].w} : u32x2{tab.s[0].x, tab.s[0].y};
            cv[0] = bf16_lo(c.x); cv[1] = bf16_hi(c.x); cv[2] = bf16_lo(c.y); cv[3] = bf16_hi(c.y);
            sv[0] = bf16_lo(s.x); sv[1] = bf16_hi(s.x); sv[2] = bf16_lo(s.y); sv[3] = bf16_hi(s.y);
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) cv[i] = __uint_as_float(tab.c[0][i]), sv[i] = __uint_as_float(tab.s[0][i]);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float y0 = y[2 * i], y1 = y[2 * i + 1];
            const float p00 = y0 * cv[i], p11 = y1 * sv[i], p01 = y0 * sv[i], p10 = y1 * cv[i];
            x[2 * i] = p00 - p11;
            x[2 * i + 1] = p01 + p10;
        }
        round8_to_bf16(x);
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++) x[e] = y[e];
    }
    if (!valid) {
#pragma unroll
        for (int e = 0; e < 8; e++) x[e] = 0.0f;
    }
}

// ---------------------------------------------------------------------------
// Per-block INT8 quantization.  NT threads (`tid` counts them) per block of BLK tokens of one
// (b,h); the BLK x D tile lives in registers between the absmax pass and the encode pass, so
// HBM sees one read of bf16 and one write of int8.
// ---------------------------------------------------------------------------
// Q (IS_K false): x = f32(q) * chmul[d].  K (IS_K true): x = (f32(k) - mean[d]) * chmul[d];
// tokens that are masked or beyond N count for nothing and get code 0.
// rowdot (Q only, may be null): <f32(q) * cmul, mean> per row.
// HAVE: the threads have requested the block's rows before (have: as the loop below loads them).
template <int D, int BLK, bool IS_K, int PRE, int NT, bool HAVE = false>
__device__ __forceinline__ void quant_i8_block(
    int t, int h, int b, int tid, const uint16_t* __restrict__ x, int64_t sb, int64_t sh, int64_t sn,
    int N, int H, int64_t n_pad, const KeyMask& km, const float* __restrict__ mean,
    const float* __restrict__ chmul, float cmul,
    int8_t* __restrict__ codes, float* __restrict__ scales, float* __restrict__ rowdot, float* red,
    const PreOp& pre, const u32x4* have = nullptr) {
    constexpr int CPR = D / 8;                 // 16-byte chunks per row
    constexpr int NCH = BLK * CPR / NT;        // chunks per thread
    static_assert(BLK * CPR % NT == 0, "tile must split evenly over the threads");
    static_assert(NT % CPR == 0, "a thread keeps one column group for all its chunks");
    const int r0 = t * BLK;
    const int col = (tid % CPR) * 8;
    const int64_t bh = (int64_t)b * H + h;
    const uint16_t* src = x + b * sb + h * sh;

    u32x4 raw[NCH];
#pragma unroll
    for (int i = 0; i < NCH; i++) {
        if constexpr (HAVE) {
            raw[i] = have[i];
        } else {
            const int row = r0 + (i * NT + tid) / CPR;
            raw[i] = u32x4{0u, 0u, 0u, 0u};
            if (row < N) raw[i] = *reinterpret_cast<const u32x4*>(src + (int64_t)row * sn + col);
        }
    }
    float mul[8], mu[8];
    load8(chmul + col, mul);
    if (IS_K || rowdot != nullptr) load8(mean + col, mu);

    float v[NCH][8];
    float amax = 0.0f;
    float inv[NCH], gain[8];
    constexpr int AHEAD = HAVE && PRE == 2 ? 1 : 2;      // (four take the kernel from three waves per SIMD to two)
    RopeTab<PRE> tab[AHEAD];
    auto clamped = [&](int i) { return min(r0 + (i * NT + tid) / CPR, N - 1); };
    RopeAt rope{};
    if constexpr (PRE) {
        rope = rope_at<D>(pre, b, h, H, col);
#pragma unroll
        for (int i = 0; i < AHEAD && i < NCH; i++) rope_load<PRE>(rope, clamped(i), tab[i]);
        pre_gains(pre, h, D, col, gain);
        if (pre.row_inv == nullptr) {
            row_inverses<D, NCH>(pre.eps, raw, inv);
        } else {
#pragma unroll
            for (int i = 0; i < NCH; i++) inv[i] = pre.row_inv[(int64_t)b * pre.row_n + clamped(i)];
        }
    }
#pragma unroll
    for (int i = 0; i < NCH; i++) {
        const int row = r0 + (i * NT + tid) / CPR;
        unpack8(raw[i], v[i]);
        if constexpr (PRE) {
            pre_apply<D, PRE>(pre, col, row < N, inv[i], gain, tab[i % AHEAD], v[i]);
            if (i + AHEAD < NCH) rope_load<PRE>(rope, clamped(i + AHEAD), tab[i % AHEAD]);
        }
        bool counts;
        if (IS_K) {
            counts = key_kept(row, N, km);
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float d = v[i][e] - mu[e];
                v[i][e] = d * mul[e];
            }
        } else {
            counts = row < N;
            if (rowdot != nullptr) {
                // <pre-scaled query row, K mean>: the amount K smoothing lowers every score
                // of this row by; the CPR lanes that share a row are adjacent in the wave.
                float dot = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; e++) dot += (v[i][e] * cmul) * mu[e];
#pragma unroll
                for (int off = CPR / 2; off > 0; off >>= 1) dot += __shfl_xor(dot, off, 64);
                if ((tid % CPR) == 0) rowdot[bh * n_pad + row] = dot;
            }
#pragma unroll
            for (int e = 0; e < 8; e++) v[i][e] *= mul[e];
        }
        if (counts) {
#pragma unroll
            for (int e = 0; e < 8; e += 2) amax = fmaxf(fmaxf(amax, fabsf(v[i][e])), fabsf(v[i][e + 1]));
        }
    }

    amax = wave_max(amax);
    if ((tid & 63) == 0) red[tid >> 6] = amax;
    __syncthreads();
    amax = red[0];
#pragma unroll
    for (int w = 1; w < NT / 64; w++) amax = fmaxf(amax, red[w]);

    const float sc = amax > 0.0f ? amax / 127.0f : 1.0f;      // blocks without a counting token: amax == 0
    if (tid == 0) scales[bh * (n_pad / BLK) + t] = sc;
    const bool fast = sc >= 0x1p-100f && sc <= 0x1p100f;
    const float rinv = 1.0f / sc;

    uint32_t pk[NCH][2];
    float far[NCH] = {};        // per 16-byte chunk: how close the thread's products come to a rounding tie
    const bool all_careful = !fast;
    {
        // The common case, three operations per element and no test: t = x * rinv + 1.5 * 2^23 in one
        // fused step IS rint of the exact product p, as an integer in the low bits of t (its lowest
        // byte is the code: |p| <= 127 (1 + 2^-22) for every token that counts, so nothing needs
        // clamping); d = p minus that integer.  p differs from the true quotient by at most
        // 128 * 2^-24 (the rounding of rinv) and the true quotient is itself rounded by at most
        // 2^-18, so wherever |d| <= 1/2 - 2^-16 all three round to the same integer.  The largest
        // |d| of each chunk of eight is looked at after the loop: a chunk in which some lane of the
        // wave comes closer to a tie is encoded again with the true quotient (about one chunk in
        // seventy).  A NaN takes no part in any maximum and ends as code 0 here as there; an infinite
        // input makes the scale infinite, and such a block is encoded with the true quotient throughout.
        float kRound = 12582912.0f;                            // 1.5 * 2^23
        float rv = rinv;
        // (vector registers: the operations below then carry neither a scalar operand nor a literal,
        // and issue at the short rate)
        asm volatile("" : "+v"(rv), "+v"(kRound));
#pragma unroll
        for (int i = 0; i < NCH; i++) {
            const int row = r0 + (i * NT + tid) / CPR;
            const bool counts = IS_K ? key_kept(row, N, km) : row < N;
            uint32_t tb[8];
            float dm = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                const float t0 = fmaf(v[i][e], rv, kRound), t1 = fmaf(v[i][e + 1], rv, kRound);
                const float d0 = fmaf(v[i][e], rv, -(t0 - kRound)), d1 = fmaf(v[i][e + 1], rv, -(t1 - kRound));
                dm = fmaxf(fmaxf(dm, fabsf(d0)), fabsf(d1));
                tb[e] = __float_as_uint(t0);
                tb[e + 1] = __float_as_uint(t1);
            }
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const uint32_t lo = __builtin_amdgcn_perm(tb[4 * j + 1], tb[4 * j], 0x0c0c0400u);
                const uint32_t hi = __builtin_amdgcn_perm(tb[4 * j + 3], tb[4 * j + 2], 0x0c0c0400u);
                pk[i][j] = counts ? __builtin_amdgcn_perm(hi, lo, 0x05040100u) : 0u;
            }
            far[i] = counts ? dm : 0.0f;
        }
    }
#pragma unroll
    for (int i = 0; i < NCH; i++) {
        if (__builtin_expect(all_careful || __any(!(far[i] <= 0.5f - 0x1p-16f)), 0)) {
            asm volatile("" ::: "memory");
            const int row = r0 + (i * NT + tid) / CPR;
            pk[i][0] = pk[i][1] = 0u;
            if (IS_K ? key_kept(row, N, km) : row < N) {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    float r = rint_quotient(v[i][e], sc, rinv, fast);
                    r = r > 127.0f ? 127.0f : r;               // (comparisons: a NaN stays one; the conversion instruction makes it 0)
                    r = r < -127.0f ? -127.0f : r;
                    pk[i][e >> 2] |= ((uint32_t)((int)r) & 0xFFu) << ((e & 3) * 8);
                }
            }
        }
    }
#pragma unroll
    for (int i = 0; i < NCH; i++) {
        const int row = r0 + (i * NT + tid) / CPR;
        *reinterpret_cast<u32x2*>(codes + (bh * n_pad + row) * D + col) = u32x2{pk[i][0], pk[i][1]};
    }
}

// ---------------------------------------------------------------------------
// K channel statistics of one group of 256 tokens.  Sums follow a fixed tree, all in fp64:
//   leaf  = 16 consecutive tokens, added in ascending order by one lane
//   group = 16 consecutive leaves, added in ascending order
//   total = groups added in ascending order (stats_final_kernel)
// Tokens that are masked or beyond N add +0.0 and take no part in the minimum / maximum.
// Executed by 16*(D/8) consecutive threads; `tid` is the index among them; g < 0: idle.
// ---------------------------------------------------------------------------
// Results of the leaves on their way to the thread that adds a channel's: channel 8 c + e of a lane that holds chunk c
// sits at e * D/8 + c, so that a wave's lanes write next to each other (as channel 8 c + e the sixteen lanes of a row met
// in two or four banks), and rows are padded to the next banks.  K statistics of [1,4608,24,128] 8.9 -> 8.6 us, the
// one-launch stage of [1,1024,8,64] 9.2 -> 8.4, with one test for a whole leaf in front of its sixteen loads.
template <int D>
struct KGroupSmem {
    static constexpr int CPR = D / 8, LD = D + CPR;
    double leafsum[16][LD];
    float leafmin[16][LD];
    float leafmax[16][LD];
};
// D is the number of channels this call covers, starting at channel col0 of a head of DFULL
// channels (the statistics are per channel, so a 256-channel head is done as two windows of 128).
// Result in gsum, gmn, gmx of the threads tid < D (channel col0 + leaf_channel(tid)).
// IN_LDS: the group's rows are at `rows` in LDS, those that do not count as zeros.
template <int D, int PRE, int DFULL = D, bool IN_LDS = false>
__device__ __forceinline__ void kstats_group(
    int g, int h, int b, int tid, const uint16_t* __restrict__ k, int64_t sb, int64_t sh, int64_t sn,
    int N, int H, const KeyMask& km, KGroupSmem<D>& sm, const PreOp& pre, int col0, double& gsum, float& gmn, float& gmx,
    const u32x4* rows = nullptr) {
    static_assert(!PRE || DFULL == D, "the fused pre-ops need the whole row in one call");
    constexpr int CPR = D / 8;
    const int leaf = tid / CPR, col = (tid % CPR) * 8;
    const uint16_t* src = k + b * sb + h * sh + col0 + col;
    const int s0 = g * kGroup + leaf * kLeaf;

    // (a group past the end: its waves only meet the barrier.  Whole waves are idle or not)
    if (g >= 0) {
    u32x4 w[kLeaf];
    // every token of this leaf counts (no ragged end, no masked range inside it)
    const bool all_kept = s0 + kLeaf <= N && !(s0 < km.hi && s0 + kLeaf > km.lo);
    if constexpr (IN_LDS) {
    } else if (__all(all_kept)) {
#pragma unroll
        for (int i = 0; i < kLeaf; i++) w[i] = *reinterpret_cast<const u32x4*>(src + (int64_t)(s0 + i) * sn);
    } else {
#pragma unroll
        for (int i = 0; i < kLeaf; i++) {
            w[i] = u32x4{0u, 0u, 0u, 0u};
            if (key_kept(s0 + i, N, km)) w[i] = *reinterpret_cast<const u32x4*>(src + (int64_t)(s0 + i) * sn);
        }
    }
    double acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    float mn[8], mx[8], xprev[8];
#pragma unroll
    for (int e = 0; e < 8; e++) { mn[e] = INFINITY; mx[e] = -INFINITY; xprev[e] = 0.0f; }
    float inv[kLeaf], gain[8];
    constexpr int AHEAD = PRE == 2 ? 2 : 4;
    RopeTab<PRE> tab[AHEAD];
    auto clamped = [&](int i) { return min(s0 + i, N - 1); };
    RopeAt rope{};
    if constexpr (PRE) {
        rope = rope_at<D>(pre, b, h, H, col);
#pragma unroll
        for (int i = 0; i < AHEAD; i++) rope_load<PRE>(rope, clamped(i), tab[i]);
        pre_gains(pre, h, D, col, gain);
        if (pre.row_inv == nullptr) {
            row_inverses<D, kLeaf>(pre.eps, w, inv);
        } else {
#pragma unroll
            for (int i = 0; i < kLeaf; i++) inv[i] = pre.row_inv[(int64_t)b * pre.row_n + clamped(i)];
        }
    }
    static_assert(kLeaf % 2 == 0, "tokens are taken in pairs");
    auto token = [&](int i, bool odd, const u32x4& raw) {
        float x[8];
        unpack8(raw, x);
        const bool kept = key_kept(s0 + i, N, km);
        if constexpr (PRE) {
            pre_apply<D, PRE>(pre, col, kept, inv[i], gain, tab[i % AHEAD], x);
            if (i + AHEAD < kLeaf) rope_load<PRE>(rope, clamped(i + AHEAD), tab[i % AHEAD]);
        }
        // tokens that do not count are +0.0 here, which leaves a double sum unchanged
#pragma unroll
        for (int e = 0; e < 8; e++) acc[e] += (double)x[e];
        if (all_kept) {
            // (the common case, two tokens per three-operand instruction; written as instructions because the
            // compiler puts a canonicalising v_max in front of every operand of fminf / fmaxf that comes out of
            // bit operations — six instructions per element instead of one)
            if (odd) {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    asm("v_min3_f32 %0, %0, %1, %2" : "+v"(mn[e]) : "v"(xprev[e]), "v"(x[e]));
                    asm("v_max3_f32 %0, %0, %1, %2" : "+v"(mx[e]) : "v"(xprev[e]), "v"(x[e]));
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) xprev[e] = x[e];
            }
        } else if (kept) {
#pragma unroll
            for (int e = 0; e < 8; e++) { mn[e] = fminf(mn[e], x[e]); mx[e] = fmaxf(mx[e], x[e]); }
        }
    };
    if constexpr (IN_LDS) {
#pragma unroll 1
        for (int i0 = 0; i0 < kLeaf; i0 += 4) {                // (registers for four rows, not sixteen)
            u32x4 raw[4];
#pragma unroll
            for (int i = 0; i < 4; i++) raw[i] = rows[(leaf * kLeaf + i0 + i) * CPR + tid % CPR];
#pragma unroll
            for (int i = 0; i < 4; i++) token(i0 + i, i & 1, raw[i]);
        }
    } else {
#pragma unroll
        for (int i = 0; i < kLeaf; i++) token(i, i & 1, w[i]);
    }
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const int at = e * CPR + (col >> 3);
        sm.leafsum[leaf][at] = acc[e];
        sm.leafmin[leaf][at] = mn[e];
        sm.leafmax[leaf][at] = mx[e];
    }
    }
    __syncthreads();
    gsum = 0.0;
    gmn = INFINITY; gmx = -INFINITY;
    if (tid < D && g >= 0) {
#pragma unroll
        for (int u = 0; u < 16; u++) {
            gsum += sm.leafsum[u][tid];
            gmn = fminf(gmn, sm.leafmin[u][tid]);
            gmx = fmaxf(gmx, sm.leafmax[u][tid]);
        }
    }
}

template <int D, int PRE, int DFULL = D, bool IN_LDS = false>
__device__ __forceinline__ void kstats_group_body(
    int g, int h, int b, int tid, const uint16_t* __restrict__ k, int64_t sb, int64_t sh, int64_t sn,
    int N, int H, int ngroups, const KeyMask& km, double* __restrict__ part_sum, float* __restrict__ part_mm,
    KGroupSmem<D>& sm, const PreOp& pre, int col0 = 0, const u32x4* rows = nullptr) {
    double gsum;
    float gmn, gmx;
    kstats_group<D, PRE, DFULL, IN_LDS>(g, h, b, tid, k, sb, sh, sn, N, H, km, sm, pre, col0, gsum, gmn, gmx, rows);
    if (tid < D && g >= 0) {
        const int64_t o = (((int64_t)b * H + h) * ngroups + g) * DFULL + col0 + leaf_channel<D>(tid);
        part_sum[o] = gsum;
        part_mm[2 * o] = gmn;
        part_mm[2 * o + 1] = gmx;
    }
}

// ---------------------------------------------------------------------------
// V repack: bf16 [.., N, D] -> fp16 tiles [.., N/64, D, 64]; key k of a tile goes to slot
// v_slot_f16(k).  One workgroup per (tile, h, b): rows are read coalesced, staged in LDS and
// written back channel-major in 16-byte runs.  Rows that are masked or beyond N become 0.
// ---------------------------------------------------------------------------
// LDS tile: 64 slots x D halves, unpadded; the 16-byte chunk index of a row is XORed with
// 2*(slot/8) so that both the row-wise 16-byte writes and the column-wise dword reads below
// touch every bank once (D = 128: 16 chunks; D = 64: 8 chunks, XOR with slot/8 instead).
template <int D>
__device__ __forceinline__ int v_tile_chunk(int slot, int chunk) {
    // (D = 256: 32 chunks, XOR with 4*(slot/8))
    return D == 256 ? (chunk ^ (((slot >> 3) & 7) << 2)) : D == 128 ? (chunk ^ (((slot >> 3) & 7) << 1)) : (chunk ^ ((slot >> 3) & 7));
}

// A tile in LDS -> memory, channel-major.
template <int D, int NT>
__device__ __forceinline__ void store_v_f16_tile(int tid, const uint16_t* tile, uint16_t* dst) {
    // work item = (channel pair, 8 consecutive slots): eight dword reads, two 16-byte stores
    const uint32_t* tile32 = reinterpret_cast<const uint32_t*>(tile);
#pragma unroll
    for (int i = 0; i < (D / 2) * 8 / NT; i++) {
        const int c = i * NT + tid;
        const int dp = c >> 3, s0 = (c & 7) * 8;            // channels 2*dp, 2*dp+1
        uint32_t w[8];
#pragma unroll
        for (int e = 0; e < 8; e++)
            w[e] = tile32[(s0 + e) * (D / 2) + v_tile_chunk<D>(s0 + e, dp >> 2) * 4 + (dp & 3)];
        u32x4 lo, hi;
        lo.x = __builtin_amdgcn_perm(w[1], w[0], 0x05040100u); hi.x = __builtin_amdgcn_perm(w[1], w[0], 0x07060302u);
        lo.y = __builtin_amdgcn_perm(w[3], w[2], 0x05040100u); hi.y = __builtin_amdgcn_perm(w[3], w[2], 0x07060302u);
        lo.z = __builtin_amdgcn_perm(w[5], w[4], 0x05040100u); hi.z = __builtin_amdgcn_perm(w[5], w[4], 0x07060302u);
        lo.w = __builtin_amdgcn_perm(w[7], w[6], 0x05040100u); hi.w = __builtin_amdgcn_perm(w[7], w[6], 0x07060302u);
        *reinterpret_cast<u32x4*>(dst + (2 * dp) * 64 + s0) = lo;
        *reinterpret_cast<u32x4*>(dst + (2 * dp + 1) * 64 + s0) = hi;
    }
}

template <int D, int NT = 256>
__device__ __forceinline__ void quant_v_f16_body(
    int t, int h, int b, int tid, const uint16_t* __restrict__ v, int64_t sb, int64_t sh, int64_t sn,
    int N, int H, int64_t n_pad, const KeyMask& km, uint16_t* __restrict__ out, uint16_t* tile) {
    constexpr int CPR = D / 8;
    const uint16_t* src = v + b * sb + h * sh;
    u32x4 raw[64 * CPR / NT];
#pragma unroll
    for (int i = 0; i < 64 * CPR / NT; i++) {
        const int c = i * NT + tid;
        const int key = c / CPR, col = (c % CPR) * 8;
        const int row = t * 64 + key;
        raw[i] = u32x4{0u, 0u, 0u, 0u};
        if (key_kept(row, N, km)) raw[i] = *reinterpret_cast<const u32x4*>(src + (int64_t)row * sn + col);
    }
#pragma unroll
    for (int i = 0; i < 64 * CPR / NT; i++) {
        const int c = i * NT + tid;
        const int key = c / CPR, chunk = c % CPR;
        float x[8];
        unpack8(raw[i], x);
        u32x4 o;
        o.x = f16_pair_sat(x[0], x[1]);
        o.y = f16_pair_sat(x[2], x[3]);
        o.z = f16_pair_sat(x[4], x[5]);
        o.w = f16_pair_sat(x[6], x[7]);
        const int slot = v_slot_f16(key);
        *reinterpret_cast<u32x4*>(&tile[slot * D + v_tile_chunk<D>(slot, chunk) * 8]) = o;
    }
    __syncthreads();
    store_v_f16_tile<D, NT>(tid, tile, out + ((((int64_t)b * H + h) * (n_pad / 64)) + t) * (int64_t)(D * 64));
}

// ---------------------------------------------------------------------------
// V channel maxima of one group of 256 tokens (e4m3 variant; max is order-free).
// ---------------------------------------------------------------------------
template <int D, int NT = 256>
__device__ __forceinline__ void v_absmax_group_body(
    int g, int h, int b, const uint16_t* __restrict__ v, int64_t sb, int64_t sh, int64_t sn,
    int N, int H, int ngroups, const KeyMask& km, float* __restrict__ part, float (*red)[D + D / 8]) {
    constexpr int CPR = D / 8;
    constexpr int ROWS = NT / CPR;                        // rows covered per step
    const int tid = threadIdx.x;
    const int col = (tid % CPR) * 8, r = tid / CPR;
    const uint16_t* src = v + b * sb + h * sh + col;
    float m[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll 4
    for (int i = 0; i < kGroup / ROWS; i++) {
        const int row = g * kGroup + i * ROWS + r;
        if (key_kept(row, N, km)) {
            u32x4 w = *reinterpret_cast<const u32x4*>(src + (int64_t)row * sn);
            float x[8];
            unpack8(w, x);
#pragma unroll
            for (int e = 0; e < 8; e++) m[e] = fmaxf(m[e], fabsf(x[e]));
        }
    }
#pragma unroll
    for (int e = 0; e < 8; e++) red[r][e * CPR + (col >> 3)] = m[e];        // (as in KGroupSmem)
    __syncthreads();
    if (tid < D) {
        float mm = 0.0f;
#pragma unroll
        for (int i = 0; i < ROWS; i++) mm = fmaxf(mm, red[i][tid]);
        part[(((int64_t)b * H + h) * ngroups + g) * D + leaf_channel<D>(tid)] = mm;
    }
}

// V tile -> e4m3 with the per-channel scales, tiled layout (slot order v_slot_fp8).
//
// The code of an element is e4m3(RN(x / sc)).  The common case takes neither a divide nor the
// conversion in integer arithmetic: with y = RN(1 / sc) (one true divide per channel and thread),
// q0 = RN(x y), r = x - q0 sc (exact in one fused step) and q1 = RN(q0 + r y), q1 IS the correctly
// rounded quotient (Markstein's correction step; it needs y correctly rounded, q0 within an ulp
// and the significand of sc not all ones), and the conversion instruction rounds to nearest even
// and reaches 448 exactly where the quotient's magnitude is 448 (1 + 2^-23) at most, which the
// scale guarantees.  A wave that sees a non-finite input, or a scale outside the range where none
// of this can underflow, or with an all-ones significand, takes the plain formula.
struct VScale8 {
    float sc[8], y[8];
    bool odd;                                              // a scale that the short way does not take
    __device__ __forceinline__ explicit VScale8(const float* vscale) {
        load8(vscale, sc);
        odd = false;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            y[e] = 1.0f / sc[e];
            odd = odd || !(sc[e] >= 0x1p-60f && sc[e] <= 0x1p60f) || (__float_as_uint(sc[e]) & 0x7FFFFFu) == 0x7FFFFFu;
        }
    }
    // whether some lane of the wave needs the plain formula for these chunks
    template <int N> __device__ __forceinline__ bool plain_for(const u32x4 (&w)[N]) const {
        uint32_t mag = 0u;
#pragma unroll
        for (int i = 0; i < N; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) mag = bf16_mag_max(mag, w[i][e]);
        return __any(odd || !bf16_mag_finite(mag));
    }
    __device__ __forceinline__ void codes(const u32x4& w, bool plain, uint32_t (&pk)[2]) const {
        float x[8];
        unpack8(w, x);
        pk[0] = pk[1] = 0u;
        if (__builtin_expect(plain, 0)) {
#pragma unroll
            for (int e = 0; e < 8; e++) pk[e >> 2] |= f32_to_e4m3(x[e] / sc[e]) << ((e & 3) * 8);
        } else {
            float q[8];
#pragma unroll
            for (int e = 0; e < 8; e++) {
                // (the residual as -(q0 sc - x): an input of -0 then stays -0 through both steps, as it
                // does through the divide)
                const float q0 = x[e] * y[e];
                q[e] = fmaf(-fmaf(q0, sc[e], -x[e]), y[e], q0);
            }
#pragma unroll
            for (int j = 0; j < 2; j++) {
                int p2 = __builtin_amdgcn_cvt_pk_fp8_f32(q[4 * j], q[4 * j + 1], 0, false);
                p2 = __builtin_amdgcn_cvt_pk_fp8_f32(q[4 * j + 2], q[4 * j + 3], p2, true);
                pk[j] = (uint32_t)p2;
            }
        }
    }
};
// Codes of a tile in LDS (row = slot, LD bytes) -> the tile in memory: 16 consecutive slots of a channel at a time.
template <int D, int NT>
__device__ __forceinline__ void store_v_fp8_tile(int tid, const uint8_t* tile, uint8_t* dst) {
    constexpr int LD = D + 16;
#pragma unroll
    for (int i = 0; i < D * 4 / NT; i++) {
        const int c = i * NT + tid;
        const int d = c >> 2, s0 = (c & 3) * 16;
        uint32_t pk[4] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int e = 0; e < 16; e++) pk[e >> 2] |= (uint32_t)tile[(s0 + e) * LD + d] << ((e & 3) * 8);
        *reinterpret_cast<u32x4*>(dst + d * 64 + s0) = u32x4{pk[0], pk[1], pk[2], pk[3]};
    }
}

template <int D, int NT>
__device__ __forceinline__ void quant_v_fp8_body(
    int t, int h, int b, int tid, const uint16_t* __restrict__ v, int64_t sb, int64_t sh, int64_t sn,
    int N, int H, int64_t n_pad, const KeyMask& km, const float* __restrict__ vscale,
    uint8_t* __restrict__ out, uint8_t* tile) {
    constexpr int CPR = D / 8;
    constexpr int LD = D + 16;                             // padded row (bytes)
    constexpr int NCH = 64 * CPR / NT;
    static_assert(NT % CPR == 0, "a thread keeps one column group for all its chunks");
    const int64_t bh = (int64_t)b * H + h;
    const uint16_t* src = v + b * sb + h * sh;
    const int col = (tid % CPR) * 8;
    u32x4 w[NCH];
#pragma unroll
    for (int i = 0; i < NCH; i++) {
        const int row = t * 64 + (i * NT + tid) / CPR;
        w[i] = u32x4{0u, 0u, 0u, 0u};
        if (key_kept(row, N, km)) w[i] = *reinterpret_cast<const u32x4*>(src + (int64_t)row * sn + col);
    }
    const VScale8 vs(vscale + col);
    const bool plain = vs.plain_for(w);
#pragma unroll
    for (int i = 0; i < NCH; i++) {
        const int key = (i * NT + tid) / CPR;
        uint32_t pk[2];
        vs.codes(w[i], plain, pk);
        *reinterpret_cast<u32x2*>(&tile[v_slot_fp8(key) * LD + col]) = u32x2{pk[0], pk[1]};
    }
    __syncthreads();
    uint8_t* dst = out + ((bh * (n_pad / 64)) + t) * (int64_t)(D * 64);
    store_v_fp8_tile<D, NT>(tid, tile, dst);
}

// ---------------------------------------------------------------------------
// Launch 1: independent passes over V and K as workgroup roles of one grid (one launch fills
// the chip where each pass alone is too short to).
// ---------------------------------------------------------------------------
template <int D, int PRE>
__global__ __launch_bounds__(256) void prep_kernel(PrepArgs a) {
    constexpr int DK = D > 128 ? 128 : D;                 // channels per K statistics call
    constexpr int GPW = 256 / (16 * (DK / 8));            // K groups per workgroup (D = 256: one group, one half of the channels)
    union Smem {
        uint16_t tile[64 * D];
        float red[256 / (D / 8)][D + D / 8];
        KGroupSmem<DK> kg[GPW];
    };
    __shared__ __attribute__((aligned(16))) Smem sm;
    // Consecutive workgroups take the same unit of consecutive heads: in [.., N, H, D] memory those
    // are neighbours, so the workgroups in flight together read whole DRAM pages between them.  The
    // K-statistics units (longer) are dealt evenly among the V units instead of coming last.
    const int per_bh = a.nv_units + a.nk_wg;
    const int bh = blockIdx.x % a.n_bh, slot = blockIdx.x / a.n_bh;
    const int k_before = (int)(((int64_t)slot * a.nk_wg) / per_bh);
    const bool is_k = (int)(((int64_t)(slot + 1) * a.nk_wg) / per_bh) > k_before;
    const int r = is_k ? a.nv_units + k_before : slot - k_before;
    const int b = bh / a.H, h = bh % a.H;
    if (r < a.nv_units) {
        if (a.vmode == 0)
            quant_v_f16_body<D>(r, h, b, threadIdx.x, a.v.p, a.v.sb, a.v.sh, a.v.sn, a.Nkv, a.H, a.nkv_pad, a.km, a.v16, sm.tile);
        else
            v_absmax_group_body<D>(r, h, b, a.v.p, a.v.sb, a.v.sh, a.v.sn, a.Nkv, a.H, a.ngroups, a.km, a.vpart, sm.red);
    } else if constexpr (D > 128) {
        const int u = r - a.nv_units;                     // (group, channel half)
        kstats_group_body<DK, 0, D>(u >> 1, h, b, threadIdx.x, a.k.p, a.k.sb, a.k.sh, a.k.sn, a.Nkv, a.H, a.ngroups,
                                        a.km, a.kpart_sum, a.kpart_mm, sm.kg[0], a.pre_k, (u & 1) * DK);
    } else {
        const int sub = threadIdx.x / (16 * (D / 8));
        const int g = (r - a.nv_units) * GPW + sub;
        // groups past the end still take part in the barrier inside; they read nothing and
        // store nothing
        kstats_group_body<D, PRE>(g < a.ngroups ? g : -1, h, b, threadIdx.x % (16 * (D / 8)), a.k.p, a.k.sb, a.k.sh,
                                  a.k.sn, a.Nkv, a.H, a.ngroups, a.km, a.kpart_sum, a.kpart_mm, sm.kg[sub], a.pre_k);
    }
}

// The K statistics behind the pre-ops, and with e4m3 the V channel maxima, where there are no more K groups than compute units.  A wave per SIMD norms and rotates
// sixteen rows one after the other there, and that chain is the launch.  Here a group's 256 rows go to four times as many
// threads, four rows each, and through LDS to those that add them up, in the same order.  The call, us: [1,8 heads,768,64] 25.1 ->
// 21.4, [2,12,2000,64] 53.8 -> 49.1, [1,19,1153,128] 47.2 -> 44.0, [2,16,2048,128] (256 groups) 92.8 -> 89.8; but past one
// workgroup per unit [1,30,2304,128] (270) 121.9 -> 125.0, [1,24,4608,128] 240 -> 245.  e4m3 [1,8,1000,64] 25.8 -> 22.4, [1,24,2304,64]
// 67.6 -> 60.3, [1,19,1153,128] 47.7 -> 44.9; but [1,32,2000,128] (256 and as many of V) 93.1 -> 94.1.
template <int D, int PRE>
__global__ __launch_bounds__(64 * (D / 8)) void prep_rows_kernel(PrepArgs a) {
    constexpr int CPR = D / 8, NR = 4, PASS = kGroup / NR, AHEAD = PRE == 2 ? 2 : NR;
    union Smem {
        float red[64][D + D / 8];
        KGroupSmem<D> kg;
    };
    __shared__ __attribute__((aligned(16))) Smem sm;
    __shared__ __attribute__((aligned(16))) u32x4 rows[kGroup * CPR];
    const int bh = blockIdx.x % a.n_bh, g = blockIdx.x / a.n_bh;
    const int b = bh / a.H, h = bh % a.H;
    if (g >= a.ngroups) {                                  // (behind the K groups, which are the longer ones)
        v_absmax_group_body<D, 64 * CPR>(g - a.ngroups, h, b, a.v.p, a.v.sb, a.v.sh, a.v.sn, a.Nkv, a.H, a.ngroups, a.km, a.vpart, sm.red);
        return;
    }
    const int tid = threadIdx.x, col = (tid % CPR) * 8, first = g * kGroup + tid / CPR;
    const uint16_t* src = a.k.p + b * a.k.sb + h * a.k.sh + col;
    u32x4 w[NR];
    RopeTab<PRE> tab[AHEAD];
    const RopeAt rope = rope_at<D>(a.pre_k, b, h, a.H, col);
    auto clamped = [&](int i) { return min(first + i * PASS, a.Nkv - 1); };
#pragma unroll
    for (int i = 0; i < NR; i++) {
        w[i] = u32x4{0u, 0u, 0u, 0u};
        if (key_kept(first + i * PASS, a.Nkv, a.km)) w[i] = *reinterpret_cast<const u32x4*>(src + (int64_t)(first + i * PASS) * a.k.sn);
    }
#pragma unroll
    for (int i = 0; i < AHEAD; i++) rope_load<PRE>(rope, clamped(i), tab[i]);
    float inv[NR], gain[8];
    pre_gains(a.pre_k, h, D, col, gain);
    if (a.pre_k.row_inv == nullptr) {
        row_inverses<D, NR>(a.pre_k.eps, w, inv);
    } else {
#pragma unroll
        for (int i = 0; i < NR; i++) inv[i] = a.pre_k.row_inv[(int64_t)b * a.pre_k.row_n + clamped(i)];
    }
#pragma unroll
    for (int i = 0; i < NR; i++) {
        float x[8];
        unpack8(w[i], x);
        pre_apply<D, PRE>(a.pre_k, col, key_kept(first + i * PASS, a.Nkv, a.km), inv[i], gain, tab[i % AHEAD], x);
        if (i + AHEAD < NR) rope_load<PRE>(rope, clamped(i + AHEAD), tab[i % AHEAD]);
        u32x4 y;                                           // (bf16 values: nothing below their upper halves)
#pragma unroll
        for (int e = 0; e < 4; e++) y[e] = __builtin_amdgcn_perm(__float_as_uint(x[2 * e + 1]), __float_as_uint(x[2 * e]), 0x07060302u);
        rows[(i * PASS + tid / CPR) * CPR + tid % CPR] = y;
    }
    __syncthreads();
    // (16 leaves; the other waves only meet the barrier inside)
    kstats_group_body<D, 0, D, true>(tid < 16 * CPR ? g : -1, h, b, tid, a.k.p, a.k.sb, a.k.sh, a.k.sn, a.Nkv, a.H, a.ngroups, a.km, a.kpart_sum,
                                     a.kpart_mm, sm.kg, a.pre_k, 0, rows);
}

// ---------------------------------------------------------------------------
// Launch 0: whole-row RMSNorm statistic.  One workgroup of 256 threads per token, exactly the
// reference's reduction (serenitymojo/ops/norm.mojo:56-72): thread t adds the squares of
// channels t, t+256, ... in turn (multiply and add rounded separately), then the 256 partial
// sums fold in halves through LDS, far pairs first.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void row_inv_kernel(View q, View k, int H, int Nq, int Nkv, int D, int rows_q, float eps,
                                                      float* __restrict__ inv_q, float* __restrict__ inv_k) {
    __shared__ float part[256];
    const int tid = threadIdx.x;
    int r = blockIdx.x;
    const bool is_k = r >= rows_q;
    if (is_k) r -= rows_q;
    const View& x = is_k ? k : q;
    const int N = is_k ? Nkv : Nq;
    const int b = r / N, n = r % N;
    const uint16_t* row = x.p + b * x.sb + (int64_t)n * x.sn;
    const int cols = H * D;
    float local = 0.0f;
    for (int c = tid; c < cols; c += 256) {
        const float v = __uint_as_float((uint32_t)row[(int64_t)(c / D) * x.sh + (c % D)] << 16);
        const float sq = v * v;
        local = local + sq;
    }
    part[tid] = local;
    __syncthreads();
    for (int active = 128; active > 0; active >>= 1) {
        if (tid < active) part[tid] = part[tid] + part[tid + active];
        __syncthreads();
    }
    if (tid == 0) {
        const float mean = part[0] / (float)cols;
        (is_k ? inv_k : inv_q)[r] = 1.0f / sqrtf(mean + eps);
    }
}

hipError_t launch_row_inv(const View& q, const View& k, int B, int H, int Nq, int Nkv, int D, float eps,
                          float* inv_q, float* inv_k, hipStream_t st) {
    const int64_t rows_q = (int64_t)B * Nq, rows = rows_q + (int64_t)B * Nkv;
    if (rows > 0x7FFFFFFF) return hipErrorInvalidValue;
    hipLaunchKernelGGL(row_inv_kernel, dim3((unsigned)rows), dim3(256), 0, st, q, k, H, Nq, Nkv, D, (int)rows_q, eps, inv_q, inv_k);
    return hipGetLastError();
}

// Which instantiation the pre-ops take (see RopeTab).
static int pre_kind(const PreOp& p) { return p.gain == nullptr ? 0 : p.cos != nullptr && p.halfsplit && !p.tables_bf16 ? 2 : 1; }

hipError_t launch_prep(const PrepArgs& a_in, int B, int D, hipStream_t st) {
    PrepArgs a = a_in;
    a.ngroups = (a.Nkv + kGroup - 1) / kGroup;
    // K groups per workgroup: 2 at D = 64, 1 at D = 128; at D = 256 a group takes two workgroups
    a.nk_wg = a.kpart_sum == nullptr ? 0 : D == 256 ? a.ngroups * 2 : D == 128 ? a.ngroups : (a.ngroups + 1) / 2;
    a.nv_units = a.vmode == 0 ? (int)(a.nkv_pad / 64) : (a.vmode == 1 ? a.ngroups : 0);
    a.n_bh = B * a.H;
    const int has_pre = pre_kind(a.pre_k);
    const int64_t total = (int64_t)B * a.H * (a.nv_units + a.nk_wg);
    if (total == 0) return hipSuccess;
    if (total > 0x7FFFFFFF) return hipErrorInvalidValue;
    dim3 grid((unsigned)total), block(256);
    // (more groups than compute units: prep_kernel's smaller workgroups fill the chip by themselves.  A workgroup of 128 channels
    // has a unit to itself, and its V blocks count; of 64 two share one)
    const int64_t groups = (int64_t)B * a.H * a.ngroups, blocks = groups + (int64_t)B * a.H * a.nv_units;
    if (D <= 128 && has_pre && a.kpart_sum != nullptr && a.vmode != 0 && (D == 64 ? groups : blocks) <= compute_units()) {
        const dim3 each((unsigned)blocks), threads(8 * D);
        if (D == 128 && has_pre == 2) hipLaunchKernelGGL((prep_rows_kernel<128, 2>), each, threads, 0, st, a);
        else if (D == 128) hipLaunchKernelGGL((prep_rows_kernel<128, 1>), each, threads, 0, st, a);
        else if (has_pre == 2) hipLaunchKernelGGL((prep_rows_kernel<64, 2>), each, threads, 0, st, a);
        else hipLaunchKernelGGL((prep_rows_kernel<64, 1>), each, threads, 0, st, a);
        return hipGetLastError();
    }
    if (D == 128 && has_pre == 2) hipLaunchKernelGGL((prep_kernel<128, 2>), grid, block, 0, st, a);
    else if (D == 128 && has_pre) hipLaunchKernelGGL((prep_kernel<128, 1>), grid, block, 0, st, a);
    else if (D == 128) hipLaunchKernelGGL((prep_kernel<128, 0>), grid, block, 0, st, a);
    else if (D == 64 && has_pre == 2) hipLaunchKernelGGL((prep_kernel<64, 2>), grid, block, 0, st, a);
    else if (D == 64 && has_pre) hipLaunchKernelGGL((prep_kernel<64, 1>), grid, block, 0, st, a);
    else if (D == 64) hipLaunchKernelGGL((prep_kernel<64, 0>), grid, block, 0, st, a);
    else if (D == 256 && !has_pre) hipLaunchKernelGGL((prep_kernel<256, 0>), grid, block, 0, st, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Launch 2: one thread per (b, h, channel).
//   K: sum of the group sums in group order -> mean = fp32(sum / kept) (0 without smoothing);
//      amax = max(|kmax - mean|, |kmin - mean|) — rounding is monotone, so this IS the largest
//      |k - mean| over the kept keys; s = sqrt(amax) (1 when amax is 0 or without balancing);
//      kmul = 1/s, qmul = cmul*s.
//   V: vscale = amax/448 (1 when 0).
// ---------------------------------------------------------------------------
// Groups added up, strictly in group order; the loads go NB groups at a time (taken one by one, each waits
// out a memory latency).
template <int NB>
__device__ __forceinline__ void k_totals(const FinalArgs& a, int64_t bh, int d, float& mean, float& s) {
    mean = 0.0f;
    s = 1.0f;
    if (a.kpart_sum == nullptr) return;
    const double* p = a.kpart_sum + bh * a.ngroups * a.D + d;
    const float* q = a.kpart_mm + 2 * (bh * a.ngroups * a.D + d);
    double sum = 0.0;
    float mn = INFINITY, mx = -INFINITY;
    for (int g0 = 0; g0 < a.ngroups; g0 += NB) {
        double v[NB];
        float lo[NB], hi[NB];
#pragma unroll
        for (int j = 0; j < NB; j++) {
            const int64_t g = g0 + j < a.ngroups ? g0 + j : a.ngroups - 1;
            v[j] = p[g * a.D];
            lo[j] = q[2 * g * a.D];
            hi[j] = q[2 * g * a.D + 1];
        }
#pragma unroll
        for (int j = 0; j < NB; j++)
            if (g0 + j < a.ngroups) { sum += v[j]; mn = fminf(mn, lo[j]); mx = fmaxf(mx, hi[j]); }
    }
    k_final(sum, mn, mx, a.kept, a.flags, mean, s);
}
template <int NB>
__device__ __forceinline__ float v_total(const FinalArgs& a, int64_t bh, int d) {
    const float* p = a.vpart + bh * a.ngroups * a.D + d;
    float amax = 0.0f;
    for (int g0 = 0; g0 < a.ngroups; g0 += NB) {
        float v[NB];
#pragma unroll
        for (int j = 0; j < NB; j++) v[j] = p[(int64_t)(g0 + j < a.ngroups ? g0 + j : a.ngroups - 1) * a.D];
#pragma unroll
        for (int j = 0; j < NB; j++) amax = fmaxf(amax, v[j]);
    }
    return amax > 0.0f ? amax / 448.0f : 1.0f;
}

__global__ __launch_bounds__(64) void stats_final_kernel(FinalArgs a) {
    const int64_t i = (int64_t)blockIdx.x * 64 + threadIdx.x;      // (bh, d)
    if (i >= a.total) return;
    const int64_t bh = i / a.D;
    const int d = (int)(i % a.D);
    if (a.kmean != nullptr) {
        float mean, s;
        k_totals<32>(a, bh, d, mean, s);
        a.kmean[i] = mean;
        a.kmul[i] = 1.0f / s;
        a.qmul[i] = a.cmul * s;
    }
    if (a.vscale != nullptr) a.vscale[i] = v_total<32>(a, bh, d);
}

hipError_t launch_stats_final(const FinalArgs& a, hipStream_t st) {
    if (a.total <= 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(stats_final_kernel, dim3((unsigned)((a.total + 63) / 64)), dim3(64), 0, st, a);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Launch 3: Q blocks, K blocks and (e4m3 variant) V tiles as workgroup roles.
// ---------------------------------------------------------------------------
// Threads per workgroup.  At 256 channels a Q block of 128 rows is 128 elements to each of 256 threads, twice what it is at
// 128, and its chain is what the launch lasts; with 512 the call takes, us, [1,1153,18,256] 52.2 -> 49.3, e4m3 69.0 -> 65.8,
// [1,4608,18,256] 346 -> 337, [2,300,30,256] 39.5 -> 36.7.  (512 at 128 channels, i.e. fewer registers and more waves per
// SIMD, measured slower; so did rows requested ahead of FIN's sums, whose registers halve the waves: [1,1153,24,128] 36.1 -> 41.6.)
template <int D, int PRE> constexpr int quant_threads() { return D > 128 ? 512 : 256; }

// FIN: launch 2 is left out — every workgroup adds up the group results it needs for itself (the same additions,
// so the same bits), the first of a head's K and V workgroups also leave them for later launches.
// SETS: Q and K blocks are dealt by set_member (sage_grid.h; where: launch_quant).
template <int D, int PRE, bool FIN, bool SETS>
__global__ __launch_bounds__((quant_threads<D, PRE>())) void quant_kernel(QuantArgs a, FinalArgs f) {
    constexpr int NT = quant_threads<D, PRE>();
    union Smem {
        float red[NT / 64];
        uint8_t tile8[64 * (D + 16)];
        uint16_t tile16[64 * D];
    };
    __shared__ __attribute__((aligned(16))) Smem sm;
    // consecutive workgroups take the same rows of consecutive heads: in [.., N, H, D] memory those
    // are neighbours, so the workgroups in flight together read whole DRAM pages between them
    int bh = blockIdx.x % a.n_bh, r = blockIdx.x / a.n_bh;
    if constexpr (SETS) {
        const int id = blockIdx.x;
        if (id < a.n_sets) {
            const SetMember m = set_member(id, a.members);
            const int heads = a.n_bh / a.batches, run = m.set / heads, which = m.member / a.batches;
            const bool is_k = which >= a.q_per;
            const int t = is_k ? run * a.k_per + which - a.q_per : run * a.q_per + which;
            if (t >= (is_k ? a.nk_blk : a.nq_blk)) return;           // (also the sets past the last one)
            bh = m.member % a.batches * heads + m.set % heads;
            r = is_k ? a.nq_blk + t : t;
        } else {
            bh = (id - a.n_sets) % a.n_bh;
            r = a.nq_blk + a.nk_blk + (id - a.n_sets) / a.n_bh;
        }
    }
    const int b = bh / a.H, h = bh % a.H;
    const KeyMask none{0, 0};
    __shared__ __attribute__((aligned(16))) float s_fin[FIN ? 3 : 1][FIN ? D : 4];      // mean, kmul, qmul; or vscale
    if constexpr (FIN) {
        const bool is_v = r >= a.nq_blk + a.nk_blk;
        if (threadIdx.x < D && !(is_v && a.v16 != nullptr)) {
            const int d = threadIdx.x;
            const int64_t i = (int64_t)bh * D + d;
            if (is_v) {
                const float sc = v_total<8>(f, bh, d);
                s_fin[0][d] = sc;
                if (r == a.nq_blk + a.nk_blk) f.vscale[i] = sc;
            } else {
                float mean, s;
                k_totals<8>(f, bh, d, mean, s);
                const float kmul = 1.0f / s, qmul = f.cmul * s;
                s_fin[0][d] = mean; s_fin[1][d] = kmul; s_fin[2][d] = qmul;
                if (r == a.nq_blk) { f.kmean[i] = mean; f.kmul[i] = kmul; f.qmul[i] = qmul; }
            }
        }
        __syncthreads();
    }
    if (r < a.nq_blk) {
        const float* mul = FIN ? s_fin[FIN ? 2 : 0] : a.qmul + (int64_t)bh * D;
        const float* mean = FIN ? s_fin[0] : a.kmean + (int64_t)bh * D;
#define SAGE_Q(BLK) quant_i8_block<D, BLK, false, PRE, NT>(r, h, b, threadIdx.x, a.q.p, a.q.sb, a.q.sh, a.q.sn, a.Nq, a.H, a.nq_pad, none, \
                                                       mean, mul, a.cmul, a.q8, a.qscale, a.rowdot, sm.red, a.pre_q)
        if (a.blkq == 128) SAGE_Q(128);
        else if (a.blkq == 64) SAGE_Q(64);
        else SAGE_Q(32);
#undef SAGE_Q
    } else if (r < a.nq_blk + a.nk_blk) {
        const int t = r - a.nq_blk;
        const float* mul = FIN ? s_fin[FIN ? 1 : 0] : a.kmul + (int64_t)bh * D;
        const float* mean = FIN ? s_fin[0] : a.kmean + (int64_t)bh * D;
#define SAGE_K(BLK) quant_i8_block<D, BLK, true, PRE, NT>(t, h, b, threadIdx.x, a.k.p, a.k.sb, a.k.sh, a.k.sn, a.Nkv, a.H, a.nkv_pad, a.km, \
                                                      mean, mul, 0.0f, a.k8, a.kscale, nullptr, sm.red, a.pre_k)
        if (a.blkk == 128) SAGE_K(128);
        else if (a.blkk == 64) SAGE_K(64);
        else SAGE_K(32);
#undef SAGE_K
    } else if (a.v16 != nullptr) {
        quant_v_f16_body<D, NT>(r - a.nq_blk - a.nk_blk, h, b, threadIdx.x, a.v.p, a.v.sb, a.v.sh, a.v.sn, a.Nkv, a.H, a.nkv_pad, a.km, a.v16, sm.tile16);
    } else {
        quant_v_fp8_body<D, NT>(r - a.nq_blk - a.nk_blk, h, b, threadIdx.x, a.v.p, a.v.sb, a.v.sh, a.v.sn, a.Nkv, a.H, a.nkv_pad, a.km,
                            FIN ? s_fin[0] : a.vscale + (int64_t)bh * D, a.v8, sm.tile8);
    }
}

// Where launch 2 is left out.  It costs 3 us, the start and end of a kernel that does next to nothing; adding up
// costs every workgroup the group results of its head from L2, 16 bytes per group and channel next to the 128 (Q:
// 256) bytes per channel it encodes.  Stage of K and V, us, three launches -> two: [1,1153,24,128] 15.7 -> 12.7,
// [2,1248,30,128] 24.5 -> 22.5, [1,2304,24,128] (9 groups) 19.8 -> 17.1, [1,3000,24,128] (12) 24.0 -> 22.9,
// [1,4608,24,128] (18) 28.4 -> 30.2, [1,1153,18,256] 20.4 -> 16.9.  e4m3, with 32-row Q blocks: [1,1800,24,128] (8)
// 24.9 -> 23.2, [1,2304,24,128] (9) 27.1 -> 28.1.
bool quant_adds_up(const QuantArgs& a) {
    const int groups = (a.Nkv + kGroup - 1) / kGroup;
    return a.k8 != nullptr && groups <= (a.v8 != nullptr ? 8 : 10);
}

hipError_t launch_quant(const QuantArgs& a_in, const FinalArgs* f, int B, int D, hipStream_t st) {
    QuantArgs a = a_in;
    a.nq_blk = a.q8 != nullptr ? (int)(a.nq_pad / a.blkq) : 0;
    a.nk_blk = a.k8 != nullptr ? (int)(a.nkv_pad / a.blkk) : 0;
    a.nv_tile = (a.v8 != nullptr || a.v16 != nullptr) ? (int)(a.nkv_pad / 64) : 0;
    if (a.q8 != nullptr && a.nq_pad % a.blkq != 0) return hipErrorInvalidValue;
    if (a.k8 != nullptr && a.nkv_pad % a.blkk != 0) return hipErrorInvalidValue;
    a.n_bh = B * a.H;
    const int has_pre = pre_kind(a.pre_q);
    int64_t total = (int64_t)B * a.H * (a.nq_blk + a.nk_blk + a.nv_tile);
    a.n_sets = 0;
    // Tables of 16 MiB and more, 128 channels: the blocks that read the same table rows share an XCD's L2.  A row of both tables
    // is twice a row of Q or K, and four blocks (two batches) read it.  This launch, us, blocks in the order of heads -> in sets:
    // [2,4352,30,128] 98.9 -> 88.0, [1,4608,24,128] 42.8 -> 36.8, e4m3 [1,9216,40,128] 181.7 -> 165.7, [2,2000,19,128] (19 MB) 34.4 ->
    // 31.1; but e4m3 [2,1001,30,128] (15 MB) 31.8 -> 32.7, [1,700,32,128] 13.4 -> 14.6: the divisions of the mapping are on every
    // workgroup's way (as a branch of the one kernel half a microsecond of small calls too, so it is a kernel of its own), and
    // small tables come from the memory-side cache fast enough.  At 64 channels, workgroups of half the
    // work, that is 1.5 us at any size ([2,4352,24,64] 35.3 -> 36.5).
    // In Q blocks of 32 rows (e4m3 P.V) a set of one batch is six workgroups, half of them short.  With half-split tables nothing is gained
    // (the call, sets against none, 1.00 to 1.02 on average over 63 draws of either batch count, [1,1117,40,128] 73.1 -> 76.0); with
    // interleaved ones and one batch it is level up to 32 MiB and 2 % ahead past it.
    const int64_t table_row = (int64_t)(D / 2) * (a.pre_q.tables_bf16 ? 4 : 8);
    const int batches = a.pre_q.batch_rows == 0 ? B : 1;
    const bool small = a.q8 != nullptr && a.blkq < 128;
    const int64_t from = batches == 1 && small ? 32 << 20 : 16 << 20;
    if (D == 128 && a.pre_q.cos != nullptr && !(small && has_pre == 2) && (int64_t)a.Nq * a.H * table_row * (a.pre_q.batch_rows == 0 ? 1 : B) >= from) {
        // (a run is 128 rows: a block of 128, or several smaller ones)
        a.batches = batches;
        a.q_per = a.q8 != nullptr ? 128 / a.blkq : 0;
        a.k_per = a.k8 != nullptr ? 128 / a.blkk : 0;
        a.members = a.batches * (a.q_per + a.k_per);
        const int64_t runs = max(a.q_per ? (a.nq_blk + a.q_per - 1) / a.q_per : 0, a.k_per ? (a.nk_blk + a.k_per - 1) / a.k_per : 0);
        const int64_t n = set_grid(runs * (a.n_bh / a.batches), a.members);
        total = n + (int64_t)B * a.H * a.nv_tile;
        a.n_sets = (int)min(n, (int64_t)0x7FFFFFFF);
    }
    if (total <= 0 || total > 0x7FFFFFFF) return hipErrorInvalidValue;
    dim3 grid((unsigned)total);
#define SAGE_LAUNCH_QUANT(DD, PP, SETS)                                                                                              \
    do {                                                                                                                             \
        if (f != nullptr) hipLaunchKernelGGL((quant_kernel<DD, PP, true, SETS>), grid, dim3((quant_threads<DD, PP>())), 0, st, a, *f); \
        else hipLaunchKernelGGL((quant_kernel<DD, PP, false, SETS>), grid, dim3((quant_threads<DD, PP>())), 0, st, a, FinalArgs{});    \
    } while (0)
    if (a.n_sets > 0 && has_pre == 2) SAGE_LAUNCH_QUANT(128, 2, true);
    else if (a.n_sets > 0) SAGE_LAUNCH_QUANT(128, 1, true);
    else if (D == 128 && has_pre == 2) SAGE_LAUNCH_QUANT(128, 2, false);
    else if (D == 128 && has_pre) SAGE_LAUNCH_QUANT(128, 1, false);
    else if (D == 128) SAGE_LAUNCH_QUANT(128, 0, false);
    else if (D == 64 && has_pre == 2) SAGE_LAUNCH_QUANT(64, 2, false);
    else if (D == 64 && has_pre) SAGE_LAUNCH_QUANT(64, 1, false);
    else if (D == 64) SAGE_LAUNCH_QUANT(64, 0, false);
    else if (D == 256 && !has_pre) SAGE_LAUNCH_QUANT(256, 0, false);
    else return hipErrorInvalidValue;
#undef SAGE_LAUNCH_QUANT
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// The three launches as one, for short key sequences.  A workgroup of the K and Q roles first computes its
// head's K statistics by itself — the same leaves, groups and order, so the same bits — and then encodes
// one block per half of its threads; a V workgroup takes the head's channel maxima (e4m3) the same way.
// Every workgroup re-reads the head's K (or V) from L2, which is what a short sequence is for: three
// dependent launches of 4 to 6 us each do almost nothing but start and drain there (see quant_short_workgroups).
// ---------------------------------------------------------------------------
constexpr int kShortThreads = 512;

template <int D>
__global__ __launch_bounds__(kShortThreads) void quant_short_kernel(QuantArgs a, FinalArgs f) {
    constexpr int DK = D > 128 ? 128 : D;                 // channels per K statistics call
    constexpr int NWIN = D / DK;                          // windows of DK channels
    constexpr int TPG = 16 * (DK / 8);                    // threads per K group
    constexpr int GPW = kShortThreads / TPG;              // groups at a time
    constexpr int VROWS = kShortThreads / (D / 8);
    constexpr int UNITS = kShortThreads / 256;            // blocks or tiles per workgroup
    union Smem {
        KGroupSmem<DK> kg[GPW];
        float vred[VROWS][D + D / 8];
        float red[UNITS][4];
        uint8_t tile8[UNITS][64 * (D + 16)];
        uint16_t tile16[UNITS][64 * D];
    };
    __shared__ __attribute__((aligned(16))) Smem sm;
    __shared__ __attribute__((aligned(16))) float s_mean[D], s_kmul[D], s_qmul[D];
    __shared__ double s_gsum[GPW][DK];
    __shared__ float s_gmm[GPW][DK][2];
    const int bh = blockIdx.x % a.n_bh;
    int r = blockIdx.x / a.n_bh;
    const int b = bh / a.H, h = bh % a.H;
    const int tid = threadIdx.x, unit = tid >> 8, utid = tid & 255;
    const KeyMask none{0, 0};
    const int nk_wg = (a.nk_blk + UNITS - 1) / UNITS, nq_wg = (a.nq_blk + UNITS - 1) / UNITS;
    if (r < nk_wg + nq_wg) {
        const int sub = tid / TPG, t = tid % TPG;
        // (an odd count: the last workgroup's halves encode the same block)
        const bool is_k = r < nk_wg;
        const int blk = is_k ? min(r * UNITS + unit, a.nk_blk - 1) : min((r - nk_wg) * UNITS + unit, a.nq_blk - 1);
        // The block's rows are requested ahead of the statistics where it has the size the one-shot call gives it.
        constexpr int CPR = D / 8, RPC = 256 / CPR;           // rows per chunk of the half's threads
        u32x4 rows[128 / RPC];
        const int ahead = D <= 128 ? (is_k ? (a.blkk == 64 ? 64 : 0) : (a.blkq == 128 ? 128 : 0)) : 0;
        if constexpr (D <= 128) {
            const View& x = is_k ? a.k : a.q;
            const int n = is_k ? a.Nkv : a.Nq;
            const uint16_t* src = x.p + b * x.sb + h * x.sh + (utid % CPR) * 8;
#pragma unroll
            for (int i = 0; i < 128 / RPC; i++) {
                const int row = blk * ahead + i * RPC + utid / CPR;
                rows[i] = u32x4{0u, 0u, 0u, 0u};
                if (i * RPC < ahead && row < n) rows[i] = *reinterpret_cast<const u32x4*>(src + (int64_t)row * x.sn);
            }
        }
#pragma unroll
        for (int w = 0; w < NWIN; w++) {
            double sum = 0.0;
            float mn = INFINITY, mx = -INFINITY;
            if (f.flags & 3) {
                for (int g0 = 0; g0 < f.ngroups; g0 += GPW) {
                    double gsum;
                    float gmn, gmx;
                    const int g = g0 + sub;
                    kstats_group<DK, 0, D>(g < f.ngroups ? g : -1, h, b, t, a.k.p, a.k.sb, a.k.sh, a.k.sn, a.Nkv, a.H, a.km,
                                             sm.kg[sub], a.pre_k, w * DK, gsum, gmn, gmx);
                    if (f.ngroups == 1) {                   // (nothing to exchange)
                        if (tid < DK) { sum += gsum; mn = fminf(mn, gmn); mx = fmaxf(mx, gmx); }
                        if (NWIN > 1) __syncthreads();      // (the next window's leaves)
                        break;
                    }
                    if (t < DK) { s_gsum[sub][t] = gsum; s_gmm[sub][t][0] = gmn; s_gmm[sub][t][1] = gmx; }
                    __syncthreads();
                    if (tid < DK) {
#pragma unroll
                        for (int u = 0; u < GPW; u++)
                            if (g0 + u < f.ngroups) {
                                sum += s_gsum[u][tid];
                                mn = fminf(mn, s_gmm[u][tid][0]);
                                mx = fmaxf(mx, s_gmm[u][tid][1]);
                            }
                    }
                    __syncthreads();
                }
            }
            if (tid < DK) {
                float mean, s;
                k_final(sum, mn, mx, f.kept, f.flags, mean, s);
                const int d = w * DK + leaf_channel<DK>(tid);
                const float kmul = 1.0f / s, qmul = f.cmul * s;
                s_mean[d] = mean; s_kmul[d] = kmul; s_qmul[d] = qmul;
                if (r == 0) {
                    const int64_t i = (int64_t)bh * D + d;
                    f.kmean[i] = mean; f.kmul[i] = kmul; f.qmul[i] = qmul;
                }
            }
        }
        __syncthreads();
#define SAGE_K(BLK, HAVE) quant_i8_block<D, BLK, true, 0, 256, HAVE>(blk, h, b, utid, a.k.p, a.k.sb, a.k.sh, a.k.sn, a.Nkv, a.H, a.nkv_pad, a.km, \
                                                       s_mean, s_kmul, 0.0f, a.k8, a.kscale, nullptr, sm.red[unit], a.pre_k, rows)
#define SAGE_Q(BLK, HAVE) quant_i8_block<D, BLK, false, 0, 256, HAVE>(blk, h, b, utid, a.q.p, a.q.sb, a.q.sh, a.q.sn, a.Nq, a.H, a.nq_pad, none, \
                                                        s_mean, s_qmul, a.cmul, a.q8, a.qscale, a.rowdot, sm.red[unit], a.pre_q, rows)
        constexpr bool HAVE = D <= 128;
        if (is_k) {
            if (a.blkk == 128) SAGE_K(128, false);
            else if (a.blkk == 64) SAGE_K(64, HAVE);
            else SAGE_K(32, false);
        } else {
            if (a.blkq == 128) SAGE_Q(128, HAVE);
            else if (a.blkq == 64) SAGE_Q(64, false);
            else SAGE_Q(32, false);
        }
#undef SAGE_Q
#undef SAGE_K
        return;
    }
    const int t = (r - nk_wg - nq_wg) * UNITS + unit;     // (the key padding makes the tile count even)
    if (a.v16 != nullptr) {
        quant_v_f16_body<D>(t, h, b, utid, a.v.p, a.v.sb, a.v.sh, a.v.sn, a.Nkv, a.H, a.nkv_pad, a.km, a.v16, sm.tile16[unit]);
        return;
    }
    {
        constexpr int CPR = D / 8;
        const int col = (tid % CPR) * 8, row0 = tid / CPR;
        const uint16_t* src = a.v.p + b * a.v.sb + h * a.v.sh + col;
        float m[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll 8
        for (int row = row0; row < a.Nkv; row += VROWS) {
            u32x4 w = {0u, 0u, 0u, 0u};
            if (key_kept(row, a.Nkv, a.km)) w = *reinterpret_cast<const u32x4*>(src + (int64_t)row * a.v.sn);
            float x[8];
            unpack8(w, x);
#pragma unroll
            for (int e = 0; e < 8; e++) m[e] = fmaxf(m[e], fabsf(x[e]));
        }
#pragma unroll
        for (int e = 0; e < 8; e++) sm.vred[row0][e * CPR + (col >> 3)] = m[e];
        __syncthreads();
        if (tid < D) {
            float amax = 0.0f;
#pragma unroll
            for (int i = 0; i < VROWS; i++) amax = fmaxf(amax, sm.vred[i][tid]);
            const float sc = amax > 0.0f ? amax / 448.0f : 1.0f;
            const int d = leaf_channel<D>(tid);
            s_mean[d] = sc;
            if (r == nk_wg + nq_wg) f.vscale[(int64_t)bh * D + d] = sc;
        }
        __syncthreads();
    }
    quant_v_fp8_body<D, 256>(t, h, b, utid, a.v.p, a.v.sb, a.v.sh, a.v.sn, a.Nkv, a.H, a.nkv_pad, a.km, s_mean, a.v8, sm.tile8[unit]);
}

static void short_units(QuantArgs& a, int B, bool with_q) {
    a.nq_blk = with_q ? (int)(a.nq_pad / a.blkq) : 0;
    a.nk_blk = (int)(a.nkv_pad / a.blkk);
    a.nv_tile = (int)(a.nkv_pad / 64);
    a.n_bh = B * a.H;
}
static int64_t short_workgroups(const QuantArgs& a) { return (int64_t)a.n_bh * ((a.nq_blk + 1) / 2 + (a.nk_blk + 1) / 2 + a.nv_tile / 2); }

// One launch where a workgroup gets through its head's statistics in one pass (1024 keys at 64 channels, 512
// at 128; at 256 channels, where they take two windows, 256) and all workgroups are resident at once (two
// per compute unit).  Measured over 4 to 60 heads, stage of three launches -> one, us: 11.5-15 -> 7.5-9.5 up
// to 256 keys, 13-15 -> 9-12.8 at 512 keys of 128 channels, 12-13.4 -> 8.4-10.7 at 1024 keys of 64; a second
// pass costs 4 us and a second generation of workgroups 7, which is what the two launches less are worth.
// Never with the pre-ops in front: a workgroup would norm and rotate every key of its head, a longer chain than the launch
// saved.  The call, us, one launch -> two, the first of them prep_rows_kernel: [1,8 heads,128,64] 21.7 -> 18.5, [1,24,512,64] 26.6 ->
// 22.6, [2,30,200,128] 31.9 -> 30.6, [1,24,333,128] 35.8 -> 30.2, [2,30,500,64] level; e4m3 [1,8,300,64] 22.5 -> 20.0, [1,24,512,64]
// 34.9 -> 20.9, [2,30,200,128] 39.2 -> 30.5, [1,19,150,128] 24.9 -> 24.4.
static int64_t short_rule(const QuantArgs& a, int D) {
    const int groups = (a.Nkv + kGroup - 1) / kGroup, most = D == 64 ? 4 : D == 128 ? 2 : 1;
    const int64_t wgs = short_workgroups(a);
    return groups <= most && wgs <= 512 ? wgs : 0;
}
int64_t quant_short_workgroups(const QuantArgs& a_in, int B, int D) {
    QuantArgs a = a_in;
    short_units(a, B, a.q8 != nullptr);
    if (a.pre_k.gain != nullptr) return 0;
    return short_rule(a, D);
}
int64_t quant_short_workgroups(int B, int H, int Nq, int Nkv, int D, int blkq, int blkk, bool with_q) {
    QuantArgs a{};
    a.H = H; a.Nkv = Nkv; a.blkq = blkq; a.blkk = blkk;
    a.nq_pad = pad_to(Nq, kTileQ); a.nkv_pad = pad_to(Nkv, kPadKV);
    short_units(a, B, with_q);
    return short_rule(a, D);
}

hipError_t launch_quant_short(const QuantArgs& a_in, const FinalArgs& f_in, int B, int D, hipStream_t st) {
    QuantArgs a = a_in;
    short_units(a, B, a.q8 != nullptr);
    if ((a.q8 != nullptr && a.nq_pad % a.blkq != 0) || a.nkv_pad % a.blkk != 0 || a.k8 == nullptr || (a.v8 == nullptr && a.v16 == nullptr))
        return hipErrorInvalidValue;
    const int64_t total = short_workgroups(a);
    if (total <= 0 || total > 0x7FFFFFFF || (a.nv_tile & 1)) return hipErrorInvalidValue;
    const dim3 grid((unsigned)total), block(kShortThreads);
    if (a.pre_q.gain != nullptr || a.pre_k.gain != nullptr) return hipErrorInvalidValue;
    if (D == 128) hipLaunchKernelGGL(quant_short_kernel<128>, grid, block, 0, st, a, f_in);
    else if (D == 64) hipLaunchKernelGGL(quant_short_kernel<64>, grid, block, 0, st, a, f_in);
    else if (D == 256) hipLaunchKernelGGL(quant_short_kernel<256>, grid, block, 0, st, a, f_in);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// The whole stage as one launch with the statistics handed over between workgroups.  A workgroup takes a group of 256 keys,
// keeps its rows in registers, publishes the group's sums, minima and maxima, waits for those of the head's other groups and
// encodes: K (and, for e4m3, V) is read once instead of twice, and two launches' starts and ends go.
//
// The hand-over.  Results and flags are written and read by relaxed atomics of agent scope only: these go past the L2s of the
// XCDs, which are not coherent with each other inside a kernel, and need none of the write-backs and invalidations that a
// fence of that scope is.  A flag is raised when the wave's stores are complete (vmcnt) behind a barrier of the workgroup.
// Flags hold a number that no other call of the process uses, so memory may hold anything before; a call under capture, whose
// replays would all use one number, takes the launches.
// The wait is bounded.  A workgroup that sees a flag missing after `polls` looks computes the missing groups of its head itself, the same values
// into the same places, and raises their flags: nothing depends on which workgroups are resident together, only the time does.  To have
// them resident, heads come in chunks (OnceArgs::heads), their K groups first: a group waits for workgroups in front of it and a few
// behind it.
// Where another stream's kernel holds the chip they are not, and who waits keeps a compute unit from whoever it waits for: hence a bound of few looks.  Beside
// back-to-back e4m3 [1,16896,24,128] calls of another stream, us a call and ms for twelve of the other's, by launches / with 1024 looks and all groups
// computed by whoever gave up / now: [1,4608,24,128] 778 and 28.2 / 912 and 30.7 / 702 and 28.3; [2,2048,32,128] 550 and 26.9 / 840 and 28.8 / 608
// and 26.6; [1,2304,12,64] 398 / 212 / 216.  The same calls on two streams at once, us a call: [1,1153,24,128] 30.5 / 28.8 / 28.8,
// [2,2048,32,128] 134 / 126 / 124, but [1,4608,24,128] 195 / 216 to 271 / 214: the launches' small workgroups find room beside those of the
// attention kernel, a group's does not (one stream: 229 / 221 / 221).
// Every workgroup adds up the group results of its head itself, in group order.
// What a K workgroup's time goes to at [1,1153,24,128] (one per compute unit), us: rows 1.6, sums and handing over 3, waiting 1.7, adding up 0.9,
// encoding 2.6, next to 3 of the launch's start and end; bandwidth comes first from about 400 groups on.  (Encoding was 3.4 with a pass over
// the rows for the blocks' largest values, which a leaf's extremes say without one, and the true quotient inside the unrolled loop:
// e4m3 [1,256 x 1971,24,64] 22.0 -> 21.3 us, [1,2432,12,128] 51.8 -> 50.6, bias [1,1153,24,128] 49.9 -> 49.5.)  (Statistics
// published once per head by the last group's workgroup: 6 us instead of 1.8 of waiting and adding up at 18 groups.  At 256 channels a
// workgroup has a compute unit to itself: [2,2688,32,256] 503 -> 790 us; not built.)
// ---------------------------------------------------------------------------

template <typename T> __device__ __forceinline__ T agent_load(const T* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
template <typename T> __device__ __forceinline__ void agent_store(T* p, T v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
// (stores of this wave have reached the place agent-scope loads read)
__device__ __forceinline__ void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

template <int D> struct OnceShape {
    static constexpr int CH = 4, CPR = D / CH, NT = 16 * CPR;       // channels per thread, threads per leaf and group
    static constexpr int WPB = 4 * CPR / 64;                                      // waves per scale block of 64 keys
    static constexpr int LD = D + D / 8;
    static constexpr int VT = D == 128 ? 2 : 1;                                   // fp16 V tiles per workgroup
    static constexpr int CPR8 = D / 8, RP = NT / CPR8;                            // rows per pass in chunks of eight channels
};
template <int D, int PRE> union OnceSmem {
    using S = OnceShape<D>;
    struct { double sum[16][S::LD]; float mn[16][S::LD], mx[16][S::LD]; } leaf;
    u32x4 rows[PRE ? kGroup * S::CPR8 : 1];
    float vred[S::RP][S::LD];
    uint8_t tile8[4][64 * (D + 16)];
    uint16_t tile16[4][64 * D];
    float red[16];
};
template <int D> struct OnceHead { float mean[D], kmul[D], qmul[D]; };             // mean: also V's scales

// flags[0 .. n) hold tag, within `polls` looks.  One wave calls it.
__device__ __forceinline__ bool flags_up(const uint64_t* flags, int n, uint64_t tag, int polls, int lane) {
    for (int p = 0; p < polls; p++) {
        bool up = true;
        for (int i = lane; i < n; i += 64) up = up && agent_load(flags + i) == tag;
        if (__all(up)) return true;
        __builtin_amdgcn_s_sleep(2);
    }
    return false;
}

// Groups that workgroups computed after they had waited for them, since the last reset (mi355_sage_quant_once_helps).
static __device__ unsigned int g_once_helps;

// The groups 0 .. n - 1 whose flag is missing, by this workgroup, from `from` on in a ring: group(g) leaves its results in memory, complete
// behind a barrier.  Their flags are raised for whoever else waits.  (ok: in LDS, read by all before.)
template <typename F>
__device__ __forceinline__ void help_missing(uint64_t* flags, int n, int from, uint64_t tag, bool raise, int tid, int& ok, F group) {
    int g = from;
#pragma unroll 1
    do {
        __syncthreads();
        asm volatile("" : "+s"(tag));               // (or vector registers hold it from one group to the next)
        if (tid == 0) ok = agent_load(flags + g) == tag;
        __syncthreads();
        if (ok == 0) {
            group(g);
            if (tid == 0) {
                atomicAdd(&g_once_helps, 1u);
                if (raise) agent_store(flags + g, tag);
            }
        }
        g = g + 1 == n ? 0 : g + 1;
    } while (g != from);
}

// One group of keys in registers: a leaf of CH channels per thread.
template <int D, int PRE>
struct OnceGroup {
    using S = OnceShape<D>;
    static constexpr int CH = S::CH, W = CH / 2;
    uint32_t w[kLeaf][W];
    uint32_t ext[CH];                               // smallest and largest value of this thread's leaf per channel, as the bf16 they are (publish)
    bool ext_known;                                 // ... which they are in all of the wave's leaves
    bool all_kept;                                  // every token of the wave's leaves counts
    __device__ static __forceinline__ int leaf(int tid) { return tid / S::CPR; }
    __device__ static __forceinline__ int col(int tid) { return tid % S::CPR * CH; }

    // (what was computed from the rows is computed again behind this, not kept in registers)
    __device__ __forceinline__ void pin() {
#pragma unroll
        for (int i = 0; i < kLeaf; i++)
#pragma unroll
            for (int e = 0; e < W; e++) asm volatile("" : "+v"(w[i][e]));
    }

    // Rows of group g; what does not count is zero.  (With the pre-ops: meets two barriers.)
    __device__ __forceinline__ void load(const QuantArgs& a, int g, int h, int b, int tid, OnceSmem<D, PRE>& sm) {
        asm volatile("" : "+v"(tid));               // (row addresses are formed where they are used, not held from one call to the next)
        const int s0 = g * kGroup + leaf(tid) * kLeaf, N = a.Nkv;
        all_kept = __all(s0 + kLeaf <= N && !(s0 < a.km.hi && s0 + kLeaf > a.km.lo));
        if constexpr (PRE) {
            constexpr int CPR8 = S::CPR8, NR = 2, AHEAD = PRE == 2 ? 1 : 2;
            const int c8 = tid % CPR8 * 8;
            const uint16_t* src = a.k.p + b * a.k.sb + h * a.k.sh + c8;
            const RopeAt rope = rope_at<D>(a.pre_k, b, h, a.H, c8);
            float gain[8];
            pre_gains(a.pre_k, h, D, c8, gain);
#pragma unroll 1
            for (int r0 = 0; r0 < kGroup; r0 += NR * S::RP) {          // (registers for four rows at a time)
                const int first = g * kGroup + r0 + tid / CPR8;
                auto clamped = [&](int i) { return min(first + i * S::RP, N - 1); };
                u32x4 raw[NR];
                RopeTab<PRE> tab[AHEAD];
#pragma unroll
                for (int i = 0; i < NR; i++) raw[i] = *reinterpret_cast<const u32x4*>(src + (int64_t)clamped(i) * a.k.sn);
#pragma unroll
                for (int i = 0; i < AHEAD; i++) rope_load<PRE>(rope, clamped(i), tab[i]);
                float inv[NR];
                row_inverses<D, NR>(a.pre_k.eps, raw, inv);
#pragma unroll
                for (int i = 0; i < NR; i++) {
                    float x[8];
                    unpack8(raw[i], x);
                    pre_apply<D, PRE>(a.pre_k, c8, key_kept(first + i * S::RP, N, a.km), inv[i], gain, tab[i % AHEAD], x);
                    if (i + AHEAD < NR) rope_load<PRE>(rope, clamped(i + AHEAD), tab[i % AHEAD]);
                    u32x4 y;                                           // (bf16 values: nothing below their upper halves)
#pragma unroll
                    for (int e = 0; e < 4; e++) y[e] = __builtin_amdgcn_perm(__float_as_uint(x[2 * e + 1]), __float_as_uint(x[2 * e]), 0x07060302u);
                    sm.rows[(r0 + i * S::RP) * CPR8 + tid] = y;
                }
            }
            __syncthreads();
            const uint32_t* r32 = reinterpret_cast<const uint32_t*>(sm.rows);
#pragma unroll
            for (int i = 0; i < kLeaf; i++) {
                const u32x2 v = *reinterpret_cast<const u32x2*>(r32 + ((leaf(tid) * kLeaf + i) * D + col(tid)) / 2);
                w[i][0] = v.x; w[i][1] = v.y;
            }
            __syncthreads();                                       // (the leaves' results go where the rows are)
        } else {
            const uint16_t* src = a.k.p + b * a.k.sb + h * a.k.sh + col(tid);
#pragma unroll
            for (int i = 0; i < kLeaf; i++) {
                const u32x2 v = *reinterpret_cast<const u32x2*>(src + (int64_t)min(s0 + i, N - 1) * a.k.sn);
                w[i][0] = v.x; w[i][1] = v.y;
            }
            if (!all_kept) {
#pragma unroll
                for (int i = 0; i < kLeaf; i++)
                    if (!key_kept(s0 + i, N, a.km)) {
#pragma unroll
                        for (int e = 0; e < W; e++) w[i][e] = 0u;
                    }
            }
        }
    }

    // The rows once more, without what publish keeps of them.
    __device__ __forceinline__ void reload(const QuantArgs& a, int g, int h, int b, int tid, OnceSmem<D, PRE>& sm) {
        load(a, g, h, b, tid, sm);
        ext_known = false;
#pragma unroll
        for (int e = 0; e < CH; e++) ext[e] = 0u;
    }

    // The group's sums, minima and maxima to memory: the tree of kstats_group.  (Meets two barriers; stores complete behind them.)
    __device__ __forceinline__ void publish(const QuantArgs& a, const FinalArgs& f, int64_t bh, int g, int tid, OnceSmem<D, PRE>& sm) {
        asm volatile("" : "+v"(tid));
        __builtin_assume(tid >= 0);                                // (or its sign is a register of its own)
        const int s0 = g * kGroup + leaf(tid) * kLeaf, c = col(tid);
        double acc[CH];
        float mn[CH], mx[CH];
#pragma unroll
        for (int e = 0; e < CH; e++) { acc[e] = 0.0; mn[e] = INFINITY; mx[e] = -INFINITY; }
#pragma unroll
        for (int i = 0; i < kLeaf; i += 2) {
            __builtin_amdgcn_sched_barrier(0);                     // (or all sixteen tokens are converted first)
            float x[2][CH];
#pragma unroll
            for (int r = 0; r < 2; r++)
#pragma unroll
                for (int e = 0; e < W; e++) { x[r][2 * e] = bf16_lo(w[i + r][e]); x[r][2 * e + 1] = bf16_hi(w[i + r][e]); }
            // (tokens that do not count are +0.0, which leaves a double sum unchanged)
#pragma unroll
            for (int r = 0; r < 2; r++)
#pragma unroll
                for (int e = 0; e < CH; e++) acc[e] += (double)x[r][e];
            if (!all_kept) {
                // (a quiet NaN takes no part in a minimum or maximum; nor does one that signals in a leaf that is cut, as in kstats_group.
                // The pre-ops leave none)
                const bool whole = s0 + kLeaf <= a.Nkv && !(s0 < a.km.hi && s0 + kLeaf > a.km.lo);
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    const bool kept = key_kept(s0 + i + r, a.Nkv, a.km);
                    if constexpr (!PRE) {
#pragma unroll
                        for (int e = 0; e < CH; e++) x[r][e] = whole ? x[r][e] : __builtin_canonicalizef(x[r][e]);
                    }
                    if (!kept)
#pragma unroll
                        for (int e = 0; e < CH; e++) x[r][e] = __builtin_nanf("");
                }
            }
            // (as instructions: see kstats_group)
#pragma unroll
            for (int e = 0; e < CH; e++) {
                asm("v_min3_f32 %0, %0, %1, %2" : "+v"(mn[e]) : "v"(x[0][e]), "v"(x[1][e]));
                asm("v_max3_f32 %0, %0, %1, %2" : "+v"(mx[e]) : "v"(x[0][e]), "v"(x[1][e]));
            }
        }
        // (where a leaf's values do not add up to a number, one of them may be a NaN that signals: min3 and max3 put it in the extreme's place)
        if constexpr (!PRE) {
            bool odd = false;
#pragma unroll
            for (int e = 0; e < CH; e++) odd = odd || acc[e] != acc[e];
            ext_known = !__any(odd);
        }
#pragma unroll
        for (int e = 0; e < CH; e++) {
            const int at = ((c + e) & 7) * S::CPR8 + (c >> 3);      // (as in KGroupSmem)
            sm.leaf.sum[leaf(tid)][at] = acc[e];
            sm.leaf.mn[leaf(tid)][at] = mn[e];
            sm.leaf.mx[leaf(tid)][at] = mx[e];
            ext[e] = __builtin_amdgcn_perm(__float_as_uint(mx[e]), __float_as_uint(mn[e]), 0x07060302u);
        }
        __syncthreads();
        if (tid < D) {
            double sum = 0.0;
#pragma unroll
            for (int u = 0; u < 16; u++) sum += sm.leaf.sum[u][tid];
            agent_store(f.kpart_sum + (bh * f.ngroups + g) * D + leaf_channel<D>(tid), sum);
        } else if (tid < 2 * D) {
            const int t = tid - D;
            float lo = INFINITY, hi = -INFINITY;
#pragma unroll
            for (int u = 0; u < 16; u++) {
                lo = fminf(lo, sm.leaf.mn[u][t]);
                hi = fmaxf(hi, sm.leaf.mx[u][t]);
            }
            agent_store(reinterpret_cast<uint64_t*>(f.kpart_mm) + (bh * f.ngroups + g) * D + leaf_channel<D>(t),
                        (uint64_t)__float_as_uint(lo) | (uint64_t)__float_as_uint(hi) << 32);
        }
        stores_done();
        __syncthreads();
    }

    // Codes and scales of the group's blocks of 64 keys.  (Meets a barrier.)
    __device__ __forceinline__ void encode(const QuantArgs& a, int64_t bh, int g, int h, int b, int tid, OnceSmem<D, PRE>& sm, const OnceHead<D>& hd) {
        asm volatile("" : "+v"(tid));
        const int s0 = g * kGroup + leaf(tid) * kLeaf, c = col(tid), wave = tid >> 6;
        float mu[CH], mul[CH];
#pragma unroll
        for (int e = 0; e < CH; e++) { mu[e] = hd.mean[c + e]; mul[e] = hd.kmul[c + e]; }
        float am = 0.0f;
        if constexpr (PRE) {
            // (the extremes, kept that long, are one register too many here)
#pragma unroll
            for (int i = 0; i < kLeaf; i++)
                if (all_kept || key_kept(s0 + i, a.Nkv, a.km)) {
#pragma unroll
                    for (int e = 0; e < CH; e++) {
                        const float d = (e & 1 ? bf16_hi(w[i][e >> 1]) : bf16_lo(w[i][e >> 1])) - mu[e];
                        am = fmaxf(am, fabsf(d * mul[e]));
                    }
                }
        } else if (__builtin_expect(!ext_known, 0)) {
            const uint16_t* src = a.k.p + b * a.k.sb + h * a.k.sh + c;
#pragma unroll 1
            for (int i = 0; i < kLeaf; i++) {
                if (!key_kept(s0 + i, a.Nkv, a.km)) continue;
                const u32x2 v = *reinterpret_cast<const u32x2*>(src + (int64_t)(s0 + i) * a.k.sn);
#pragma unroll
                for (int e = 0; e < CH; e++) {
                    const float d = (e & 1 ? bf16_hi(v[e >> 1]) : bf16_lo(v[e >> 1])) - mu[e];
                    am = fmaxf(am, fabsf(d * mul[e]));
                }
            }
        } else {
            // (rounding is monotone: a leaf's largest |(k - mean) mul| in a channel is that of its largest or its smallest k)
#pragma unroll
            for (int e = 0; e < CH; e++) {
                const float mn = bf16_lo(ext[e]), mx = bf16_hi(ext[e]);
                if (mn <= mx) {                                     // (not: a leaf without a key that counts)
                    const float hi = mx - mu[e], lo = mn - mu[e];
                    am = fmaxf(fmaxf(am, fabsf(hi * mul[e])), fabsf(lo * mul[e]));
                }
            }
        }
        pin();
        am = wave_max(am);
        if constexpr (S::WPB == 2) {
            if ((tid & 63) == 0) sm.red[wave] = am;
            __syncthreads();
            am = fmaxf(am, sm.red[wave ^ 1]);
        }
        const float sc = am > 0.0f ? am / 127.0f : 1.0f;
        const bool there = s0 < a.nkv_pad;                          // (whole leaves)
        if (there && (tid & (64 * S::WPB - 1)) == 0) a.kscale[bh * (a.nkv_pad / 64) + (s0 >> 6)] = sc;
        const bool fast = sc >= 0x1p-100f && sc <= 0x1p100f;
        const float rinv = 1.0f / sc;
        int8_t* out = a.k8 + (bh * a.nkv_pad + s0) * D + c;
        // two tokens of four channels as one chunk of eight values
        auto chunk = [&](int i, const uint32_t (&w0)[W], const uint32_t (&w1)[W], float (&x)[8]) {
#pragma unroll
            for (int r = 0; r < 2; r++) {
                const bool kept = all_kept || key_kept(s0 + i + r, a.Nkv, a.km);
#pragma unroll
                for (int e = 0; e < CH; e++) {
                    const uint32_t u = r ? w1[e >> 1] : w0[e >> 1];
                    const float d = (e & 1 ? bf16_hi(u) : bf16_lo(u)) - mu[e];
                    x[r * CH + e] = d * mul[e];
                    if (!kept) x[r * CH + e] = 0.0f;
                }
            }
        };
        auto put = [&](int i, const u32x2& o) {
            if (!there) return;
            *reinterpret_cast<uint32_t*>(out + i * D) = o.x;
            *reinterpret_cast<uint32_t*>(out + (i + 1) * D) = o.y;
        };
        uint32_t redo = fast ? 0u : (1u << (kLeaf / 2)) - 1u;
#pragma unroll
        for (int i = 0; i < kLeaf; i += 2) {
            __builtin_amdgcn_sched_barrier(0);
            float x[8];
            bool near;
            chunk(i, w[i], w[i + 1], x);
            put(i, encode8_common(x, rinv, near));
            redo |= near ? 1u << (i / 2) : 0u;
        }
        redo_chunks(redo, [&](int j) {
            uint32_t w0[W], w1[W];
#pragma unroll
            for (int e = 0; e < W; e++) {
                w0[e] = w[0][e];
                w1[e] = w[1][e];
#pragma unroll
                for (int i = 2; i < kLeaf; i += 2) {
                    w0[e] = j == i / 2 ? w[i][e] : w0[e];
                    w1[e] = j == i / 2 ? w[i + 1][e] : w1[e];
                    asm volatile("" : "+v"(w0[e]), "+v"(w1[e]));    // (or the rows go to memory, to be indexed there)
                }
            }
            float x[8];
            chunk(j * 2, w0, w1, x);
            put(j * 2, encode8_quotient(x, sc, rinv, fast));
        });
    }
};

// The head's K statistics into hd, for a workgroup of NT threads; `leave`: and into memory, for later launches.
// Returns false where it computed the groups itself: what the caller held in registers is then to be loaded again.
template <int D, int PRE>
__device__ __forceinline__ bool once_k_head(const OnceArgs& a, int64_t bh, int h, int b, int from, int tid, bool leave, OnceSmem<D, PRE>& sm, OnceHead<D>& hd, int& s_ok) {
    const FinalArgs& f = a.f;
    if (tid < 64) {
        const bool up = flags_up(a.flags + bh * a.flag_words, f.ngroups, a.tag, a.polls, tid);
        if (tid == 0) s_ok = up;
    }
    __syncthreads();
    const bool ok = s_ok != 0;
    if (__builtin_expect(!ok, 0)) {
        help_missing(a.flags + bh * a.flag_words, f.ngroups, (int)((unsigned)from % (unsigned)f.ngroups), a.tag, a.raise, tid, s_ok, [&](int g) {
            OnceGroup<D, PRE> grp;
            grp.load(a.q, g, h, b, tid, sm);
            grp.publish(a.q, f, bh, g, tid, sm);
        });
    }
    if (tid < D) {
        constexpr int NB = 12;
        const double* p = f.kpart_sum + bh * f.ngroups * D + tid;
        const uint64_t* mm = reinterpret_cast<const uint64_t*>(f.kpart_mm) + bh * f.ngroups * D + tid;
        double sum = 0.0;
        float mn = INFINITY, mx = -INFINITY, mean, s;
        for (int g0 = 0; g0 < f.ngroups; g0 += NB) {
            double v[NB];
            uint64_t lh[NB];
#pragma unroll
            for (int j = 0; j < NB; j++) {
                const int g = min(g0 + j, f.ngroups - 1);
                v[j] = agent_load(p + g * D);
                lh[j] = agent_load(mm + g * D);
            }
#pragma unroll
            for (int j = 0; j < NB; j++)
                if (g0 + j < f.ngroups) {
                    sum += v[j];
                    mn = fminf(mn, __uint_as_float((uint32_t)lh[j]));
                    mx = fmaxf(mx, __uint_as_float((uint32_t)(lh[j] >> 32)));
                }
        }
        k_final(sum, mn, mx, f.kept, f.flags, mean, s);
        const float kmul = 1.0f / s, qmul = f.cmul * s;
        if (leave) {
            const int64_t i = bh * D + tid;
            f.kmean[i] = mean; f.kmul[i] = kmul; f.qmul[i] = qmul;
        }
        hd.mean[tid] = mean; hd.kmul[tid] = kmul; hd.qmul[tid] = qmul;
    }
    __syncthreads();
    return ok;
}

// A group of 256 values of V: channel maxima, then e4m3 tiles.  The same hand-over.
template <int D> struct OnceV {
    using S = OnceShape<D>;
    static constexpr int NCH = kGroup / S::RP;
    u32x4 w[NCH];
    __device__ __forceinline__ void pin() {
#pragma unroll
        for (int i = 0; i < NCH; i++) asm volatile("" : "+v"(w[i]));
    }
    __device__ __forceinline__ void load(const QuantArgs& a, int g, int h, int b, int tid) {
        asm volatile("" : "+v"(tid));               // (as in OnceGroup)
        const uint16_t* src = a.v.p + b * a.v.sb + h * a.v.sh + tid % S::CPR8 * 8;
#pragma unroll
        for (int i = 0; i < NCH; i++) {
            const int row = g * kGroup + i * S::RP + tid / S::CPR8;
            w[i] = *reinterpret_cast<const u32x4*>(src + (int64_t)min(row, a.Nkv - 1) * a.v.sn);
        }
        if (g * kGroup + kGroup > a.Nkv || a.km.hi > a.km.lo) {
#pragma unroll
            for (int i = 0; i < NCH; i++)
                if (!key_kept(g * kGroup + i * S::RP + tid / S::CPR8, a.Nkv, a.km)) w[i] = u32x4{0u, 0u, 0u, 0u};
        }
    }
    __device__ __forceinline__ void publish(const FinalArgs& f, int64_t bh, int g, int tid, float (*red)[S::LD]) const {
        float m[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < NCH; i++) {
            float x[8];
            unpack8(w[i], x);
#pragma unroll
            for (int e = 0; e < 8; e++) m[e] = fmaxf(m[e], fabsf(x[e]));
        }
#pragma unroll
        for (int e = 0; e < 8; e++) red[tid / S::CPR8][e * S::CPR8 + tid % S::CPR8] = m[e];      // (as in KGroupSmem)
        __syncthreads();
        if (tid < D) {
            float mm = 0.0f;
#pragma unroll
            for (int i = 0; i < S::RP; i++) mm = fmaxf(mm, red[i][tid]);
            agent_store(f.vpart + (bh * f.ngroups + g) * D + leaf_channel<D>(tid), mm);
        }
        stores_done();
        __syncthreads();
    }
};

// The fp16 tiles of a group of 256 values of V whose rows are in registers.  (Meets a barrier.)
template <int D>
__device__ __forceinline__ void once_v_f16(const QuantArgs& a, int64_t bh, int g, int tid, const OnceV<D>& v, uint16_t (*tile)[64 * D]) {
    using S = OnceShape<D>;
#pragma unroll
    for (int i = 0; i < OnceV<D>::NCH; i++) {
        const int key = i * S::RP + tid / S::CPR8, slot = v_slot_f16(key & 63);
        float x[8];
        unpack8(v.w[i], x);
        const u32x4 o = {f16_pair_sat(x[0], x[1]), f16_pair_sat(x[2], x[3]), f16_pair_sat(x[4], x[5]), f16_pair_sat(x[6], x[7])};
        *reinterpret_cast<u32x4*>(&tile[key >> 6][slot * D + v_tile_chunk<D>(slot, tid % S::CPR8) * 8]) = o;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; j++)
        if ((g * 4 + j) * 64 < a.nkv_pad)
            store_v_f16_tile<D, S::NT>(tid, tile[j], a.v16 + (bh * (a.nkv_pad / 64) + g * 4 + j) * (int64_t)(D * 64));
}

// Block r of BLK queries, whose rows are requested ahead of the wait.
template <int D, int PRE, int BLK>
__device__ __forceinline__ void once_q_block(const OnceArgs& o, int64_t bh, int h, int b, int r, int tid, OnceSmem<D, PRE>& sm, OnceHead<D>& hd, int& s_ok) {
    using S = OnceShape<D>;
    constexpr int NCH = BLK * S::CPR8 / S::NT;
    const QuantArgs& a = o.q;
    u32x4 rows[NCH];
    auto load = [&] {
        const uint16_t* src = a.q.p + b * a.q.sb + h * a.q.sh + tid % S::CPR8 * 8;
#pragma unroll
        for (int i = 0; i < NCH; i++) {
            const int row = r * BLK + i * S::RP + tid / S::CPR8;
            rows[i] = u32x4{0u, 0u, 0u, 0u};
            if (row < a.Nq) rows[i] = *reinterpret_cast<const u32x4*>(src + (int64_t)row * a.q.sn);
        }
    };
    load();
    if (!once_k_head<D, PRE>(o, bh, h, b, r, tid, false, sm, hd, s_ok)) load();
    quant_i8_block<D, BLK, false, PRE, S::NT, true>(r, h, b, tid, a.q.p, a.q.sb, a.q.sh, a.q.sn, a.Nq, a.H, a.nq_pad, KeyMask{0, 0}, hd.mean, hd.qmul,
                                                    a.cmul, a.q8, a.qscale, a.rowdot, sm.red, a.pre_q, rows);
}

template <int D, int PRE>
__global__ __launch_bounds__((OnceShape<D>::NT), 4) void quant_once_kernel(OnceArgs o) {
    using S = OnceShape<D>;
    constexpr int NT = S::NT;
    __shared__ __attribute__((aligned(16))) OnceSmem<D, PRE> sm;
    __shared__ __attribute__((aligned(16))) OnceHead<D> hd;
    __shared__ int s_ok;
    const QuantArgs& a = o.q;
    const FinalArgs& f = o.f;
    // heads in chunks; inside one, K groups, V, Q blocks, and consecutive workgroups take the same rows of consecutive heads
    const int per = o.nk + o.nv + o.nkb + a.nq_blk, chunk = (int)blockIdx.x / (o.heads * per), in = (int)blockIdx.x - chunk * o.heads * per;
    const int heads = min(o.heads, a.n_bh - chunk * o.heads);
    const int unit = in / heads, bh = chunk * o.heads + in % heads;
    const int b = bh / a.H, h = bh % a.H, tid = threadIdx.x;
    uint64_t* flags = o.flags + (int64_t)bh * o.flag_words;
    if (unit < o.nk) {
        OnceGroup<D, PRE> grp;
        grp.load(a, unit, h, b, tid, sm);
        grp.publish(a, f, bh, unit, tid, sm);
        if (tid == 0 && o.raise) agent_store(flags + unit, o.tag);
        if (PRE == 0 && o.k_apart) return;
        if (o.v_in) {
            OnceV<D> v;
            grp.pin();
            v.load(a, unit, h, b, tid);
            once_v_f16<D>(a, bh, unit, tid, v, sm.tile16);
            __syncthreads();
        }
        if (!once_k_head<D, PRE>(o, bh, h, b, unit, tid, unit == 0, sm, hd, s_ok)) grp.reload(a, unit, h, b, tid, sm);
        grp.encode(a, bh, unit, h, b, tid, sm, hd);
    } else if (unit < o.nk + o.nv) {
        const int t = unit - o.nk;
        if (a.v16 != nullptr) {
            constexpr int UT = NT / S::VT;
            quant_v_f16_body<D, UT>(t * S::VT + tid / UT, h, b, tid % UT, a.v.p, a.v.sb, a.v.sh, a.v.sn, a.Nkv, a.H, a.nkv_pad, a.km, a.v16, sm.tile16[tid / UT]);
            return;
        }
        flags += f.ngroups;
        OnceV<D> v;
        v.load(a, t, h, b, tid);
        v.publish(f, bh, t, tid, sm.vred);
        if (tid == 0 && o.raise) agent_store(flags + t, o.tag);
        if (tid < 64) {
            const bool up = flags_up(flags, f.ngroups, o.tag, o.polls, tid);
            if (tid == 0) s_ok = up;
        }
        __syncthreads();
        if (__builtin_expect(s_ok == 0, 0)) {
            help_missing(flags, f.ngroups, t, o.tag, o.raise, tid, s_ok, [&](int g) {
                OnceV<D> x;
                x.load(a, g, h, b, tid);
                x.publish(f, bh, g, tid, sm.vred);
            });
            v.load(a, t, h, b, tid);
        }
        if (tid < D) {
            constexpr int NB = 16;
            const float* p = f.vpart + (int64_t)bh * f.ngroups * D + tid;
            float amax = 0.0f;
            for (int g0 = 0; g0 < f.ngroups; g0 += NB) {
                float x[NB];
#pragma unroll
                for (int j = 0; j < NB; j++) x[j] = agent_load(p + min(g0 + j, f.ngroups - 1) * D);
#pragma unroll
                for (int j = 0; j < NB; j++) amax = fmaxf(amax, x[j]);
            }
            const float sc = amax > 0.0f ? amax / 448.0f : 1.0f;
            if (t == 0) f.vscale[(int64_t)bh * D + tid] = sc;
            hd.mean[tid] = sc;
        }
        __syncthreads();
        const int col = tid % S::CPR8 * 8;
        v.pin();
        const VScale8 vs(&hd.mean[col]);
        const bool plain = vs.plain_for(v.w);
#pragma unroll
        for (int i = 0; i < OnceV<D>::NCH; i++) {
            const int key = i * S::RP + tid / S::CPR8;               // in the group
            uint32_t pk[2];
            vs.codes(v.w[i], plain, pk);
            *reinterpret_cast<u32x2*>(&sm.tile8[key >> 6][v_slot_fp8(key & 63) * (D + 16) + col]) = u32x2{pk[0], pk[1]};
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int tile = t * 4 + j;
            if (tile * 64 < a.nkv_pad) store_v_fp8_tile<D, NT>(tid, sm.tile8[j], a.v8 + ((int64_t)bh * (a.nkv_pad / 64) + tile) * (int64_t)(D * 64));
        }
    } else {
        const int r = unit - o.nk - o.nv - o.nkb;
        if constexpr (PRE == 0) {
            if (unit < o.nk + o.nv + o.nkb) {              // (rows ahead of the wait, as in once_q_block)
                constexpr int NCH = 64 * S::CPR8 / NT;
                const int blk = unit - o.nk - o.nv;
                u32x4 rows[NCH];
                auto load = [&] {
                    const uint16_t* src = a.k.p + b * a.k.sb + h * a.k.sh + tid % S::CPR8 * 8;
#pragma unroll
                    for (int i = 0; i < NCH; i++) rows[i] = *reinterpret_cast<const u32x4*>(src + (int64_t)min(blk * 64 + i * S::RP + tid / S::CPR8, a.Nkv - 1) * a.k.sn);
                };
                load();
                if (!once_k_head<D, PRE>(o, bh, h, b, blk, tid, blk == 0, sm, hd, s_ok)) load();
                quant_i8_block<D, 64, true, PRE, NT, true>(blk, h, b, tid, a.k.p, a.k.sb, a.k.sh, a.k.sn, a.Nkv, a.H, a.nkv_pad, a.km, hd.mean, hd.kmul,
                                                           0.0f, a.k8, a.kscale, nullptr, sm.red, a.pre_k, rows);
                return;
            }
        }
        if (a.blkq == 128) once_q_block<D, PRE, 128>(o, bh, h, b, r, tid, sm, hd, s_ok);
        else if (a.blkq == 64) once_q_block<D, PRE, 64>(o, bh, h, b, r, tid, sm, hd, s_ok);
        else once_q_block<D, PRE, 32>(o, bh, h, b, r, tid, sm, hd, s_ok);
    }
}

// Where the stage is one launch by hand-over: both sides of each line, us a call on one card, by the launches or quant_short_kernel -> by hand-over.
// Up to 32 groups of a head, all of which every workgroup adds up: [1,8192,8,128] 208.1 -> 203.2, e4m3 171.9 -> 164.4.  Past that it still gains, less and
// less ([1,9216,12,128] 392.9 -> 383.7, [1,12288,8,128] 448.5 -> 441.8, 64 channels 315.4 -> 318.6): the line is on the safe side.
// Without the pre-ops, and with e4m3, up to 512 groups in all, which are resident at once: [1,5376,24,128] (504) 273.4 -> 264.8, e4m3 234.4 -> 226.2; e4m3, whose V
// groups are as many again, loses by some numbers past that ([1,5632,24,128] 270.6 -> 283.9, [2,3072,24,128] 195.7 -> 201.8, [2,4416,30,128] 448 -> 489, but
// [2,2176,40,128] 177.8 -> 168.2; with norm + RoPE [1,5184,30,128] 363.1 -> 367.6, [1,9216,30,128] 941 -> 978), fp16 by the most ([2,3072,24,128]
// 216.2 -> 209.2, [2,4416,30,128] (1080) 512.6 -> 518.4).
// Behind the pre-ops the second norm and rotation of K is what it saves: fp16 [1,2304,30,128] 119.0 -> 106.7, [2,4352,30,128] 517.0 -> 495.1, level at the 4096
// groups of [4,8192,32,128] (3223 -> 3227).  But prep_rows_kernel has a group's norms done by four times as many threads, which is shorter for few keys and groups
// of 64 channels: fp16 under four groups of a head ([1,256,40,64] 19.9 -> 20.9, [1,500,40,64] 24.9 -> 25.7; [1,1000,16,64] 26.3 -> 25.7), e4m3 under 72
// in all ([1,256,40,64] 18.5 -> 20.1, [1,500,16,64] 19.6 -> 20.5, [1,1000,16,64] (64) 24.8 level; [1,2304,8,64] (72) 40.1 -> 38.1, [1,500,40,64] (80) 26.0 -> 24.8)
// and, of 128, e4m3 with one group ([1,256,16,128] 22.2 -> 22.5; [1,500,16,128] 25.2 -> 24.5; fp16 [1,256,16,128] 25.3 -> 23.2).
// Of the calls that quant_short_kernel takes (a workgroup there computes its head's statistics itself and waits for nobody), those with fp16 V of two and more
// groups, three at 64 channels, up to 56 groups of 128 channels in all: [1,333,8,128] 18.0 -> 17.3, [1,500,16,128] 20.0 -> 19.3, [1,500,28,128] (56) 24.5 -> 24.4,
// [1,500,30,128] (60) 24.6 -> 24.7; [1,600,8,64] 16.4 -> 14.8, [1,1024,8,64] 16.6 -> 15.9, [1,500,16,64] 14.1 -> 14.0, [1,500,40,64] 19.9 -> 20.2; e4m3 [1,333,8,128]
// 16.1 -> 17.1, [1,500,16,64] 13.9 -> 15.8, though not with many heads ([1,500,40,64] 24.2 -> 21.5, [1,900,30,64] 31.2 -> 25.7), where no line is drawn yet.
bool quant_once_rule(int B, int H, int Nkv, int D, int blkk, int k_flags, bool v_fp8, bool pre, bool full_row, bool short_form) {
    const int ngroups = (Nkv + kGroup - 1) / kGroup;
    const int64_t groups = (int64_t)ngroups * B * H;
    if (pre && (D == 64 ? (v_fp8 ? groups < 72 : ngroups < 4) : v_fp8 && ngroups < 2)) return false;
    if (short_form && (v_fp8 || ngroups < (D == 64 ? 3 : 2) || groups * D > 56 * 128)) return false;
    return D <= 128 && ngroups <= 32 && blkk == 64 && (k_flags & 3) != 0 && !full_row && (pre && !v_fp8 ? groups <= 4096 : groups <= 512);
}

int64_t quant_once_flag_words(int B, int H, int Nkv, bool v_fp8) {
    const int64_t groups = (Nkv + kGroup - 1) / kGroup;
    return (int64_t)B * H * groups * (v_fp8 ? 2 : 1);
}

hipError_t launch_quant_once(const OnceArgs& o_in, int B, int D, hipStream_t st) {
    OnceArgs o = o_in;
    QuantArgs& a = o.q;
    const int pre = pre_kind(a.pre_k);
    const bool v_fp8 = a.v8 != nullptr;
    if (a.k8 == nullptr || (a.v8 == nullptr && a.v16 == nullptr) || a.blkk != 64 || a.pre_k.row_inv != nullptr || o.f.kpart_sum == nullptr ||
        (a.q8 != nullptr && a.nq_pad % a.blkq != 0) || o.flags == nullptr || o.polls <= 0 || pre_kind(a.pre_q) != pre)
        return hipErrorInvalidValue;
    a.n_bh = B * a.H;
    a.nq_blk = a.q8 != nullptr ? (int)(a.nq_pad / a.blkq) : 0;
    o.nk = o.f.ngroups;
    o.nv = v_fp8 ? o.f.ngroups : (int)(a.nkv_pad / 64) / (D == 128 ? 2 : 1);
    o.flag_words = (int)(quant_once_flag_words(1, 1, a.Nkv, v_fp8));
    // K's blocks by workgroups of their own, which start on them when the statistics are there, where the groups leave compute units
    // without one (a group's encoding is 2.6 us in one workgroup, a block's 1); not behind the pre-ops, which they would do
    // again, nor with e4m3, whose V groups are as long.  The call, us, with the groups -> apart: [1,1024,8,64] 19.0 -> 16.9,
    // [2,24 heads,364,128] 55.2 -> 54.2, [2,24,1024,64] 36.4 -> 34.7; but 120 groups of 128 channels, [1,1153,24,128] bias, 49.8 -> 51.5.
    const int64_t groups = (int64_t)o.nk * a.n_bh;
    o.k_apart = !pre && !v_fp8 && groups * D <= 100 * 128;
    o.nkb = o.k_apart ? (int)(a.nkv_pad / 64) : 0;
    // fp16 V by K's workgroups, while the other groups' statistics are on their way, where they take more than one round of the
    // compute units: [2,1248,30,128] 276.9 -> 270.4 (300 groups), norm + RoPE [2,4352,30,128] 516 -> 506 (1020); but
    // [1,8,4224,128] (136) level, [2,24,1024,64] (192) 36.4 -> 39.1.
    o.v_in = !o.k_apart && !v_fp8 && groups > compute_units();
    if (o.v_in) o.nv = 0;
    // (two workgroups to a compute unit are resident together where nothing else runs on the device; elsewhere the bound on the wait counts)
    o.heads = max(1, min(a.n_bh, 2 * compute_units() / (o.nk * (v_fp8 ? 2 : 1))));
    const int64_t total = (int64_t)a.n_bh * (o.nk + o.nv + o.nkb + a.nq_blk);
    if (total <= 0 || total > 0x7FFFFFFF) return hipErrorInvalidValue;
    const dim3 grid((unsigned)total);
#define SAGE_ONCE(DD, PP) hipLaunchKernelGGL((quant_once_kernel<DD, PP>), grid, dim3(OnceShape<DD>::NT), 0, st, o)
    if (D == 128 && pre == 2) SAGE_ONCE(128, 2);
    else if (D == 128 && pre) SAGE_ONCE(128, 1);
    else if (D == 128) SAGE_ONCE(128, 0);
    else if (D == 64 && pre == 2) SAGE_ONCE(64, 2);
    else if (D == 64 && pre) SAGE_ONCE(64, 1);
    else if (D == 64) SAGE_ONCE(64, 0);
    else return hipErrorInvalidValue;
#undef SAGE_ONCE
    return hipGetLastError();
}

int quant_once_helps(int reset) {
    unsigned n = 0;
    hipError_t e = hipMemcpyFromSymbol(&n, HIP_SYMBOL(g_once_helps), sizeof(n));
    if (e == hipSuccess && reset) {
        const unsigned zero = 0;
        e = hipMemcpyToSymbol(HIP_SYMBOL(g_once_helps), &zero, sizeof(zero));
    }
    return e == hipSuccess ? (int)n : -(int)e;
}

}  // namespace sage
