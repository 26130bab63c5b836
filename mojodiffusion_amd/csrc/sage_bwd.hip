// sage_bwd.hip — backward of scaled-dot-product attention in bf16 for gfx950.
//
// Flash-style: no N_q x N_kv matrix is ever stored.  From Q, K, V, O, dO (bf16) and the forward's
// log-sum-exp Stats (fp32) the probabilities are recomputed tile by tile,
//     P = exp(scale * Q K^T - Stats[row]),   Delta[row] = sum_d dO * O,
//     dV = P^T dO,   dS = P * (dO V^T - Delta),   dQ = scale * dS K,   dK = scale * dS^T Q,
// with v_mfma_f32_32x32x16_bf16, fp32 accumulation, P and dS rounded to bf16 as matrix operands.
//
// Two launches:
//   1. bwd_prep_kernel     -Delta and Stats * log2(e) per query row (padding rows: +inf, so their
//                          probabilities vanish); and a vector c close to the mean key.  F32 callers: dO is
//                          rounded here, and launch 2 stores F32, instead of a launch for each of the two casts:
//                          the autograd call, us, [1,2304,12,64] 122.8 -> 115.0, [1,2304,12,128] 222 -> 207,
//                          [2,1248,30,128] 370 -> 338, [1,4608,24,128] 1206 -> 1155.  Same values.
//   2. bwd_fused_kernel    one grid of two kinds of 8-wave workgroups (4-wave at head dim 64), the longer kind first:
//        dQ     owner = 256 (128) query rows, loop over key tiles, as scale * (dS K - rowsum(dS) c)
//               = scale * dS (K - c)                                          (bwd_pass_body<D,0>)
//        dK,dV  owner = 128 keys, loop over query tiles; pairs of waves share 32 keys, one wave
//               carrying P and dV, the other dS and dK                        (bwd_dkdv_body)
//               (head dim 64: every wave both products of 32 keys — bwd_pass_body<D,1>)
// In both kinds a wave owns 32 rows ("x"), keeps their bf16 row blocks resident as B operands
// and walks the other side ("y") in tiles of 64 rows staged in LDS by register-bypassing copies,
// a ring of three slots, one barrier per tile.  A 32x32 block of scores T[y,x] lands in the accumulator
// layout with the owner row as the lane's column, which is exactly the B-operand layout of the
// products that contract over y — so P and dS go from registers straight into the next matrix
// instruction.  Those products' A operands are transposed (rows = head channel, k = y); they come from
// the same row-major tile through the transposing LDS read (ds_read_b64_tr_b16), so every tile is
// fetched once and nothing is rearranged in memory.
//
// What bounds it: a matrix instruction (32 clocks on its SIMD) takes 1 KiB of fragment from LDS (8 clocks of the
// CU's 128 bytes each), and four SIMDs share the LDS — the two run neck and neck, and every byte the
// copies write into LDS comes on top.  With pre-transposed copies of K, Q and dO made by launch 1, as the
// first form had them, each tile was copied twice; owner rows were loaded and results stored as 64 separate
// pieces per instruction.  Measured, one kernel trace of both, us (before -> now):
//   [2,1248,30,128]  launch 1 25.8 -> 9.6, launch 2 231 -> 204 (best 218 -> 185)
//   [1,4608,24,128]  launch 1 31.2 -> 11.7, launch 2 969 -> 864
//   [1,2304,12,64]   launch 1 8.1 -> 4.9, launch 2 75.9 -> 72.5
#include "sage_grid.h"
#include "sage_internal.h"
#include <type_traits>

namespace sage {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef __fp16 v2h __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

namespace {

constexpr float kLog2e = 1.4426950408889634f;

// ---- LDS layouts -------------------------------------------------------------------------
// Tile [64 rows][D] bf16 in 16-byte chunks, CPR per row, the chunk position XORed with a function of the row.
// Two access patterns meet in it:  fragments along the channels (16 consecutive rows, one logical chunk:
// the 16 lanes must land in 16 different 16-byte bank groups), and transposed fragments (4 consecutive rows
// times 4 neighbouring chunks per 32 lanes, 8 bytes each: the 16 chunks must be different ones).  With the
// row's low two bits moved into the chunk's upper bits both are free of conflicts.
template <int CPR> __device__ __forceinline__ int nat_pos(int row, int c) {
    if constexpr (CPR == 16) return c ^ (((row & 3) << 2) | ((row >> 2) & 3));
    else return c ^ ((((row >> 1) & 1) << 2) | ((row >> 2) & 3));       // (row & 1 is the half of the 64 banks)
}
template <int CPR> __device__ __forceinline__ int nat_off(int row, int c) { return (row * CPR + nat_pos<CPR>(row, c)) << 4; }

__device__ __forceinline__ uint32_t lds_addr(const void* p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}
// 16 (4) bytes per lane from global memory straight into LDS: lane l lands at base + 16*l (4*l).
__device__ __forceinline__ void dma16(const void* gbase_uniform, uint32_t goff, uint32_t lds_base_uniform) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(lds_base_uniform), "v"(goff), "s"(gbase_uniform)
                 : "memory");
}
__device__ __forceinline__ void dma4(const void* gbase_uniform, uint32_t goff, uint32_t lds_base_uniform) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
                 :
                 : "s"(lds_base_uniform), "v"(goff), "s"(gbase_uniform)
                 : "memory");
}
// Wait until at most N of this wave's copies are still in flight (they complete in order).
template <int N> __device__ __forceinline__ void dma_wait() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    const v2f f = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, v2bf));       // round to nearest even
}

// Transposed fragment of a tile: lane l gets channel (l & 31) of a 32-channel block, rows half * 4 + 0..3 in
// the first two registers and 8 + half * 4 + 0..3 in the others (half = l >> 5), counted from a 16-row block —
// the order in which an accumulator lane holds its rows, i.e. the A operand that goes with P and dS.
// ds_read_b64_tr_b16 works on 16 lanes: lane i names 8 bytes (row i / 4, channels (i % 4) * 4 .. + 3 of a
// 4 x 16 block) and receives channel i of the four rows.
typedef short v4s __attribute__((ext_vector_type(4)));
template <int CPR> __device__ __forceinline__ int tr_frag_off(int lane, int row0, int d) {
    const int row = row0 + (lane >> 5) * 4 + ((lane & 15) >> 2);
    const int ch = d * 32 + ((lane >> 4) & 1) * 16 + (lane & 3) * 4;
    return nat_off<CPR>(row, ch >> 3) + (ch & 7) * 2;
}
__device__ __forceinline__ v4i tr_read(const uint8_t* lo, const uint8_t* hi) {
    using lds_v4s = __attribute__((address_space(3))) v4s;
    const u32x2 a = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)lo));
    const u32x2 b = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)hi));
    return v4i{(int)a.x, (int)a.y, (int)b.x, (int)b.y};
}

}  // namespace

// ---- the owner rows of a wave, in and out ----------------------------------------------------
// A lane wants its own row's chunks as operands and ends up with pieces of its own row: as plain loads and
// stores these are 64 separate pieces per instruction.  Whole rows move instead, through LDS.
// 32 rows of D bf16 -> LDS at `dst` (64 * D bytes, chunks XORed as in a tile); rows past `last` repeat it.
template <int D>
__device__ __forceinline__ void rows_in(const uint16_t* head, int64_t sn, int row0, int last, uint32_t dst, int lane) {
    constexpr int CPR = D / 8, RPI = 64 / CPR;
#pragma unroll
    for (int i = 0; i < 32 / RPI; i++) {
        const int r = i * RPI + lane / CPR;
        dma16(head, (uint32_t)min(row0 + r, last) * (uint32_t)(sn * 2) + nat_pos<CPR>(r, lane % CPR) * 16,
              __builtin_amdgcn_readfirstlane(dst + i * 1024));
    }
}
// channels ch .. ch + 3 (ch = d * 32 + g * 8 + half * 4) of the lane's row -> LDS
template <int D>
__device__ __forceinline__ void row_put(uint8_t* os, int l32, int half, int d, int g, u32x2 w) {
    *reinterpret_cast<u32x2*>(os + nat_off<D / 8>(l32, d * 4 + g) + half * 8) = w;
}
// ... and from there to the rows below n of the caller's tensor (`at`: elements up to this head), 16 bytes per lane; with
// `f32` the same values as F32, 16 bytes to a lane of 4 channels.
template <int D>
__device__ __forceinline__ void rows_out(const uint8_t* os, uint16_t* p, int64_t at, int64_t sn, int row0, int n, int lane, int f32) {
    constexpr int CPR = D / 8, RPI = 64 / CPR;
    asm volatile("" : "+v"(lane));      // (the row numbers of rows_in are formed again, not kept across the loop in between)
    if (f32) {
        float* op = reinterpret_cast<float*>(p) + at + (lane % (2 * CPR)) * 4;
#pragma unroll
        for (int i = 0; i < 64 / RPI; i++) {
            const int r = i * (RPI / 2) + lane / (2 * CPR);
            const u32x2 w = *reinterpret_cast<const u32x2*>(os + nat_off<CPR>(r, lane % (2 * CPR) >> 1) + (lane & 1) * 8);
            if (row0 + r < n)
                *reinterpret_cast<u32x4*>(op + (int64_t)(row0 + r) * sn) = u32x4{w.x << 16, w.x & 0xFFFF0000u, w.y << 16, w.y & 0xFFFF0000u};
        }
        return;
    }
    uint16_t* op = p + at + (lane % CPR) * 8;
#pragma unroll
    for (int i = 0; i < 32 / RPI; i++) {
        const int r = i * RPI + lane / CPR;
        const u32x4 w = *reinterpret_cast<const u32x4*>(os + nat_off<CPR>(r, lane % CPR));
        if (row0 + r < n) *reinterpret_cast<u32x4*>(op + (int64_t)(row0 + r) * sn) = w;
    }
}

// ---------------------------------------------------------------------------------------------
// Launch 1.  Per (b,h): workgroups with the row statistics of 64 query rows each, and one with the
// mean of 64 keys.
// ---------------------------------------------------------------------------------------------
template <int D>
__global__ __launch_bounds__(256) void bwd_prep_kernel(BwdArgs a) {
    constexpr int CPR = D / 8, RPP = 256 / CPR;     // threads per row, rows per pass of the workgroup
    __shared__ float red[RPP * D];
    const int ntq = (int)(a.nq_pad / 64);
    const int bh = blockIdx.x / (ntq + 1);
    const int r = blockIdx.x % (ntq + 1);
    const int b = bh / a.H, h = bh % a.H;
    const int tid = threadIdx.x;
    const int col = (tid % CPR) * 8;

    if (r < ntq) {
        const uint16_t* po = a.o.p + b * a.o.sb + h * a.o.sh + col;
        const uint16_t* pg = a.dout.p + b * a.dout.sb + h * a.dout.sh + col;
        u32x4 wo[64 / RPP], wg[64 / RPP];
#pragma unroll
        for (int i = 0; i < 64 / RPP; i++) {
            const int64_t row = min(r * 64 + i * RPP + tid / CPR, a.valid_q - 1);
            wo[i] = *reinterpret_cast<const u32x4*>(po + row * a.o.sn);
            if (a.dout32 == nullptr) wg[i] = *reinterpret_cast<const u32x4*>(pg + row * a.dout.sn);
        }
        if (a.dout32 != nullptr) {                  // (the rounded rows also go where launch 2 reads them)
            const float* pf = a.dout32 + b * a.dout.sb + h * a.dout.sh + col;
            v4f f[64 / RPP][2];
#pragma unroll
            for (int i = 0; i < 64 / RPP; i++)
#pragma unroll
                for (int e = 0; e < 2; e++)
                    f[i][e] = *reinterpret_cast<const v4f*>(pf + (int64_t)min(r * 64 + i * RPP + tid / CPR, a.valid_q - 1) * a.dout.sn + e * 4);
#pragma unroll
            for (int i = 0; i < 64 / RPP; i++) {
                wg[i] = u32x4{pack_bf16(f[i][0][0], f[i][0][1]), pack_bf16(f[i][0][2], f[i][0][3]), pack_bf16(f[i][1][0], f[i][1][1]),
                              pack_bf16(f[i][1][2], f[i][1][3])};
                const int row = r * 64 + i * RPP + tid / CPR;
                if (row < a.valid_q) *reinterpret_cast<u32x4*>(const_cast<uint16_t*>(pg) + (int64_t)row * a.dout.sn) = wg[i];
            }
        }
#pragma unroll
        for (int i = 0; i < 64 / RPP; i++) {
            float sum = 0.0f;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                sum = fmaf(__uint_as_float(wo[i][e] << 16), __uint_as_float(wg[i][e] << 16), sum);
                sum = fmaf(__uint_as_float(wo[i][e] & 0xFFFF0000u), __uint_as_float(wg[i][e] & 0xFFFF0000u), sum);
            }
#pragma unroll
            for (int m = 1; m < CPR; m <<= 1) sum += __shfl_xor(sum, m);
            if (tid % CPR == 0) {
                const int row = r * 64 + i * RPP + tid / CPR;
                const int64_t idx = (int64_t)bh * a.nq_pad + row;
                const bool valid = row < a.valid_q;
                a.ndelta[idx] = valid ? -sum : 0.0f;
                a.lse2[idx] = valid ? a.stats[(int64_t)bh * a.Nq + row] * kLog2e : INFINITY;
            }
        }
        return;
    }

    // Rows of dS sum to zero in exact arithmetic, so dS K = dS (K - c) for any vector c; when O and
    // Stats come from a forward of other precision the row sum is small but not zero, and dS K
    // would multiply it by the keys' common offset.  The dQ pass therefore also sums every row of
    // dS (the rounded values the matrix instruction takes) and subtracts rowsum * c at the end,
    // with c close to the mean key: the mean of 64 keys spread evenly over the valid ones, computed
    // here once per head.  (Centring K itself would round K - c to bf16 a second time.)
    const uint16_t* sp = a.k.p + b * a.k.sb + h * a.k.sh + col;
    float part[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 64 / RPP; i++) {
        const int64_t key = ((int64_t)(i * RPP + tid / CPR) * a.valid_kv) >> 6;
        const u32x4 w = *reinterpret_cast<const u32x4*>(sp + key * a.k.sn);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            part[2 * e] += __uint_as_float(w[e] << 16);
            part[2 * e + 1] += __uint_as_float(w[e] & 0xFFFF0000u);
        }
    }
#pragma unroll
    for (int e = 0; e < 8; e++) red[(tid / CPR) * D + col + e] = part[e];
    __syncthreads();
    if (tid < D) {
        float sum = 0.0f;
        for (int g = 0; g < RPP; g++) sum += red[g * D + tid];
        a.kcen[(int64_t)bh * D + tid] = sum * (1.0f / 64.0f);
    }
}

// ---------------------------------------------------------------------------------------------
// Launch 2, the form in which one wave carries every product of its 32 owner rows: the dQ
// workgroups (PASS 0), and the dK/dV workgroups at head dim 64 (PASS 1).
// ---------------------------------------------------------------------------------------------
// Waves per workgroup.  At 64 channels four waves' ring is 50 KiB and two workgroups share a compute unit: the waves of a
// SIMD then meet no common barrier, so that one's matrix instructions run beside the other's exponentials, and a
// grid that does not fill the chip leaves less of it idle.  Both launches, us, eight waves -> four: [2,1248,30,64] 86.5 ->
// 78.2, [1,2304,12,64] 74.4 -> 71.6, [1,4608,24,64] 459 -> 454, [1,700,16,64] 19.6 -> 15.2.  (At 128 channels that form
// takes tiles of 32 rows and twice the copies: 11 % fewer clocks at [2,1248,30,128], which the chip, at its power limit,
// turns into a lower clock: 176.4 us against 174.4.)
template <int D> constexpr int kBwdWaves = D > 64 ? 8 : 4;

template <int D, int PASS>
struct PassLds {
    static constexpr int TILE_BYTES = 64 * D * 2, SLOT = 2 * TILE_BYTES, SLOTS = 3;
    static constexpr int ROW_BYTES = PASS == 1 ? 2048 : 0;                   // [slot][lse | -Delta][64], PASS 1 only
    // The ring, and during the prologue the owner rows (2 x 32 rows per wave) behind its first slot.
    static constexpr int OWNER = ROW_BYTES + SLOT;
    static constexpr int RING_END = ROW_BYTES + SLOTS * SLOT, OWNER_END = OWNER + kBwdWaves<D> * 2 * 64 * D;
    static constexpr int BYTES = RING_END > OWNER_END ? RING_END : OWNER_END;
};

template <int D, int PASS>
__device__ __forceinline__ void bwd_pass_body(const BwdArgs& a, uint8_t* smem, int bh, int xt) {
    using L = PassLds<D, PASS>;
    constexpr int NW = kBwdWaves<D>;
    constexpr int XROWS = NW * 32;                  // owner rows per workgroup
    constexpr int CPR = D / 8;                      // 16-byte chunks per row
    constexpr int TILE_BYTES = L::TILE_BYTES;
    constexpr int RUNS = TILE_BYTES / 1024;         // 1 KiB copies per tile
    constexpr int RPW = RUNS / NW;                  // per wave
    constexpr int KS = D / 16;                      // matrix-instruction steps over the head dim
    constexpr int DB = D / 32;                      // 32-channel output blocks
    constexpr int NTR = PASS == 0 ? 1 : 2;          // transposed operands per tile
    static_assert(RUNS % NW == 0, "tile copies must divide over the waves");

    const int Nx = PASS == 0 ? a.Nq : a.Nkv;
    const int valid_x = PASS == 0 ? a.valid_q : a.valid_kv;
    const int valid_y = PASS == 0 ? a.valid_kv : a.valid_q;
    const int b = bh / a.H, h = bh % a.H;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const int x0 = xt * XROWS + wave * 32;          // this wave's first row
    const int x = x0 + l32;

    // y side
    const View& yv1 = PASS == 0 ? a.k : a.q;
    const View& yv2 = PASS == 0 ? a.v : a.dout;
    const uint8_t* y1 = reinterpret_cast<const uint8_t*>(yv1.p + b * yv1.sb + h * yv1.sh);
    const uint8_t* y2 = reinterpret_cast<const uint8_t*>(yv2.p + b * yv2.sb + h * yv2.sh);
    const uint8_t* rows_l = reinterpret_cast<const uint8_t*>(a.lse2 + (int64_t)bh * a.nq_pad);
    const uint8_t* rows_d = reinterpret_cast<const uint8_t*>(a.ndelta + (int64_t)bh * a.nq_pad);
    // owners that are all padding have nothing to compute: they only store zeros
    const int ntiles = xt * XROWS < valid_x ? (valid_y + 63) / 64 : 0;

    // per-lane pieces of the copy addresses: run i of this wave covers physical chunks
    // (i*NW + wave)*64 + lane of a tile
    int nat_row[RPW], nat_col[RPW];
#pragma unroll
    for (int i = 0; i < RPW; i++) {
        const int P = (i * NW + wave) * 64 + lane;
        nat_row[i] = P / CPR;
        nat_col[i] = nat_pos<CPR>(P / CPR, P % CPR) * 16;          // the XOR is its own inverse
    }
    const uint32_t row_base = lds_addr(smem), nat_base = row_base + L::ROW_BYTES;
    const uint32_t ys1 = (uint32_t)(yv1.sn * 2), ys2 = (uint32_t)(yv2.sn * 2);
    auto copy_tile = [&](int t, int slot) {
        if constexpr (PASS == 1) {                  // (first, so that a wait for the 2 * RPW copies below covers it)
            if (wave == 0) dma4(rows_l + (int64_t)t * 256, lane * 4, __builtin_amdgcn_readfirstlane(row_base + (slot * 2 + 0) * 256));
            if (wave == 1) dma4(rows_d + (int64_t)t * 256, lane * 4, __builtin_amdgcn_readfirstlane(row_base + (slot * 2 + 1) * 256));
        }
#pragma unroll
        for (int i = 0; i < RPW; i++) {
            const uint32_t row = (uint32_t)min(t * 64 + nat_row[i], valid_y - 1);      // padding repeats the last valid row
            const uint32_t dst = (uint32_t)((i * NW + wave) * 1024) + nat_base + slot * L::SLOT;
            dma16(y1, row * ys1 + nat_col[i], __builtin_amdgcn_readfirstlane(dst));
            dma16(y2, row * ys2 + nat_col[i], __builtin_amdgcn_readfirstlane(dst + TILE_BYTES));
        }
    };

    // owner side: two resident row blocks (B operands: column = owner row, k = head channel).
    // (rows past the valid length are never read: what the caller keeps there — NaNs included — must
    // not reach a valid row's gradient through a product with a zero probability)
    const View& xv1 = PASS == 0 ? a.q : a.k;
    const View& xv2 = PASS == 0 ? a.dout : a.v;
    v4i b1[KS], b2[KS];
    const int last_x = max(valid_x, 1) - 1;
    const uint32_t own = L::OWNER + wave * 2 * 64 * D;
    rows_in<D>(xv1.p + b * xv1.sb + h * xv1.sh, xv1.sn, x0, last_x, row_base + own, lane);
    rows_in<D>(xv2.p + b * xv2.sb + h * xv2.sh, xv2.sn, x0, last_x, row_base + own + 64 * D, lane);
    if (ntiles > 0) copy_tile(0, 0);
    float lse_x = 0.0f, ndelta_x = 0.0f;
    float ds_rowsum = 0.0f;                         // dQ pass: sum over the keys of this lane's dS values
    if constexpr (PASS == 0) {
        const int64_t idx = (int64_t)bh * a.nq_pad + min((int64_t)x, a.nq_pad - 1);
        lse_x = a.lse2[idx];
        ndelta_x = a.ndelta[idx];
    }
    // The plain loads above must have landed before the loop: the compiler waits for a load at the
    // first use of its result, and such a wait inside the loop would also wait for the tile copies
    // that are meant to stay in flight (they share the counter).  Using the values here puts the
    // waits here.
    dma_wait<0>();
#pragma unroll
    for (int s = 0; s < KS; s++) {
        b1[s] = *reinterpret_cast<const v4i*>(smem + own + nat_off<CPR>(l32, s * 2 + half));
        b2[s] = *reinterpret_cast<const v4i*>(smem + own + 64 * D + nat_off<CPR>(l32, s * 2 + half));
    }
#pragma unroll
    for (int s = 0; s < KS; s++) asm volatile("" : "+v"(b1[s]), "+v"(b2[s]));
    asm volatile("" : "+v"(lse_x), "+v"(ndelta_x));
    __syncthreads();                     // the owner rows' LDS becomes the ring's second and third slot
    if (ntiles > 1) copy_tile(1, 1);

    // fragment offsets inside a tile
    int nat_frag[KS];                    // [k-step]; 32-row blocks are + 64 * D bytes
#pragma unroll
    for (int s = 0; s < KS; s++) nat_frag[s] = nat_off<CPR>(l32, s * 2 + half);
    int tr_frag[DB][2];                  // [32-channel block][rows 0-7 | 8-15]; 16-row blocks are + 32 * D bytes
#pragma unroll
    for (int d = 0; d < DB; d++) tr_frag[d][0] = tr_frag_off<CPR>(lane, 0, d), tr_frag[d][1] = tr_frag_off<CPR>(lane, 8, d);

    v16f acc1[DB], acc2[PASS == 1 ? DB : 1];
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
            acc1[d][i] = 0.0f;
            if constexpr (PASS == 1) acc2[d][i] = 0.0f;
        }
    const float c = a.scale * kLog2e;
    v16f nd_splat;
    if constexpr (PASS == 0 && D == 64) {
#pragma unroll
        for (int i = 0; i < 16; i++) nd_splat[i] = ndelta_x;
        asm volatile("" : "+v"(nd_splat));          // (16 registers for the whole loop, not 16 copies per use)
    }

    auto tile = [&](auto ragged_tag, int t, int slot) {
        constexpr bool RAGGED = decltype(ragged_tag)::value;             // dQ pass: the tile's last keys are padding
        const uint8_t* n1 = smem + L::ROW_BYTES + slot * L::SLOT;
        const uint8_t* n2 = n1 + TILE_BYTES;
        const uint8_t* rows = smem + slot * 512;
        // Two 32-row blocks per tile, software-pipelined so that the vector work of one block is
        // issued between the matrix instructions of the other:
        //   scores(0) | scores(1) + exponentials(0) | products(0) + exponentials(1) | products(1)
        v16f tacc[2], gacc[2];
        uint32_t pp[2][8], sp[2][8];
        float lse[4];
        // G starts from -Delta wherever that saves the subtraction: read into the accumulators where the rows run
        // along them (PASS 1); in the dQ pass it is one value per lane, whose 16 copies there are registers for
        // at 64 channels only.
        constexpr bool G_FROM_DELTA = PASS == 1 || D == 64;
#pragma unroll
        for (int blk = 0; blk < 2; blk++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                v4f nd = {0.0f, 0.0f, 0.0f, 0.0f};
                if constexpr (PASS == 1) nd = *reinterpret_cast<const v4f*>(rows + 256 + (blk * 32 + g * 8 + half * 4) * 4);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    tacc[blk][g * 4 + e] = 0.0f;
                    gacc[blk][g * 4 + e] = PASS == 1 ? nd[e] : G_FROM_DELTA ? nd_splat[g * 4 + e] : 0.0f;
                }
            }
        // one k-step of the two score products of a block: T += Y1 . X1^T, G += Y2 . X2^T.  The
        // fragments of step ks + 1 are requested before the products of step ks are issued.
        v4i f1[2], f2[2];
        auto scores_load = [&](int blk, int ks) {
            f1[ks & 1] = *reinterpret_cast<const v4i*>(n1 + nat_frag[ks] + blk * 64 * D);
            f2[ks & 1] = *reinterpret_cast<const v4i*>(n2 + nat_frag[ks] + blk * 64 * D);
        };
        auto scores_step = [&](int blk, int ks) {
            if (ks + 1 < KS) scores_load(blk, ks + 1);
            tacc[blk] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, f1[ks & 1]), __builtin_bit_cast(v8bf, b1[ks]), tacc[blk], 0, 0, 0);
            gacc[blk] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, f2[ks & 1]), __builtin_bit_cast(v8bf, b2[ks]), gacc[blk], 0, 0, 0);
        };
        // elements i, i+1 of a block (i even): y rows (i>>2)*8 + half*4 + (i&3) (+1), column = owner row
        auto softmax_pair = [&](int blk, int i) {
            const int g = i >> 2;
            if ((i & 3) == 0) {
                if constexpr (PASS == 0) {
#pragma unroll
                    for (int e = 0; e < 4; e++) lse[e] = lse_x;
                } else {
                    const v4f vl = *reinterpret_cast<const v4f*>(rows + (blk * 32 + g * 8 + half * 4) * 4);
#pragma unroll
                    for (int e = 0; e < 4; e++) lse[e] = vl[e];
                }
            }
            float pr[2], ds[2];
#pragma unroll
            for (int e = 0; e < 2; e++) {
                float arg = fmaf(tacc[blk][i + e], c, -lse[(i & 3) + e]);
                if constexpr (RAGGED) {
                    if (t * 64 + blk * 32 + g * 8 + half * 4 + (i & 3) + e >= valid_y) arg = -INFINITY;
                }
                pr[e] = __builtin_amdgcn_exp2f(arg);
                ds[e] = pr[e] * (G_FROM_DELTA ? gacc[blk][i + e] : gacc[blk][i + e] + ndelta_x);
            }
            sp[blk][i >> 1] = pack_bf16(ds[0], ds[1]);
            // dQ pass: this lane's share of the row sum of dS, over the rounded values
            if constexpr (PASS == 0)
                ds_rowsum = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(v2bf, sp[blk][i >> 1]),
                                                            __builtin_bit_cast(v2bf, 0x3F803F80u), ds_rowsum, false);
            if constexpr (PASS == 1) pp[blk][i >> 1] = pack_bf16(pr[0], pr[1]);
        };
        // matrix instruction m of a block's accumulation: dX1^T += Y1^T . dS  (and dX2^T += Y2^T . P)
        constexpr int ACC_M = 2 * DB * NTR;
        auto acc_step = [&](int blk, int m) {
            const int which = m / (2 * DB), j2 = (m / DB) & 1, d = m % DB;
            const int rows16 = (blk * 2 + j2) * 32 * D;
            if (which == 0) {
                const v4i sb = {(int)sp[blk][j2 * 4], (int)sp[blk][j2 * 4 + 1], (int)sp[blk][j2 * 4 + 2], (int)sp[blk][j2 * 4 + 3]};
                const v4i fa = tr_read(n1 + tr_frag[d][0] + rows16, n1 + tr_frag[d][1] + rows16);
                acc1[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, fa), __builtin_bit_cast(v8bf, sb), acc1[d], 0, 0, 0);
            } else if constexpr (PASS == 1) {
                const v4i pb = {(int)pp[blk][j2 * 4], (int)pp[blk][j2 * 4 + 1], (int)pp[blk][j2 * 4 + 2], (int)pp[blk][j2 * 4 + 3]};
                const v4i fa = tr_read(n2 + tr_frag[d][0] + rows16, n2 + tr_frag[d][1] + rows16);
                acc2[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, fa), __builtin_bit_cast(v8bf, pb), acc2[d], 0, 0, 0);
            }
        };
        // (the further a wave is on its way to the next tile's barrier, the lower its priority: the two waves of a SIMD,
        // which issues from the older one first, arrive there together.  Head dim 64: 1.5 % of launch 2)
        wave_priority(3);
        scores_load(0, 0);
#pragma unroll
        for (int ks = 0; ks < KS; ks++) scores_step(0, ks);
        wave_priority(2);
        // scores of block 1 with the exponentials of block 0: 8 pairs over KS k-steps
        scores_load(1, 0);
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            scores_step(1, ks);
#pragma unroll
            for (int q = 0; q < 8 / KS; q++) softmax_pair(0, (ks * (8 / KS) + q) * 2);
        }
        wave_priority(1);
        // accumulation of block 0 with the exponentials of block 1: 8 pairs over ACC_M instructions
        // (ACC_M is 4, 8 or 16; with 16 a pair goes with every second instruction)
#pragma unroll
        for (int m = 0; m < ACC_M; m++) {
            acc_step(0, m);
            if constexpr (ACC_M <= 8) {
#pragma unroll
                for (int q = 0; q < 8 / ACC_M; q++) softmax_pair(1, (m * (8 / ACC_M) + q) * 2);
            } else {
                if (m & 1) softmax_pair(1, (m >> 1) * 2);
            }
        }
        wave_priority(0);
#pragma unroll
        for (int m = 0; m < ACC_M; m++) acc_step(1, m);
    };

    // Tile t sits in slot t % 3 and was requested two iterations earlier: the wait at the top leaves the
    // copies of tile t + 1 in flight.
    int slot = 0;
    auto next_tile = [&](int t) {
        if (t + 1 < ntiles) dma_wait<2 * RPW>();
        else dma_wait<0>();
        __syncthreads();                 // tile t is visible; every wave is done with the slot of tile t - 1
        if (t + 2 < ntiles) copy_tile(t + 2, slot == 0 ? 2 : slot - 1);
    };
    const int clean = PASS == 0 && (valid_y & 63) && ntiles > 0 ? ntiles - 1 : ntiles;
    for (int t = 0; t < clean; t++) {
        next_tile(t);
        tile(std::false_type{}, t, slot);
        slot = slot == 2 ? 0 : slot + 1;
    }
    if (PASS == 0 && clean < ntiles) {   // (a copy of the loop body: tested per element it was 64 of 273 vector instructions of every tile)
        next_tile(clean);
        tile(std::true_type{}, clean, slot);
        slot = slot == 2 ? 0 : slot + 1;
    }

    // ---- epilogue: rows of valid owners get their gradient, padding rows zeros -----------------
    // `slot` and the one after it have no readers any more (the last tile sits in the one before).
    if (ntiles == 0) __syncthreads();    // (the owner rows of the other waves are still on their way then)
    uint8_t* os = smem + L::ROW_BYTES + (slot + (wave >> 2) >= 3 ? 0 : slot + (wave >> 2)) * L::SLOT + (wave & 3) * 64 * D;
    const bool live = x < valid_x;
    // dQ = scale * (dS K - rowsum(dS) c): the two half-waves hold different keys of the same query
    float rs = 0.0f;
    if constexpr (PASS == 0) {
        const v2u r = __builtin_amdgcn_permlane32_swap(__float_as_uint(ds_rowsum), __float_as_uint(ds_rowsum), false, false);
        rs = __uint_as_float(r.x) + __uint_as_float(r.y);
    }
    const float* cen = a.kcen + (int64_t)bh * D;
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            float y[4];
#pragma unroll
            for (int e = 0; e < 4; e++) y[e] = acc1[d][g * 4 + e];
            if constexpr (PASS == 0) {
                const v4f c4 = *reinterpret_cast<const v4f*>(cen + d * 32 + g * 8 + half * 4);
#pragma unroll
                for (int e = 0; e < 4; e++) y[e] -= rs * c4[e];
            }
            const u32x2 w = {pack_bf16(y[0] * a.scale, y[1] * a.scale), pack_bf16(y[2] * a.scale, y[3] * a.scale)};
            row_put<D>(os, l32, half, d, g, live ? w : u32x2{0u, 0u});
        }
    rows_out<D>(os, PASS == 0 ? a.dq : a.dk, PASS == 0 ? b * a.dq_sb + h * a.dq_sh : b * a.dk_sb + h * a.dk_sh, PASS == 0 ? a.dq_sn : a.dk_sn, x0, Nx,
                lane, a.out32);
    if constexpr (PASS == 1) {
#pragma unroll
        for (int d = 0; d < DB; d++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const u32x2 u = {pack_bf16(acc2[d][g * 4], acc2[d][g * 4 + 1]), pack_bf16(acc2[d][g * 4 + 2], acc2[d][g * 4 + 3])};
                row_put<D>(os, l32, half, d, g, live ? u : u32x2{0u, 0u});
            }
        rows_out<D>(os, a.dv, b * a.dv_sb + h * a.dv_sh, a.dv_sn, x0, Nx, lane, a.out32);
    }
}

// ---------------------------------------------------------------------------------------------
// Launch 2, dK/dV workgroups at head dim 128.  The single-wave form above would keep 128
// accumulator and 64 operand registers per lane and so run one wave per SIMD.  Here a PAIR of waves
// shares 32 keys:
//   the P wave keeps the keys' K rows and the dV accumulators:  T = Q K^T -> P = exp2(cT - lse) -> dV += P^T dO
//   the S wave keeps the keys' V rows and the dK accumulators:  G = dO V^T, dS = P (G - Delta)  -> dK += dS^T Q
// No product is computed twice.  P goes from the P wave
// to the S wave through LDS, in the lane layout of the accumulator, which both waves share — as
// fp16 (11 significant bits, truncated): dS is P times a difference and is itself rounded to bf16,
// and a bf16 P underneath would add a second error of the same size to every term of dK.  The S wave
// runs one query tile behind the P wave, so the hand-over is ordered by the
// workgroup barrier that every tile has anyway: two slots of P, three of tiles (tile t is copied in
// iteration t - 1, read by the P waves in t and by the S waves in t + 1).
// ---------------------------------------------------------------------------------------------
template <int D>
struct DkDvLds {
    static constexpr int TILE_BYTES = 64 * D * 2, SLOT = 2 * TILE_BYTES, SLOTS = 3;
    static constexpr int ROW_BYTES = 2048;          // [slot][lse | -Delta][64]
    static constexpr int P_BYTES = 4 * 2 * 2 * 64 * 16;      // [pair][32-row block][values 0-7 | 8-15][lane], fp16 pairs
    static constexpr int RING = ROW_BYTES + 2 * P_BYTES;
    static constexpr int OWNER = RING + SLOT;       // during the prologue: 32 owner rows per wave
    static constexpr int BYTES = RING + SLOTS * SLOT;
    static_assert(8 * 64 * D <= 2 * SLOT, "the owner rows must fit behind the first slot");
};

template <int D, int ROLE>
__device__ __forceinline__ void dkdv_role(const BwdArgs& a, uint8_t* smem, int bh, int xt, int wave, int lane) {
    using L = DkDvLds<D>;
    constexpr int NW = 8;
    constexpr int CPR = D / 8;
    constexpr int TILE_BYTES = L::TILE_BYTES;
    constexpr int RUNS = TILE_BYTES / 1024;
    constexpr int RPW = RUNS / NW;
    constexpr int KS = D / 16;
    constexpr int DB = D / 32;
    static_assert(RUNS % NW == 0, "tile copies must divide over the waves");
    const int b = bh / a.H, h = bh % a.H;
    const int pair = wave & 3;
    const int l32 = lane & 31, half = lane >> 5;
    const int x0 = xt * 128 + pair * 32, x = x0 + l32;

    const uint8_t* yq = reinterpret_cast<const uint8_t*>(a.q.p + b * a.q.sb + h * a.q.sh);
    const uint8_t* yg = reinterpret_cast<const uint8_t*>(a.dout.p + b * a.dout.sb + h * a.dout.sh);
    const uint8_t* rows_l = reinterpret_cast<const uint8_t*>(a.lse2 + (int64_t)bh * a.nq_pad);
    const uint8_t* rows_d = reinterpret_cast<const uint8_t*>(a.ndelta + (int64_t)bh * a.nq_pad);
    const int ntiles = xt * 128 < a.valid_kv ? (a.valid_q + 63) / 64 : 0;

    int nat_row[RPW], nat_col[RPW];
#pragma unroll
    for (int i = 0; i < RPW; i++) {
        const int P = (i * NW + wave) * 64 + lane;
        nat_row[i] = P / CPR;
        nat_col[i] = nat_pos<CPR>(P / CPR, P % CPR) * 16;
    }
    const uint32_t row_base = lds_addr(smem), nat_base = row_base + L::RING;
    const uint32_t sq = (uint32_t)(a.q.sn * 2), sg = (uint32_t)(a.dout.sn * 2);
    auto copy_tile = [&](int t, int slot) {
#pragma unroll
        for (int i = 0; i < RPW; i++) {
            const uint32_t row = (uint32_t)min(t * 64 + nat_row[i], a.valid_q - 1);
            const uint32_t dst = (uint32_t)((i * NW + wave) * 1024) + nat_base + slot * L::SLOT;
            dma16(yq, row * sq + nat_col[i], __builtin_amdgcn_readfirstlane(dst));
            dma16(yg, row * sg + nat_col[i], __builtin_amdgcn_readfirstlane(dst + TILE_BYTES));
        }
        if (wave == 0) dma4(rows_l + (int64_t)t * 256, lane * 4, __builtin_amdgcn_readfirstlane(row_base + (slot * 2 + 0) * 256));
        if (wave == 1) dma4(rows_d + (int64_t)t * 256, lane * 4, __builtin_amdgcn_readfirstlane(row_base + (slot * 2 + 1) * 256));
    };

    // owner side: the P wave keeps K rows, the S wave V rows (B operands: column = key, k = head channel)
    const View& xv = ROLE == 0 ? a.k : a.v;
    v4i bx[KS];
    const uint32_t own = L::OWNER + wave * 64 * D;
    rows_in<D>(xv.p + b * xv.sb + h * xv.sh, xv.sn, x0, max(a.valid_kv, 1) - 1, row_base + own, lane);
    if (ntiles > 0) copy_tile(0, 0);
    dma_wait<0>();
#pragma unroll
    for (int s = 0; s < KS; s++) bx[s] = *reinterpret_cast<const v4i*>(smem + own + nat_off<CPR>(l32, s * 2 + half));
#pragma unroll
    for (int s = 0; s < KS; s++) asm volatile("" : "+v"(bx[s]));     // the wait for these stays out of the loop

    int nat_frag[KS];
#pragma unroll
    for (int s = 0; s < KS; s++) nat_frag[s] = nat_off<CPR>(l32, s * 2 + half);
    int tr_frag[DB][2];
#pragma unroll
    for (int d = 0; d < DB; d++) tr_frag[d][0] = tr_frag_off<CPR>(lane, 0, d), tr_frag[d][1] = tr_frag_off<CPR>(lane, 8, d);

    v16f acc[DB];
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[d][i] = 0.0f;
    const float c = a.scale * kLog2e;
    // this wave's part of the two hand-over slots
    u32x4* hand = reinterpret_cast<u32x4*>(smem + L::ROW_BYTES) + pair * 256 + lane;

    // iteration `it`: the P wave works on query tile it, the S wave on tile it - 1
    int slot = 0;                        // it % 3
    for (int it = 0; ntiles > 0 && it <= ntiles; it++) {
        dma_wait<0>();
        __syncthreads();                 // this iteration's tile and the previous one's P are visible; the slot of tile it - 2 is free
        const int next = slot == 2 ? 0 : slot + 1;
        const int mine = ROLE == 0 ? slot : slot == 0 ? 2 : slot - 1;
        slot = next;
        if (ROLE == 0 ? it >= ntiles : it == 0) {
            if (it + 1 < ntiles) copy_tile(it + 1, next);
            continue;
        }

        const uint8_t* nt = smem + L::RING + mine * L::SLOT + ROLE * TILE_BYTES;
        const uint8_t* rt = smem + L::RING + mine * L::SLOT + (1 - ROLE) * TILE_BYTES;
        const uint8_t* rowv = smem + (mine * 2 + ROLE) * 256;
        uint32_t hp[2][8];               // S wave: the P wave's probabilities of this tile
        if constexpr (ROLE == 1) {
#pragma unroll
            for (int blk = 0; blk < 2; blk++)
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const u32x4 w = hand[((it - 1) & 1) * (L::P_BYTES / 16) + (blk * 2 + j) * 64];
#pragma unroll
                    for (int e = 0; e < 4; e++) hp[blk][j * 4 + e] = w[e];
                }
        }
        v16f sacc[2];                    // (the S wave's start from -Delta)
        uint32_t pk[2][8];               // P (P wave) or dS (S wave), packed bf16 pairs: the next product's B operand
        uint32_t ph[2][8];               // P wave: the same P as fp16 pairs, for the S wave
        float rv[4];                     // P wave: lse
#pragma unroll
        for (int blk = 0; blk < 2; blk++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                v4f nd = {0.0f, 0.0f, 0.0f, 0.0f};
                if constexpr (ROLE == 1) nd = *reinterpret_cast<const v4f*>(rowv + (blk * 32 + g * 8 + half * 4) * 4);
#pragma unroll
                for (int e = 0; e < 4; e++) sacc[blk][g * 4 + e] = nd[e];
            }
        v4i f[2];
        auto scores_load = [&](int blk, int ks) { f[ks & 1] = *reinterpret_cast<const v4i*>(nt + nat_frag[ks] + blk * 64 * D); };
        auto scores_step = [&](int blk, int ks) {
            if (ks + 1 < KS) scores_load(blk, ks + 1);
            sacc[blk] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, f[ks & 1]), __builtin_bit_cast(v8bf, bx[ks]), sacc[blk], 0, 0, 0);
        };
        // elements i, i+1 of a block (i even): query rows (i>>2)*8 + half*4 + (i&3) (+1), column = key
        auto value_pair = [&](int blk, int i) {
            const int g = i >> 2;
            if (ROLE == 0 && (i & 3) == 0) {
                const v4f vr = *reinterpret_cast<const v4f*>(rowv + (blk * 32 + g * 8 + half * 4) * 4);
#pragma unroll
                for (int e = 0; e < 4; e++) rv[e] = vr[e];
            }
            float y[2];
            if constexpr (ROLE == 0) {
#pragma unroll
                for (int e = 0; e < 2; e++) y[e] = __builtin_amdgcn_exp2f(fmaf(sacc[blk][i + e], c, -rv[(i & 3) + e]));
                ph[blk][i >> 1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(y[0], y[1]));
            } else {
                const v2h w = __builtin_bit_cast(v2h, hp[blk][i >> 1]);
                // (as a multiply-add: one instruction with the fp16 operand's conversion in it)
                y[0] = fmaf((float)w[0], sacc[blk][i], 0.0f);
                y[1] = fmaf((float)w[1], sacc[blk][i + 1], 0.0f);
            }
            pk[blk][i >> 1] = pack_bf16(y[0], y[1]);
        };
        constexpr int ACC_M = 2 * DB;
        auto acc_step = [&](int blk, int m) {
            const int j2 = m / DB, d = m % DB;
            const int rows16 = (blk * 2 + j2) * 32 * D;
            const v4i sb = {(int)pk[blk][j2 * 4], (int)pk[blk][j2 * 4 + 1], (int)pk[blk][j2 * 4 + 2], (int)pk[blk][j2 * 4 + 3]};
            const v4i fa = tr_read(rt + tr_frag[d][0] + rows16, rt + tr_frag[d][1] + rows16);
            acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, fa), __builtin_bit_cast(v8bf, sb), acc[d], 0, 0, 0);
        };
        auto hand_over = [&](int blk) {
            if constexpr (ROLE == 0) {
#pragma unroll
                for (int j = 0; j < 2; j++)
                    hand[(it & 1) * (L::P_BYTES / 16) + (blk * 2 + j) * 64] = u32x4{ph[blk][j * 4], ph[blk][j * 4 + 1], ph[blk][j * 4 + 2], ph[blk][j * 4 + 3]};
            }
        };
        scores_load(0, 0);
#pragma unroll
        for (int ks = 0; ks < KS; ks++) scores_step(0, ks);
        // The next tile's copies: behind the first block's scores, so that the wave's matrix instructions run while it
        // stands at the vector memory path, where all eight waves' copies meet (in front of them the launch took, us:
        // [2,1248,30,128] 185.6, here 181.9; [1,3000,16,128] 268.9, 257.9; behind the second block's scores 184.3, 265.8).
        if (it + 1 < ntiles) copy_tile(it + 1, next);
        scores_load(1, 0);
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            scores_step(1, ks);
#pragma unroll
            for (int q = 0; q < 8 / KS; q++) value_pair(0, (ks * (8 / KS) + q) * 2);
        }
        hand_over(0);
#pragma unroll
        for (int m = 0; m < ACC_M; m++) {
            acc_step(0, m);
#pragma unroll
            for (int q = 0; q < 8 / ACC_M; q++) value_pair(1, (m * (8 / ACC_M) + q) * 2);
        }
        hand_over(1);
#pragma unroll
        for (int m = 0; m < ACC_M; m++) acc_step(1, m);
    }

    // The loop ends with the last tile in the slot two before `slot` (slot = (ntiles + 1) % 3), which the S
    // waves may still be reading; the P waves' output rows go through the one before `slot`, the S waves'
    // through `slot`: their last readers were one barrier ago.
    if (ntiles == 0) __syncthreads();    // (the owner rows of the other waves are still on their way then)
    uint8_t* os = smem + L::RING + (ROLE == 1 ? slot : slot == 0 ? 2 : slot - 1) * L::SLOT + pair * 64 * D;
    const bool live = x < a.valid_kv;
    const float mul = ROLE == 0 ? 1.0f : a.scale;
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const u32x2 w = {pack_bf16(acc[d][g * 4] * mul, acc[d][g * 4 + 1] * mul),
                             pack_bf16(acc[d][g * 4 + 2] * mul, acc[d][g * 4 + 3] * mul)};
            row_put<D>(os, l32, half, d, g, live ? w : u32x2{0u, 0u});
        }
    if constexpr (ROLE == 0) rows_out<D>(os, a.dv, b * a.dv_sb + h * a.dv_sh, a.dv_sn, x0, a.Nkv, lane, a.out32);
    else rows_out<D>(os, a.dk, b * a.dk_sb + h * a.dk_sh, a.dk_sn, x0, a.Nkv, lane, a.out32);
}

template <int D>
__device__ __forceinline__ void bwd_dkdv_body(const BwdArgs& a, uint8_t* smem, int bh, int xt) {
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (wave < 4) dkdv_role<D, 0>(a, smem, bh, xt, wave, lane);
    else dkdv_role<D, 1>(a, smem, bh, xt, wave, lane);
}

// keys of a dK/dV workgroup (wave pairs at 128 channels, every wave 32 keys of its own at 64), rows of a dQ workgroup
constexpr int kKeysWg = 128;
template <int D> constexpr int kRowsWg = kBwdWaves<D> * 32;
static_assert(kBwdWaves<128> * 16 == kKeysWg && kBwdWaves<64> * 32 == kKeysWg, "keys of the waves");

// One grid for both: first the dQ pass (the longer ones first), then the dK/dV pass.  In one grid the second kind starts
// on a CU as soon as the first kind runs out, instead of after its last workgroup.  (Which block a workgroup takes: bwd_block.  Launch 1 + 2, us, blocks in the order of ids -> in ranges
// over the XCDs: [2,1248,30,128] 196.7 -> 191.8, [2,2001,40,64] 310.8 -> 304.6, level where a few heads are all there is.)
template <int D>
__global__ __launch_bounds__(kBwdWaves<D> * 64, 2) void bwd_fused_kernel(BwdArgs a) {
    constexpr bool PAIRED = D > 64;
    constexpr int KV_BYTES = PAIRED ? DkDvLds<D>::BYTES : PassLds<D, 1>::BYTES;
    constexpr int BYTES = KV_BYTES > PassLds<D, 0>::BYTES ? KV_BYTES : PassLds<D, 0>::BYTES;
    __shared__ __attribute__((aligned(1024))) uint8_t smem[BYTES];
    constexpr int RW = kRowsWg<D>, KW = kKeysWg;
    const BwdBlock w = bwd_block((int)blockIdx.x, a.B * a.H, (a.Nq + RW - 1) / RW, (a.valid_q + RW - 1) / RW, (a.Nkv + KW - 1) / KW, (a.valid_kv + KW - 1) / KW);
    if (!w.dkdv) bwd_pass_body<D, 0>(a, smem, w.head, w.tile);
    else if constexpr (PAIRED) bwd_dkdv_body<D>(a, smem, w.head, w.tile);
    else bwd_pass_body<D, 1>(a, smem, w.head, w.tile);
}

template <int D>
static hipError_t launch_bwd_d(const BwdArgs& a, hipStream_t st) {
    const int64_t bh = (int64_t)a.B * a.H;
    const int64_t prep = bh * (a.nq_pad / 64 + 1);
    const int64_t gq = bh * ((a.Nq + kRowsWg<D> - 1) / kRowsWg<D>), gk = bh * ((a.Nkv + kKeysWg - 1) / kKeysWg);
    if (prep > 0x7FFFFFFF || gq + gk > 0x7FFFFFFF) return hipErrorInvalidValue;
    hipLaunchKernelGGL((bwd_prep_kernel<D>), dim3((unsigned)prep), dim3(256), 0, st, a);
    hipLaunchKernelGGL((bwd_fused_kernel<D>), dim3((unsigned)(gq + gk)), dim3(kBwdWaves<D> * 64), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_bwd(const BwdArgs& a, hipStream_t st) {
    if (a.D == 128) return launch_bwd_d<128>(a, st);
    if (a.D == 64) return launch_bwd_d<64>(a, st);
    return hipErrorInvalidValue;
}

}  // namespace sage
