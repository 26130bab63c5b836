// sage_attn_short.hip — attention on quantized operands for problems too small to fill the chip with
// 256-row workgroups (gfx950).
//
// The main kernel (sage_attn.hip) gives a workgroup 256 query rows and all keys.  At a few hundred
// tokens that is a few dozen workgroups on 256 compute units, each walking every key tile in turn.
// Here a workgroup owns 32 or 64 query rows and its waves split the KEYS: wave (r, w) computes rows
// 32 r .. 32 r + 31 against the w-th of KW equal runs of key steps, and the KW partial results (row
// maximum, row sum, unnormalised output) meet in LDS at the end — the same online-softmax merge a wave
// does from step to step, done once across waves.  The matrix layouts are the main kernel's:
// S^T = K . Q^T, O^T = V^T . P^T, probabilities straight from the score accumulators.
//
// No wave shares a key with another, so every wave keeps one step's K and V^T in an LDS region of its own,
// filled by register-bypassing copies (contiguous runs, swizzled on the source side like the main kernel's
// tiles): K of the next step as soon as the scores have read theirs, V^T once P.V has.  The waits are the
// wave's own copy counters; the loop has no barrier.  (Fragments loaded from L2 straight into registers —
// no LDS at all — were built first: a fragment is 64 separate 16-byte pieces, an address cycle each, and
// the first step alone took 6.4 us at [1,256,30,128].)  Per key tile a compute unit moves 8 times the main
// kernel's operand bytes per query row, which is why the choice of form (below) leaves it where the main kernel's
// workgroups start to fill the chip.
#include "sage_attn_common.h"
#include "sage_grid.h"
#include "sage_quant_common.h"

#include <algorithm>
#include <atomic>

namespace sage {

static std::atomic<int> g_short_mode{0};       // see attn_short_override
template <int D> constexpr int kMainRows = D > 128 ? 128 : 256;               // rows per workgroup of the main kernel
template <int D> constexpr int short_waves() { return D > 128 ? 4 : 8; }      // 256 channels: a wave needs a SIMD's registers

// ---- the whole call in one launch -----------------------------------------------------------------
// At 256 keys (512 of 64 channels) the quantizers' launch and this one last 7 to 9 us each, of which 2.5 are its start and
// end, the rest latencies of loads and barriers and a chain of little work per wave.  Here every workgroup quantizes
// its head's keys and values for itself, into LDS, where the form above keeps the pieces its waves copy in: the
// statistics by the same leaves, groups and order, the codes by the same arithmetic, so the same bits.  All eight waves
// share either: K as sixteen tokens of four channels to a thread, which holds them from the sums to the codes; V as four neighbouring
// keys of eight channels to a thread, one write per channel in the slots' order.  (K by four of the waves and V by the
// others was 14.3 us at [1,256,30,128], 13.4 so.)  One-shot, two launches -> one, us: [1,256,30,128] 16.5 -> 13.4, [1,64,4,128]
// 13.9 -> 11.2, [1,512,8,64] 13.7 -> 12.7, with Stats [1,256,30,128] 19.0 -> 13.6, with a bias 17.6 -> 14.0.
// (fp16 P.V only: with the e4m3 maxima and quotients in it the same was 16.0 us against 14.8 in two launches.)
template <int D> struct FuseLds {
    static constexpr int KEYS = fused_keys(D), CPR = D / 8, LD = D + CPR;
    static constexpr int K8 = KEYS * D, V = KEYS * D * 2;
    static constexpr int LEAVES = KEYS / 16, LEAF = K8 + V, LEAF_BYTES = LEAVES * LD * 16;       // sums (double), minima, maxima
    static constexpr int BYTES = LEAF + LEAF_BYTES;
    static_assert(LEAVES * (D / 4) == 512 && KEYS / 4 * CPR == 2 * 512, "K: a leaf of four channels to a thread; V: two quads of keys");
};
template <int D> struct FuseStats { float mean[D], kmul[D], qmul[D], ks[fused_keys(D) / 64], kmax[8]; };

template <int D>
struct FuseQuant {
    using L = FuseLds<D>;
    static constexpr int CPR = L::CPR, LD = L::LD, WL = D == 128 ? 2 : 1;      // waves that share four leaves (one scale block)
    float v[kLeaf][4];                                  // the K values of this thread's leaf
    bool live;                                          // (waves whose 64 tokens are past the end only leave empty leaves: no step reads their codes)
    // this thread's leaf and first of four channels (K); first quad of keys and first of eight channels (V)
    __device__ static __forceinline__ int leaf(int tid) { return (tid >> 6) / WL * 4 + ((tid & 63) >> 4); }
    __device__ static __forceinline__ int kcol(int tid) { return ((tid >> 6) % WL * 16 + (tid & 15)) * 4; }
    __device__ static __forceinline__ int quad(int tid, int i) { return tid / CPR + i * (512 / CPR); }
    __device__ static __forceinline__ int vcol(int tid) { return tid % CPR * 8; }

    // Statistics, V^T, K values and their largest per wave.  (Meets two barriers.)
    __device__ __forceinline__ void values(const FuseArgs& f, int b, int h, int N, const KeyMask& km, int tid, uint8_t* raw, FuseStats<D>& st) {
        double* leafsum = reinterpret_cast<double*>(raw + L::LEAF);
        float* leafmin = reinterpret_cast<float*>(raw + L::LEAF + L::LEAVES * LD * 8);
        float* leafmax = leafmin + L::LEAVES * LD;
        const int s0 = leaf(tid) * kLeaf, c4 = kcol(tid), c8 = vcol(tid);
        // (every token of the wave's leaves counts: the common case)
        live = __any(s0 < N);
        const bool all_kept = __all(s0 + kLeaf <= N && !(s0 < km.hi && s0 + kLeaf > km.lo));
        u32x2 w[kLeaf];
        u32x4 wv[2][4];                                 // [item][key of the quad]
        {
            // (tokens past the end repeat the last; what does not count becomes zero)
            const uint16_t* src = f.k.p + b * f.k.sb + h * f.k.sh + c4;
#pragma unroll
            for (int i = 0; i < kLeaf; i++) w[i] = *reinterpret_cast<const u32x2*>(src + (int64_t)min(s0 + i, N - 1) * f.k.sn);
            const uint16_t* vsrc = f.v.p + b * f.v.sb + h * f.v.sh + c8;
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int r = 0; r < 4; r++) wv[i][r] = *reinterpret_cast<const u32x4*>(vsrc + (int64_t)min(quad(tid, i) * 4 + r, N - 1) * f.v.sn);
            if (!all_kept) {
#pragma unroll
                for (int i = 0; i < kLeaf; i++)
                    if (!key_kept(s0 + i, N, km)) w[i] = u32x2{0u, 0u};
            }
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (!key_kept(quad(tid, i) * 4 + r, N, km)) wv[i][r] = u32x4{0u, 0u, 0u, 0u};
        }
        double acc[4] = {0, 0, 0, 0};
        float mn[4], mx[4];
#pragma unroll
        for (int e = 0; e < 4; e++) { mn[e] = INFINITY; mx[e] = -INFINITY; }
        if (live) {
#pragma unroll
        for (int i = 0; i < kLeaf; i++) {
            v[i][0] = bf16_lo(w[i].x); v[i][1] = bf16_hi(w[i].x);
            v[i][2] = bf16_lo(w[i].y); v[i][3] = bf16_hi(w[i].y);
#pragma unroll
            for (int e = 0; e < 4; e++) acc[e] += (double)v[i][e];           // (tokens that do not count are +0.0)
        }
#pragma unroll
        for (int i = 0; i < kLeaf; i += 2) {
            float x[2][4];
#pragma unroll
            for (int r = 0; r < 2; r++)
#pragma unroll
                for (int e = 0; e < 4; e++) x[r][e] = v[i + r][e];
            if (!all_kept) {
                // (a NaN takes no part in a minimum or maximum)
#pragma unroll
                for (int r = 0; r < 2; r++)
                    if (!key_kept(s0 + i + r, N, km))
#pragma unroll
                        for (int e = 0; e < 4; e++) x[r][e] = __builtin_nanf("");
            }
            // (as instructions: fminf and fmaxf of values out of bit operations are several each, see kstats_group)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                asm("v_min3_f32 %0, %0, %1, %2" : "+v"(mn[e]) : "v"(x[0][e]), "v"(x[1][e]));
                asm("v_max3_f32 %0, %0, %1, %2" : "+v"(mx[e]) : "v"(x[0][e]), "v"(x[1][e]));
            }
        }
        }
#pragma unroll
        for (int e = 0; e < 4; e++) {
            // (channel 8 c + e at e * D/8 + c, as in KGroupSmem)
            const int at = leaf(tid) * LD + ((c4 + e) & 7) * CPR + (c4 >> 3);
            leafsum[at] = acc[e];
            leafmin[at] = mn[e];
            leafmax[at] = mx[e];
        }
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int key = quad(tid, i) * 4, slot = v_slot_f16(key & 31);
            if (!__any((key & ~31) < N)) continue;      // (no step reads it)
            uint8_t* step = raw + L::K8 + (key >> 5) * (D * 64);
            float x[4][8];
#pragma unroll
            for (int r = 0; r < 4; r++) unpack8(wv[i][r], x[r]);
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const u32x2 o = {f16_pair_sat(x[0][e], x[1][e]), f16_pair_sat(x[2][e], x[3][e])};
                *reinterpret_cast<u32x2*>(step + swz((c8 + e) * 4 + (slot >> 3)) + (slot & 7) * 2) = o;
            }
        }
        __syncthreads();
        if (tid < D) {
            double sum = 0.0;
            float lo = INFINITY, hi = -INFINITY;
            for (int g = 0; g * kGroup < N; g++) {
                double gsum = 0.0;
#pragma unroll
                for (int u = 0; u < 16; u++) {
                    gsum += leafsum[(g * 16 + u) * LD + tid];
                    lo = fminf(lo, leafmin[(g * 16 + u) * LD + tid]);
                    hi = fmaxf(hi, leafmax[(g * 16 + u) * LD + tid]);
                }
                sum += gsum;
            }
            float mean, sd;
            k_final(sum, lo, hi, f.kept, f.flags, mean, sd);
            const int d = leaf_channel<D>(tid);
            st.mean[d] = mean; st.kmul[d] = 1.0f / sd; st.qmul[d] = f.cmul * sd;
        }
        __syncthreads();
        if (!live) return;
        const v4f mu = *reinterpret_cast<const v4f*>(&st.mean[c4]), mul = *reinterpret_cast<const v4f*>(&st.kmul[c4]);
        float am = 0.0f;
#pragma unroll
        for (int i = 0; i < kLeaf; i++) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float d = v[i][e] - mu[e];
                v[i][e] = d * mul[e];
            }
            if (!all_kept && !key_kept(s0 + i, N, km)) {
#pragma unroll
                for (int e = 0; e < 4; e++) v[i][e] = 0.0f;
            }
#pragma unroll
            for (int e = 0; e < 4; e += 2) am = fmaxf(fmaxf(am, fabsf(v[i][e])), fabsf(v[i][e + 1]));
        }
        am = wave_max(am);
        if ((tid & 63) == 0) st.kmax[tid >> 6] = am;
    }

    // Codes and scales.  (Behind a barrier that publishes kmax; another one publishes them.)
    __device__ __forceinline__ void codes(int tid, uint8_t* raw, FuseStats<D>& st) {
        if (!live) return;
        const int s0 = leaf(tid) * kLeaf, c4 = kcol(tid), wave = tid >> 6;
        float am = st.kmax[wave];
        if constexpr (WL == 2) am = fmaxf(am, st.kmax[wave ^ 1]);
        const float sc = am > 0.0f ? am / 127.0f : 1.0f;
        if ((tid & (64 * WL - 1)) == 0) st.ks[s0 >> 6] = sc;
        const bool fast = sc >= 0x1p-100f && sc <= 0x1p100f;
        const float rinv = 1.0f / sc;
#pragma unroll
        for (int i = 0; i < kLeaf; i += 2) {
            // (two tokens of four channels as one encoder call of eight values)
            const float x[8] = {v[i][0], v[i][1], v[i][2], v[i][3], v[i + 1][0], v[i + 1][1], v[i + 1][2], v[i + 1][3]};
            const u32x2 o = encode8_i8(x, sc, rinv, fast);
#pragma unroll
            for (int r = 0; r < 2; r++) {
                const int key = s0 + i + r;
                *reinterpret_cast<uint32_t*>(raw + (key >> 5) * (32 * D) + swz((key & 31) * (D / 16) + (c4 >> 4)) + (c4 & 15)) = r ? o.y : o.x;
            }
        }
    }
};

// FUSE: K and V are quantized here (fz), the fields of `a` that name their codes, scales and multipliers are not read.
template <int D, int VARIANT, int KW, bool QF, bool ADDMASK, bool FUSE>
__device__ __forceinline__ void short_body(const AttnArgs& a, const FuseArgs& fz, int n_rtiles, int item0, int total_wg) {
    constexpr int NW = short_waves<D>();
    static_assert(!FUSE || (QF && D <= 128 && VARIANT == 0), "one launch: Q is encoded here too");
    constexpr int R = NW / KW;                          // 32-row blocks per workgroup
    constexpr int ROWS = 32 * R;
    constexpr int KSTEPS = D / 32, DB = D / 32, CPR = D / 8;
    constexpr int VB = VARIANT == 0 ? 2 : 1;
    constexpr int SK = VARIANT == 0 ? 32 : 64;          // keys per step (what the P.V matrix instruction divides into)
    constexpr int SKB = SK / 32;
    constexpr int NK = KSTEPS * SKB;                    // K fragments per step
    constexpr int NV = 2 * DB;                          // V^T fragments of 16 bytes per step
    constexpr int K_BYTES = SK * D, V_BYTES = D * 64;   // one step's K and V^T
    constexpr int KC = K_BYTES / 1024, VC = V_BYTES / 1024;      // 1 KiB copies of either
    constexpr int NP = 8 * SKB;                         // pairs of scores per lane and step
    constexpr int LD = D + 4;                           // floats per row of the exchange buffer (keeps 16-byte alignment, spreads banks)
    static_assert(NW % KW == 0 && ROWS <= 128, "waves = row blocks x key runs");

    struct Ring { uint8_t k[K_BYTES], v[V_BYTES], bias[ADDMASK ? BiasStage::BYTES : 16]; };
    // A wave's loop operands, then its partial output for the merge, in the same place: a wave that is done with its
    // keys leaves its output without waiting for the others.
    union Mem {
        Ring ring;
        float acc[32 * LD];
        uint8_t stride[((sizeof(Ring) > 32 * LD * 4 ? sizeof(Ring) : 32 * LD * 4) + 255) / 256 * 256];
    };
    using L = FuseLds<FUSE ? D : 128>;
    constexpr int ACC_BYTES = NW * 32 * LD * 4, RAW = L::BYTES > ACC_BYTES ? L::BYTES : ACC_BYTES;
    __shared__ __attribute__((aligned(1024))) Mem mem[FUSE ? 1 : NW];
    __shared__ __attribute__((aligned(1024))) uint8_t raw[FUSE ? RAW : 16];         // FUSE: K, V^T and the statistics' leaves, then the partial outputs
    __shared__ __attribute__((aligned(16))) FuseStats<FUSE ? D : 64> fstat;
    __shared__ float lds_shift[FUSE ? ROWS : 1];
    auto acc_of = [&](int w) -> float* { return FUSE ? reinterpret_cast<float*>(raw) + w * (32 * LD) : mem[FUSE ? 0 : w].acc; };
    __shared__ __attribute__((aligned(16))) uint8_t lds_q[QF ? ROWS * D : 16];      // this workgroup's Q codes
    __shared__ float lds_m[NW][32], lds_l[NW][32];
    __shared__ __attribute__((aligned(16))) float lds_qmax[8];

    // each XCD takes a contiguous range of workgroups, so that those sharing a head share its L2
    const int wg = xcd_item((int)blockIdx.x, total_wg);
    // item0 > 0: the main kernel has done the items (row tiles of kMainRows) below it; n_rtiles counts those
    // tiles then, and consecutive workgroups take the pieces of one
    constexpr int PIECES = kMainRows<D> / ROWS;
    const int item = item0 > 0 ? item0 + wg / PIECES : wg;
    const int rt = item0 > 0 ? item % n_rtiles * PIECES + wg % PIECES : item % n_rtiles, bh = item / n_rtiles;
    if (rt * ROWS >= a.Nq) return;                      // a piece behind the last row
    const int b = bh / a.H, h = bh % a.H;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const int kw = wave % KW, rg = wave / KW;
    const int wg_row0 = rt * ROWS, row0 = wg_row0 + rg * 32, qrow = row0 + l32;

    // causal: keys past the workgroup's last row count as the ragged end
    const int kv_valid = a.causal ? min(a.kv_valid, wg_row0 + ROWS) : a.kv_valid;
    // (steps that lie in the masked range as a whole are left out: step h stands for keys h * SK .., or those
    // `skip` steps further on from skip_at on)
    int skip_at = 0, skip = 0;
    if (!a.causal && a.km.hi > a.km.lo) {
        skip_at = (a.km.lo + SK - 1) / SK;
        skip = max(min(a.km.hi, kv_valid) / SK - skip_at, 0);
    }
    auto key_step = [&](int h) -> int { return h < skip_at ? h : h + skip; };
    const int nsteps = (kv_valid + SK - 1) / SK - skip;
    const int h0 = nsteps * kw / KW, h1 = nsteps * (kw + 1) / KW;

    // ---- one step's operands: copies into the wave's own LDS region, fragments out of it
    const uint8_t* kg = reinterpret_cast<const uint8_t*>(a.k8) + (int64_t)bh * a.nkv_pad * D;
    const uint8_t* vg = static_cast<const uint8_t*>(a.vq) + (int64_t)bh * a.nkv_pad * D * VB;
    const uint32_t k_lds = FUSE ? lds_addr(&raw[0]) : lds_addr(&mem[FUSE ? 0 : wave].ring.k[0]);
    const uint32_t v_lds = FUSE ? lds_addr(&raw[L::K8]) : lds_addr(&mem[FUSE ? 0 : wave].ring.v[0]);
    int vsrc[VC];
#pragma unroll
    for (int i = 0; i < VC; i++) {
        // (fp16: a step is half of a 64-key tile, 64 bytes of every 128-byte channel row)
        const int L = swz(i * 64 + lane);
        vsrc[i] = VARIANT == 0 ? (L >> 6) * 128 + (L & 63) : L;
    }
    auto copy_k = [&](int h) {
        const int hs = key_step(h);
        const uint8_t* g = kg + (int64_t)hs * K_BYTES;
#pragma unroll
        for (int i = 0; i < KC; i++) dma16(g, swz(i * 64 + lane), __builtin_amdgcn_readfirstlane(k_lds + i * 1024));
    };
    auto copy_v = [&](int h) {
        const int hs = key_step(h);
        const uint8_t* g = VARIANT == 0 ? vg + (int64_t)(hs >> 1) * (D * 128) + (hs & 1) * 64 : vg + (int64_t)hs * V_BYTES;
#pragma unroll
        for (int i = 0; i < VC; i++) dma16(g, vsrc[i], __builtin_amdgcn_readfirstlane(v_lds + i * 1024));
    };
    typedef const __attribute__((address_space(3))) v4i* lds_v4i_ptr;
    auto k_frag = [&](int n, int hs) -> v4i {
        return *reinterpret_cast<lds_v4i_ptr>(k_lds + (FUSE ? key_step(hs) * K_BYTES : 0) + swz(((n / KSTEPS) * 32 + l32) * (D / 16) + (n % KSTEPS) * 2 + half));
    };
    // fp16: fragment jj * DB + d = 16 keys, channels 32 d ..; e4m3: fragments 2 d, 2 d + 1 = a lane's 32 keys, channels 32 d ..
    auto v_frag = [&](int n, int hs) -> v4i {
        const int d = VARIANT == 0 ? n % DB : n >> 1;
        const int c = VARIANT == 0 ? (n / DB) * 2 + half : half * 2 + (n & 1);
        return *reinterpret_cast<lds_v4i_ptr>(v_lds + (FUSE ? key_step(hs) * V_BYTES : 0) + swz((d * 32 + l32) * 4 + c));
    };
    // (LDS reads issued before this have delivered: what they read may be overwritten)
    auto reads_done = [] { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };
    auto first_copies = [&] {
        if (!FUSE && h0 < h1) {
            copy_k(h0);
            copy_v(h0);
        }
    };

    // ---- Q^T fragments of the wave's 32 rows
    v4i qf[KSTEPS];
    float sq;
    if constexpr (!QF) {
        const int8_t* qp = a.q8 + ((int64_t)bh * a.nq_pad + qrow) * D + half * 16;
#pragma unroll
        for (int s = 0; s < KSTEPS; s++) qf[s] = *reinterpret_cast<const v4i*>(qp + s * 32);
        sq = a.qscale[(int64_t)bh * (a.nq_pad / a.blkq) + qrow / a.blkq] * kMagicUnit;
        first_copies();
    } else {
        // Q arrives as bf16: the quantizer's arithmetic, so its codes and scales.  A scale block is wider
        // than the workgroup's rows as a rule: the waves take the maxima of the whole block, 16 rows at a
        // time, and then all of them encode this workgroup's rows into LDS, a chunk or two of eight channels per
        // thread.  (By the waves that had taken those rows' maxima, two of eight, it took 0.7 us instead of 0.2.)
        const uint16_t* qb = a.q_src + b * a.qsb + h * a.qsh;
        const int cover = a.blkq > ROWS ? a.blkq : ROWS;                 // 32 .. 128 rows: the scale blocks of this workgroup
        const int cover0 = wg_row0 / cover * cover;
        constexpr int RPI = 64 / CPR;                                    // rows per load instruction
        constexpr int NI = 16 / RPI;
        constexpr int TURNS = 8 / NW;                                    // 16-row pieces of the largest block per wave
        const int col = (lane % CPR) * 8, rr = lane / CPR;
        u32x4 w[TURNS][NI];
#pragma unroll
        for (int t = 0; t < TURNS; t++)
#pragma unroll
            for (int i = 0; i < NI; i++) {
                const int piece = t * NW + wave, row = cover0 + piece * 16 + i * RPI + rr;
                w[t][i] = u32x4{0u, 0u, 0u, 0u};
                if (piece < cover / 16 && row < a.Nq) w[t][i] = *reinterpret_cast<const u32x4*>(qb + (int64_t)row * a.qsn + col);
            }
        constexpr int OWN = (ROWS * CPR + NW * 64 - 1) / (NW * 64);      // this thread's chunks of the workgroup's rows
        static_assert(ROWS * CPR % 64 == 0 && (NW * 64) % CPR == 0, "whole waves of chunks, one column per thread");
        u32x4 own[OWN];
#pragma unroll
        for (int i = 0; i < OWN; i++) {
            const int row = wg_row0 + i * (NW * 64 / CPR) + tid / CPR;
            own[i] = u32x4{0u, 0u, 0u, 0u};
            if (row < a.Nq) own[i] = *reinterpret_cast<const u32x4*>(qb + (int64_t)row * a.qsn + col);
        }
        FuseQuant<FUSE ? D : 128> fq;
        if constexpr (FUSE) fq.values(fz, b, h, a.kv_valid, a.km, tid, raw, fstat);
        float m[8];
        {
            const float* mp = FUSE ? &fstat.qmul[col] : a.qmul + (int64_t)bh * D + col;
            const v4f m0 = *reinterpret_cast<const v4f*>(mp), m1 = *reinterpret_cast<const v4f*>(mp + 4);
#pragma unroll
            for (int e = 0; e < 4; e++) m[e] = m0[e], m[4 + e] = m1[e];
        }
        first_copies();
#pragma unroll
        for (int t = 0; t < TURNS; t++) {
            float am = 0.0f;
#pragma unroll
            for (int i = 0; i < NI; i++)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    am = fmaxf(fmaxf(am, fabsf(__uint_as_float(w[t][i][e] << 16) * m[2 * e])), fabsf(__uint_as_float(w[t][i][e] & 0xFFFF0000u) * m[2 * e + 1]));
            am = wave_max(am);
            if (lane == 0) lds_qmax[t * NW + wave] = am;
        }
        __syncthreads();
        if constexpr (FUSE) fq.codes(tid, raw, fstat);
        // (all eight maxima in two reads and the block's picked: as a loop over them, one after the other, this was half a
        // microsecond each time it was asked)
        const int blk16 = a.blkq >> 4, blksh = a.blkq == 32 ? 5 : a.blkq == 64 ? 6 : 7;
        const v4f qm0 = *reinterpret_cast<const v4f*>(&lds_qmax[0]), qm1 = *reinterpret_cast<const v4f*>(&lds_qmax[4]);
        auto block_scale = [&](int row) {                                // of the scale block that holds `row`
            const int s0 = ((row - cover0) >> blksh) * blk16;
            float am = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; i++) am = i >= s0 && i < s0 + blk16 ? fmaxf(am, i < 4 ? qm0[i & 3] : qm1[i & 3]) : am;
            return am > 0.0f ? am / 127.0f : 1.0f;
        };
        sq = block_scale(row0) * kMagicUnit;
#pragma unroll
        for (int i = 0; i < OWN; i++) {
            // (a wave's rows lie in one scale block: it holds 2 to 8 of them, from a multiple of that on)
            const int row = i * (NW * 64 / CPR) + tid / CPR;
            if (ROWS * CPR < NW * 64 && row >= ROWS) break;
            const float sc = block_scale(wg_row0 + row);
            const bool fast = sc >= 0x1p-100f && sc <= 0x1p100f;
            const float rinv = 1.0f / sc;
            float x[8];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                x[2 * e] = __uint_as_float(own[i][e] << 16) * m[2 * e];
                x[2 * e + 1] = __uint_as_float(own[i][e] & 0xFFFF0000u) * m[2 * e + 1];
            }
            *reinterpret_cast<u32x2*>(&lds_q[row * D + col]) = encode8_i8(x, sc, rinv, fast);
            if (FUSE && a.stats != nullptr) {
                // <pre-scaled query row, K mean>, as the Q encoder takes it: what K smoothing lowers the row's scores by
                float dot = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const float q = e & 1 ? __uint_as_float(own[i][e >> 1] & 0xFFFF0000u) : __uint_as_float(own[i][e >> 1] << 16);
                    dot += (q * fz.cmul) * fstat.mean[col + e];
                }
#pragma unroll
                for (int off = CPR / 2; off > 0; off >>= 1) dot += __shfl_xor(dot, off, 64);
                if (tid % CPR == 0) lds_shift[row] = dot;
            }
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < KSTEPS; s++) qf[s] = *reinterpret_cast<const v4i*>(&lds_q[(rg * 32 + l32) * D + s * 32 + half * 16]);
    }

    const float* ksc = FUSE ? &fstat.ks[0] : a.kscale + (int64_t)bh * (a.nkv_pad / a.blkk);
    const int ksh = a.blkk == 32 ? 5 : a.blkk == 64 ? 6 : 7;
    // the bias of a step is loaded while the step before it runs
    BiasStage bias[SKB];
    uint8_t* bias_lds = FUSE ? &raw[L::LEAF + (ADDMASK ? wave * BiasStage::BYTES : 0)] : &mem[FUSE ? 0 : wave].ring.bias[0];
    static_assert(!FUSE || NW * BiasStage::BYTES <= L::LEAF_BYTES, "the bias takes the leaves' place");
    BiasStage::Rows brows{};
    if (ADDMASK) brows = BiasStage::rows(a.amask + b * a.amb + h * a.amh, a.amn, row0, a.Nq - 1, lane);
    auto bias_load = [&](int hs) {
        BiasStage::Rows rows = brows;
        if constexpr (D == 64 && VARIANT == 0) {
            // (one pointer of the two is formed for each step, behind an empty statement: both, kept over the loop, are one
            // register too many)
            int first = row0;
            asm volatile("" : "+s"(first));
            rows.p[1] = BiasStage::rows(a.amask + b * a.amb + h * a.amh, a.amn, first, a.Nq - 1, lane).p[1];
        }
#pragma unroll
        for (int kb = 0; kb < SKB; kb++)
            bias[kb].load(rows, key_step(min(hs, h1 - 1)) * SK + kb * 32, kv_valid, lane);
    };
    if (ADDMASK && h0 < h1) bias_load(h0);

    v16f oacc[DB], lacc;
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
        for (int i = 0; i < 16; i++) oacc[d][i] = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; i++) lacc[i] = 0.0f;
    float m_used = -3.0e38f, l_run = 0.0f;              // (finite: a step whose keys are all masked yields p = 0, not NaN)
    const v16i smagic = magic_splat<D>();
    // (e4m3 1.0 = 0x38.  As e2m1, like the main kernel's, they would take four registers less; that was measured there only.)
    const v8i ones8 = {0x38383838, 0x38383838, 0x38383838, 0x38383838, 0x38383838, 0x38383838, 0x38383838, 0x38383838};

    for (int hs = h0; hs < h1; hs++) {
        v16i s[SKB];
        if constexpr (!FUSE) dma_wait<VC>();            // K of this step has landed (V^T was requested after it)
        {
            v4i kf[NK];
#pragma unroll
            for (int n = 0; n < NK; n++) kf[n] = k_frag(n, hs);
#pragma unroll
            for (int kb = 0; kb < SKB; kb++)
#pragma unroll
                for (int st = 0; st < KSTEPS; st++)
                    s[kb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(kf[kb * KSTEPS + st], qf[st], st == 0 ? smagic : s[kb], 0, 0, 0);
        }
        const bool more = hs + 1 < h1;
        if constexpr (!FUSE) {
            reads_done();
            if (more) copy_k(hs + 1);
        }
        const int key0 = key_step(hs) * SK;
        float f[SKB];           // (taken at least so large in every step: in the branch below it was 1 % slower at 256 channels)
#pragma unroll
        for (int kb = 0; kb < SKB; kb++) f[kb] = masked_scale(sq * ksc[(key0 + kb * 32) >> ksh]);
        if (key0 + SK > kv_valid || (key0 < a.km.hi && key0 + SK > a.km.lo) || (a.causal && key0 + SK - 1 > row0)) {
            // (one signed and one unsigned comparison per score, with the lane's first key taken off the limits: spelled out
            // key by key it was 17 instructions per score, or branches over nine of them, as the compiler saw fit, and the
            // one step of a small call is this one.  The call, us, e4m3 [1,107,12,64] 14.4 -> 13.4, [1,176,30,128] 16.2 -> 15.2,
            // with Stats fp16 [1,179,8,128] 14.3 -> 13.8)
            const int first = key0 + half * 4, lim = (a.causal ? min(kv_valid, qrow + 1) : kv_valid) - first;
            const uint32_t from_lo = (uint32_t)(first - a.km.lo), width = (uint32_t)(a.km.hi - a.km.lo);
#pragma unroll
            for (int kb = 0; kb < SKB; kb++)
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int c = kb * 32 + (i >> 2) * 8 + (i & 3);
                    if ((c >= lim) | (from_lo + (uint32_t)c < width)) s[kb][i] = (int)0xFF800000;
                }
        }
        // scores in the log2 domain (the accumulators' bias taken off exactly), or the raw accumulators where
        // one multiply-add does the rest
        float x[SKB][16];
        float mt = -INFINITY;
        constexpr bool EXACT = ADDMASK || VARIANT == 1;
#pragma unroll
        for (int kb = 0; kb < SKB; kb++) {
            if constexpr (ADDMASK) {
                bias[kb].put(bias_lds, lane, key0 + kb * 32, kv_valid);
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const v4f mv = BiasStage::get(bias_lds, l32, half, g);
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        x[kb][g * 4 + e] = fmaf(mv[e], 1.4426950408889634f, (__int_as_float(s[kb][g * 4 + e]) - Magic<D>::F) * f[kb]);
                        mt = fmaxf(mt, x[kb][g * 4 + e]);
                    }
                }
            } else {
                // the maximum on the raw accumulators (monotone in the score since f > 0)
                int mi = s[kb][0];
#pragma unroll
                for (int i = 1; i < 16; i++) mi = max(mi, s[kb][i]);
                mt = fmaxf(mt, mi < 0 ? -INFINITY : (float)(mi - Magic<D>::I) * (f[kb] * (1.0f / kMagicUnit)));
#pragma unroll
                for (int i = 0; i < 16; i++) x[kb][i] = EXACT ? __int_as_float(s[kb][i]) - Magic<D>::F : __int_as_float(s[kb][i]);
            }
        }
        if constexpr (ADDMASK) bias_load(hs + 1);
        {
            const v2u r = __builtin_amdgcn_permlane32_swap(__float_as_uint(mt), __float_as_uint(mt), false, false);
            mt = fmaxf(__uint_as_float(r.x), __uint_as_float(r.y));
        }
        if (__any(mt > m_used + Lazy<VARIANT>::tau)) {
            const float m_new = Lazy<VARIANT>::integer_ref ? ceilf(fmaxf(m_used, mt)) : fmaxf(m_used, mt);
            const float corr = __builtin_amdgcn_exp2f(m_used - m_new);
            m_used = m_new;
            l_run *= corr;
            lacc[0] *= corr;
#pragma unroll
            for (int d = 0; d < DB; d++)
#pragma unroll
                for (int i = 0; i < 16; i++) oacc[d][i] *= corr;
        }
        uint32_t p[8];
#pragma unroll
        for (int k = 0; k < NP; k++) {
            const int kb = k >> 3, i = (2 * k) & 15;
            float e[2];
#pragma unroll
            for (int r = 0; r < 2; r++) {
                float arg;
                if constexpr (ADDMASK) arg = x[kb][i + r] - (m_used - Lazy<VARIANT>::log2_pscale);
                else if constexpr (EXACT) arg = fmaf(x[kb][i + r], f[kb], Lazy<VARIANT>::log2_pscale - m_used);
                else arg = fmaf(x[kb][i + r], f[kb], Lazy<VARIANT>::log2_pscale - fmaf(Magic<D>::F, f[kb], m_used));
                e[r] = __builtin_amdgcn_exp2f(arg);
            }
            if constexpr (VARIANT == 0) {
                const v2h pr = {(_Float16)e[0], (_Float16)e[1]};
                p[k] = __builtin_bit_cast(uint32_t, pr);
                l_run += e[0];
                l_run += e[1];
            } else {
                const int w = k >> 1;
                if (k & 1) p[w] = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(e[0], e[1], (int)p[w], true);
                else p[w] = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(e[0], e[1], 0, false);
            }
        }
        if constexpr (!FUSE) {
            if (more) dma_wait<KC>();                   // V^T of this step (the next step's K was requested after it)
            else dma_wait<0>();
        }
        v4i vf[NV];
#pragma unroll
        for (int n = 0; n < NV; n++) vf[n] = v_frag(n, hs);
        if constexpr (VARIANT == 0) {
#pragma unroll
            for (int n = 0; n < NV; n++) {
                const int jj = n / DB, d = n % DB;
                const v4i pw = {(int)p[jj * 4], (int)p[jj * 4 + 1], (int)p[jj * 4 + 2], (int)p[jj * 4 + 3]};
                oacc[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, vf[n]), __builtin_bit_cast(v8h, pw), oacc[d], 0, 0, 0);
            }
        } else {
            const v8i pw = {(int)p[0], (int)p[1], (int)p[2], (int)p[3], (int)p[4], (int)p[5], (int)p[6], (int)p[7]};
#pragma unroll
            for (int d = 0; d < DB; d++) {
                const v4i lo = vf[2 * d], hi = vf[2 * d + 1];
                const v8i v8 = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
                oacc[d] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(v8, pw, oacc[d], 0, 0, 0, 0, 0, 0);
            }
            lacc = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(ones8, pw, lacc, 0, 0, 0, 0, 0, 0);
        }
        if constexpr (!FUSE) {
            reads_done();
            if (more) copy_v(hs + 1);
        }
    }

    // ---- merge of the KW partial results, in LDS
    float l_row = lacc[0];
    if constexpr (VARIANT == 0) {
        const v2u r = __builtin_amdgcn_permlane32_swap(__float_as_uint(l_run), __float_as_uint(l_run), false, false);
        l_row = __uint_as_float(r.x) + __uint_as_float(r.y);
    }
    if (half == 0) {
        lds_m[wave][l32] = m_used;
        lds_l[wave][l32] = l_row;
    }
    if constexpr (FUSE) __syncthreads();                // (no wave reads K, V^T or the bias any more)
    {
        float* dst = acc_of(wave) + l32 * LD + half * 4;
#pragma unroll
        for (int d = 0; d < DB; d++)
#pragma unroll
            for (int g = 0; g < 4; g++)
                *reinterpret_cast<v4f*>(dst + d * 32 + g * 8) = v4f{oacc[d][g * 4], oacc[d][g * 4 + 1], oacc[d][g * 4 + 2], oacc[d][g * 4 + 3]};
    }
    __syncthreads();
    // ---- normalise, bf16, caller's strides: eight channels of a row per thread and turn
    for (int it = tid; it < ROWS * CPR; it += NW * 64) {
        const int row = it / CPR, ch = (it % CPR) * 8;
        const int r = row >> 5, rl = row & 31, grow = wg_row0 + row;
        if (grow >= a.Nq) continue;
        float mg = lds_m[r * KW][rl];
#pragma unroll
        for (int w = 1; w < KW; w++) mg = fmaxf(mg, lds_m[r * KW + w][rl]);
        float l_tot = 0.0f;
        v4f x0 = {0.0f, 0.0f, 0.0f, 0.0f}, x1 = x0;
#pragma unroll
        for (int w = 0; w < KW; w++) {
            const float sc = __builtin_amdgcn_exp2f(lds_m[r * KW + w][rl] - mg);
            const float* part = acc_of(r * KW + w) + rl * LD + ch;
            const v4f y0 = *reinterpret_cast<const v4f*>(part), y1 = *reinterpret_cast<const v4f*>(part + 4);
            l_tot = fmaf(lds_l[r * KW + w][rl], sc, l_tot);
#pragma unroll
            for (int e = 0; e < 4; e++) x0[e] = fmaf(y0[e], sc, x0[e]), x1[e] = fmaf(y1[e], sc, x1[e]);
        }
        const float inv = 1.0f / l_tot;
        if constexpr (VARIANT == 1) {
            const float* vs = a.vscale + (int64_t)bh * D + ch;
#pragma unroll
            for (int e = 0; e < 4; e++) x0[e] *= vs[e], x1[e] *= vs[4 + e];
        }
        const u32x4 pk = {pack_bf16(x0[0] * inv, x0[1] * inv), pack_bf16(x0[2] * inv, x0[3] * inv),
                          pack_bf16(x1[0] * inv, x1[1] * inv), pack_bf16(x1[2] * inv, x1[3] * inv)};
        *reinterpret_cast<u32x4*>(a.o + b * a.osb + h * a.osh + (int64_t)grow * a.osn + ch) = pk;
        if (a.stats != nullptr && ch == 0) {
            const float shift = FUSE ? lds_shift[row] : a.qshift != nullptr ? a.qshift[(int64_t)bh * a.nq_pad + grow] : 0.0f;
            a.stats[(int64_t)bh * a.Nq + grow] = (mg + __builtin_amdgcn_logf(l_tot) - Lazy<VARIANT>::log2_pscale + shift) * 0.6931471805599453f;
        }
    }
}

// (64 channels, fp16: two workgroups share a compute unit, which takes 128 registers at most.  Under a bias that is 10 %
// of a call whose workgroups are more than the compute units: [1,700,24,64] 31.1 us at 146 registers, 27.7 at 128.)
template <int D, int VARIANT, int KW, bool QF, bool ADDMASK>
__global__ __launch_bounds__(short_waves<D>() * 64, D == 64 && VARIANT == 0 ? 4 : 1) void sage_attn_short_kernel(AttnArgs a, int n_rtiles, int item0, int total_wg) {
    short_body<D, VARIANT, KW, QF, ADDMASK, false>(a, FuseArgs{}, n_rtiles, item0, total_wg);
}

template <int D, int KW, bool ADDMASK>
__global__ __launch_bounds__(512) void sage_attn_fused_kernel(AttnArgs a, FuseArgs f, int n_rtiles, int total_wg) {
    short_body<D, 0, KW, true, ADDMASK, true>(a, f, n_rtiles, 0, total_wg);
}

template <int D, int KW>
static hipError_t launch_fused_dk(const AttnArgs& a, const FuseArgs& f, hipStream_t st) {
    constexpr int ROWS = 32 * (8 / KW);
    const int64_t n_rtiles = (a.Nq + ROWS - 1) / ROWS, total = (int64_t)a.B * a.H * n_rtiles;
    if (total <= 0 || total > 0x7FFFFFFF || a.q_src == nullptr || a.blkk != 64 || a.variant != 0 || a.kv_valid > fused_keys(D)) return hipErrorInvalidValue;
    const dim3 grid((unsigned)total), block(512);
    if (a.amask != nullptr) hipLaunchKernelGGL((sage_attn_fused_kernel<D, KW, true>), grid, block, 0, st, a, f, (int)n_rtiles, (int)total);
    else hipLaunchKernelGGL((sage_attn_fused_kernel<D, KW, false>), grid, block, 0, st, a, f, (int)n_rtiles, (int)total);
    return hipGetLastError();
}

hipError_t launch_attn_fused(const AttnArgs& a, const FuseArgs& f, hipStream_t st) {
    if (a.D == 128) return a.short_kw == 8 ? launch_fused_dk<128, 8>(a, f, st) : launch_fused_dk<128, 4>(a, f, st);
    if (a.D == 64) return a.short_kw == 8 ? launch_fused_dk<64, 8>(a, f, st) : launch_fused_dk<64, 4>(a, f, st);
    return hipErrorInvalidValue;
}

// Where the workgroups are at most one per compute unit: each of them quantizes its head's keys again.
static int fused_runs(int units, int B, int H, int Nq, int kv_valid, int D, int variant) {
    if (variant != 0 || D > 128 || kv_valid > fused_keys(D)) return 0;
    const int64_t bh = (int64_t)B * H;
    return bh * ((Nq + 31) / 32) <= units ? 8 : bh * ((Nq + 63) / 64) <= units ? 4 : 0;
}

bool attn_fused_rule(const AttnPlan& p, int B, int H, int Nq, int kv_valid, int D, int variant, int blkq, int blkk) {
    if (p.main_items > 0 || p.short_kw == 0 || blkk != 64 || blkq != 128 || g_short_mode.load() != 0) return false;
    return fused_runs(compute_units(), B, H, Nq, kv_valid, D, variant) == p.short_kw;
}

template <int D, int VARIANT, int KW>
static hipError_t launch_short_dvk(const AttnArgs& a, hipStream_t st) {
    constexpr int NW = short_waves<D>(), ROWS = 32 * (NW / KW), PIECES = kMainRows<D> / ROWS;
    const int64_t bh = (int64_t)a.B * a.H, qtiles = (a.Nq + kMainRows<D> - 1) / kMainRows<D>;
    const int64_t n_rtiles = a.main_items > 0 ? qtiles : (a.Nq + ROWS - 1) / ROWS;
    const int64_t total = a.main_items > 0 ? (bh * qtiles - a.main_items) * PIECES : bh * n_rtiles;
    if (total <= 0 || total > 0x7FFFFFFF || a.main_items > 0x7FFFFFFF) return hipErrorInvalidValue;
    const dim3 grid((unsigned)total), block(NW * 64);
    const int item0 = (int)a.main_items;
    if (a.q_src != nullptr) {
        if (a.amask != nullptr || a.qmul == nullptr) return hipErrorInvalidValue;
        hipLaunchKernelGGL((sage_attn_short_kernel<D, VARIANT, KW, true, false>), grid, block, 0, st, a, (int)n_rtiles, item0, (int)total);
    } else if (a.amask != nullptr) {
        hipLaunchKernelGGL((sage_attn_short_kernel<D, VARIANT, KW, false, true>), grid, block, 0, st, a, (int)n_rtiles, item0, (int)total);
    } else {
        hipLaunchKernelGGL((sage_attn_short_kernel<D, VARIANT, KW, false, false>), grid, block, 0, st, a, (int)n_rtiles, item0, (int)total);
    }
    return hipGetLastError();
}

hipError_t launch_attn_short(const AttnArgs& a, hipStream_t st) {
    if (a.D == 256) return a.variant == 0 ? launch_short_dvk<256, 0, 4>(a, st) : launch_short_dvk<256, 1, 4>(a, st);
    if (a.D == 128 && a.short_kw == 8) return a.variant == 0 ? launch_short_dvk<128, 0, 8>(a, st) : launch_short_dvk<128, 1, 8>(a, st);
    if (a.D == 128) return a.variant == 0 ? launch_short_dvk<128, 0, 4>(a, st) : launch_short_dvk<128, 1, 4>(a, st);
    if (a.D == 64 && a.short_kw == 8) return a.variant == 0 ? launch_short_dvk<64, 0, 8>(a, st) : launch_short_dvk<64, 1, 8>(a, st);
    if (a.D == 64) return a.variant == 0 ? launch_short_dvk<64, 0, 4>(a, st) : launch_short_dvk<64, 1, 4>(a, st);
    return hipErrorInvalidValue;
}

// Which form, from what each costs on an MI355X: time = base + rounds (r + s steps) + fill (f + g steps) in
// microseconds, with rounds = workgroups / compute units rounded up, fill = workgroups / compute units, steps = key tiles of
// 64 (main kernel, two-run form) or key steps of the longest run (short form); the split schedule: base + per balanced key
// tile.  Four forms: the main kernel, 256 query rows and all keys per workgroup; its loop with 128 rows, the keys split
// over two halves of the waves (two runs: the same tiles, a step of them per wave, results merged in LDS at the end); and the
// short form with 64 rows in four runs or 32 in eight.  What splits the keys is for grids that do not fill the chip: a
// step takes a wave about as long with the chip half empty.  One-shot, us, without the two-run form -> with it: [1,1127,19,128] 39.0 ->
// 32.5, [1,1091,16,128] 36.4 -> 29.2, e4m3 [2,615,16,128] 34.1 -> 31.1, [1,1127,19,64] 30.6 -> 25.7, with a bias
// [1,1153,24,128] 60.2 -> 48.9.  Past about 128 row tiles its workgroups take a second round and the main kernel is ahead
// ([1,1322,30,128] 47 against 58); below 40 to 60 the short form is (eight runs: [1,256,30,128] 16.6 against 18.4).
//
// The same with workgroups of four waves, 128 rows and half of a compute unit's LDS: two share a unit, one's rows in and
// out run beside the other's products, and a last round is nearer full.  The waves copy every tile twice per unit, which is
// what keeps it out of one round and out of long key sequences ([1,4608,24,128] 215 -> 231 us).  [1,3792 x 341,40,128] 56.7 ->
// 49.1, [2,6224 x 63,30,64] 44.6 -> 36.2, [2,775,40,64] 46.2 -> 38.3, [1,2379,40,128] 123.8 -> 118.9; same bits.
//
// A problem of some rounds and a bit more takes two: the main kernel does the full rounds and another form what is left,
// spread over the whole chip, instead of one more round that is nearly empty (short form, 264 items of 32 key tiles, 128
// channels: 84 -> 66 us; of 64 channels 61 -> 43; by earlier forms of both).
// The split schedule, which balances the same problems by handing partial results over in memory, is ahead of both where
// the second of few rounds is a quarter to a half full and the key sequence is long: a sixth (64 channels) and a
// thirteenth (128) of the 788 shapes of its rule that were timed (with earlier forms of the kernels, where it was taken it
// never cost more than 0.5 %); one-shot, main kernel alone -> split: [1,4352 x 8192,19,128] 335 -> 312 us and
// [1,4352 x 8192,19,64] 230 -> 196 (323 row tiles), [1,12288,7,128] 457 -> 433.
struct FormCost {
    float base, r, s, f, g;
    float of(int64_t wgs, int64_t steps, int units) const {
        const float rounds = (float)((wgs + units - 1) / units), fill = (float)wgs / (float)units, n = (float)steps;
        return base + rounds * (r + s * n) + fill * (f + g * n);
    }
};
enum Form { MAIN = 0, TWO_RUNS = 1, RUNS4 = 2, RUNS8 = 3, FORMS = 4 };
constexpr FormCost kNoForm{1e9f, 0.0f, 0.0f, 0.0f, 0.0f};
// Up to 3072 keys, 64 and 128 channels.  Fitted to the differences between the forms of 225 one-shot calls each (120 of 500 to
// 3000 tokens, 65 cross, 40 of 64 to 4096, all forms timed), Q where sdpa_impl puts it; what all forms have in common is not
// in them.  Over those calls the choice costs 0.1 % on average over the best single form, the worst 11 %; without the two-run
// form it cost 3 to 6 % on average.
static const FormCost kCost[2][2][FORMS] = {
    {{{6.00f, 1.70f, 0.70f, 0.00f, 0.03f}, {5.94f, 2.18f, 0.46f, 0.56f, 0.02f}, {4.97f, 2.18f, 0.53f, 0.18f, 0.26f}, {5.18f, 1.40f, 0.40f, 0.00f, 0.25f}},
     {{0.30f, 5.53f, 0.57f, 3.88f, 0.00f}, {1.87f, 5.08f, 0.26f, 0.81f, 0.08f}, {0.45f, 5.44f, 0.72f, 0.00f, 0.07f}, {1.33f, 4.41f, 0.58f, 0.00f, 0.12f}}},
    {{{0.00f, 8.33f, 0.68f, 10.04f, 0.00f}, {3.91f, 5.03f, 0.35f, 5.68f, 0.02f}, {3.16f, 6.96f, 0.32f, 0.00f, 0.70f}, {3.24f, 5.57f, 0.44f, 0.00f, 0.61f}},
     {{0.00f, 6.65f, 0.72f, 9.30f, 0.00f}, {1.82f, 6.43f, 0.35f, 3.58f, 0.05f}, {0.40f, 6.76f, 0.88f, 0.21f, 0.34f}, {0.80f, 5.48f, 1.06f, 0.00f, 0.17f}}},
};
// The main kernel in workgroups of four waves, two to a compute unit (rounds and fill count two of them per unit), against
// the figures above, up to 3072 keys: 120 calls each, chosen where it is ahead it takes 1.2 to 2.5 % off them on average.
static const FormCost kCostFour[2][2] = {{{6.06f, 1.67f, 0.53f, 0.00f, 0.00f}, {1.26f, 4.06f, 0.37f, 1.06f, 0.60f}},
                                         {{1.29f, 7.39f, 0.73f, 7.76f, 0.17f}, {2.29f, 4.29f, 0.72f, 6.77f, 0.25f}}};
// Under an additive bias, fp16 P.V (50 calls of 128 to 2304 tokens at 64 channels, 110 at 128: 0.1 % and nothing).
static const FormCost kCostBias[2][FORMS] = {
    {{0.00f, 7.38f, 1.37f, 19.88f, 0.04f}, {4.24f, 3.73f, 0.78f, 11.53f, 0.00f}, {8.78f, 0.70f, 0.52f, 5.33f, 0.71f}, {7.37f, 1.30f, 0.00f, 2.40f, 1.24f}},
    {{0.00f, 14.94f, 1.53f, 14.28f, 0.06f}, {11.61f, 3.82f, 0.90f, 9.82f, 0.00f}, {10.61f, 5.30f, 0.78f, 3.42f, 0.85f}, {10.33f, 5.25f, 0.32f, 1.00f, 1.35f}},
};
// fp16 P.V with a masked key range (438 one-shot calls at 64 channels, 158 at 128, of 130 to 3072 tokens and up to a round of row
// tiles; steps: of the keys that count; taken up to 40 key tiles), and causal (218 and 555, with and without Stats).  A range costs the main kernel and the
// two-run form 2 to 6 us that the short form does not know: the steps around it go through their general bodies.  By the figures
// of plain calls the two-run form or the main kernel was taken where the short one is ahead: us, so -> by these, [2,1439,4,128] 35.1 -> 29.3,
// [1,940,30,64] 31.3 -> 28.9, causal [2,1303,12,64] 34.6 -> 30.4.  Over those calls the choice costs 0.4, 0.1, 0.5 and 0.1 % on average
// over the best single form (the worst 13 %), by the plain figures 3.9, 0.6, 2.3 and 0.7 %.
static const FormCost kCostRange[2][FORMS] = {
    {{3.23f, 5.60f, 0.61f, 7.13f, 0.00f}, {1.02f, 6.46f, 0.29f, 5.39f, 0.00f}, {3.07f, 0.67f, 0.27f, 1.66f, 0.32f}, {1.04f, 2.46f, 0.00f, 0.00f, 0.53f}},
    {{4.96f, 3.84f, 0.79f, 4.61f, 0.00f}, {0.36f, 8.41f, 0.41f, 2.37f, 0.02f}, {0.72f, 4.72f, 0.72f, 0.00f, 0.37f}, {0.26f, 4.24f, 0.69f, 0.00f, 0.36f}},
};
static const FormCost kCostCausal[2][FORMS] = {
    {{1.36f, 5.53f, 0.50f, 1.86f, 0.00f}, {4.58f, 2.83f, 0.07f, 0.84f, 0.16f}, {4.98f, 0.35f, 0.10f, 0.91f, 0.27f}, {2.72f, 0.97f, 0.00f, 1.15f, 0.24f}},
    {{7.41f, 2.10f, 0.62f, 5.27f, 0.00f}, {6.15f, 4.04f, 0.15f, 2.70f, 0.13f}, {5.09f, 4.20f, 0.10f, 0.77f, 0.51f}, {3.79f, 3.85f, 0.00f, 1.20f, 0.40f}},
};
// 256 channels with a masked range (160 one-shot calls in fp16, 147 in e4m3, of 33 to 2000 tokens and up to a round of row tiles) or
// a bias (80 and 75, up to 4000 keys).  The main kernel takes the steps around a range, and all steps under a bias, in its general
// bodies; by the figures of plain calls, below, it was taken where the short form is ahead: us, so -> by these, keymask [1,457,16,256]
// with 7 keys masked 36.0 -> 30.7, e4m3 [3,61,4,256] with one 27.4 -> 24.3, e4m3 bias [1,78 x 38,24,256] 25.9 -> 23.6.  The choice costs
// 0.1, 0.4, 0.0 and 0.0 % on average over the better form (the worst 24, the next 6 %), by the plain figures 6.9, 3.4, 10.2 and 2.3 %.
static const FormCost kCost256Range[2][FORMS] = {
    {{0.00f, 8.20f, 1.14f, 8.12f, 0.00f}, kNoForm, {0.00f, 7.09f, 0.85f, 0.00f, 0.74f}, kNoForm},
    {{0.00f, 11.99f, 1.46f, 10.95f, 0.00f}, kNoForm, {0.00f, 7.40f, 1.87f, 0.33f, 0.00f}, kNoForm},
};
static const FormCost kCost256Bias[2][FORMS] = {
    {{0.00f, 4.31f, 2.12f, 4.74f, 0.21f}, kNoForm, {0.00f, 4.17f, 1.72f, 0.77f, 0.22f}, kNoForm},
    {{0.00f, 9.07f, 1.51f, 7.38f, 0.00f}, kNoForm, {0.00f, 6.44f, 1.86f, 0.25f, 0.54f}, kNoForm},
};
// e4m3 at 256 channels, plain (with and without Stats) and causal: 134 and 165 such calls.  Below 64 tokens they had gone to the main kernel by its
// figures alone, refitted for longer calls: [1,40,30,256] 25.0 us, 23.6 so.  The choice costs 0.1 and 0.5 % over the better form, by
// those figures 0.8 and 1.7 %.
static const FormCost kCost256E4m3[2][FORMS] = {       // [plain, causal]
    {{0.00f, 8.33f, 0.99f, 3.53f, 0.07f}, kNoForm, {0.00f, 6.10f, 1.58f, 0.57f, 0.00f}, kNoForm},
    {{0.00f, 9.09f, 0.33f, 21.58f, 0.23f}, kNoForm, {0.00f, 6.93f, 0.54f, 4.78f, 0.00f}, kNoForm},
};
// All lengths, by launches and calls of up to 32 768 keys of earlier forms of the kernels (the two-run form against the
// main kernel's figures here): longer key sequences, 256 channels, and what the split schedule is compared with.
static const FormCost kCostLong[3][2][FORMS] = {        // [64, 128, 256 channels]
    {{{6.00f, 1.70f, 0.78f, 0.00f, 0.03f}, {5.94f, 2.48f, 0.46f, 0.56f, 0.02f}, {4.97f, 1.54f, 0.50f, 0.00f, 0.17f}, {5.18f, 1.19f, 0.41f, 0.14f, 0.27f}},
     {{1.91f, 3.27f, 0.76f, 1.13f, 0.06f}, {1.52f, 3.29f, 0.43f, 1.86f, 0.00f}, {3.02f, 1.61f, 1.08f, 1.28f, 0.00f}, {2.55f, 1.40f, 1.20f, 1.06f, 0.00f}}},
    {{{1.29f, 3.84f, 0.75f, 0.88f, 0.54f}, {1.85f, 4.15f, 0.35f, 0.79f, 0.35f}, {2.68f, 3.27f, 0.92f, 0.05f, 0.42f}, {2.56f, 3.24f, 0.95f, 0.04f, 0.36f}},
     {{2.15f, 4.92f, 0.95f, 1.71f, 0.11f}, {2.88f, 3.94f, 0.57f, 2.66f, 0.00f}, {2.52f, 4.17f, 1.20f, 0.18f, 0.30f}, {2.54f, 3.25f, 1.40f, 0.75f, 0.14f}}},
    {{{1.44f, 4.16f, 0.90f, 2.31f, 0.44f}, kNoForm, {2.87f, 6.05f, 1.29f, 0.20f, 0.25f}, kNoForm},
     {{3.61f, 4.01f, 1.09f, 2.79f, 0.10f}, kNoForm, {1.45f, 5.06f, 2.57f, 1.45f, 0.00f}, kNoForm}},
};
// (fp16 at 64 channels past 3072 keys: no one set meets both ends there)
static const FormCost kCost64Long[FORMS] = {{1.81f, 2.54f, 0.66f, 0.34f, 0.16f}, {1.75f, 3.32f, 0.34f, 0.90f, 0.15f}, {3.60f, 0.70f, 0.78f, 0.00f, 0.06f}, {3.72f, 0.77f, 0.55f, 0.03f, 0.18f}};
static const float kSplitCost[2][2] = {{17.0f, 0.96f}, {25.0f, 1.53f}};       // [64, 128 channels]: base, per key tile

// Microseconds a call takes more with the main kernel where its Q cannot go to the encoders for next to nothing:
// many queries on few keys, which keep Q in the kernel's prologue, and a K that takes one launch alone but not with Q.
// One-shot, main kernel against short form: [1,510 x 139,24,128] 20.8 against 19.0, [1,256 x 292,40,128] 25.0 against 22.3,
// e4m3 [2,71 x 45,32,256] 36.3 against 28.8; with as many keys as queries they are level, [1,64,24,128] 15.2 against 15.2
// to 16.0.  (64 channels: nothing to gain, or the second kind's fit is as good without; kCost has it in its figures.)
static const float kQCost[3][2][2] = {{{0.0f, 0.0f}, {0.8f, 0.0f}}, {{1.4f, 1.4f}, {0.0f, 0.0f}}, {{0.0f, 2.0f}, {0.0f, 2.0f}}};

namespace {
struct Choice { float t; AttnPlan p; };
// `rows` query rows of each of bh heads by the form that is predicted fastest, the main kernel's left out
Choice best_small(const FormCost* c, int64_t rows, int64_t bh, int D, int variant, int64_t kv, int units, bool two_runs, float range = 0.0f) {
    const int64_t tiles = (kv + kTileKV - 1) / kTileKV, steps = variant == 0 ? (kv + 31) / 32 : tiles;
    auto wgs = [&](int per) { return bh * ((rows + per - 1) / per); };
    Choice best{1e30f, AttnPlan{0, 4, 0}};
    auto offer = [&](float t, const AttnPlan& p) { if (t < best.t) best = Choice{t, p}; };
    if (two_runs) offer(c[TWO_RUNS].of(wgs(128), variant == 0 ? tiles : (tiles + 1) / 2 * 2, units) + range, AttnPlan{0, 0, 0, true});
    offer(c[RUNS4].of(wgs(D > 128 ? 32 : 64), (steps + 3) / 4, units), AttnPlan{0, 4, 0});
    if (D <= 128) offer(c[RUNS8].of(wgs(32), (steps + 7) / 8, units), AttnPlan{0, 8, 0});
    return best;
}

struct Problem {
    int units, B, H, Nq, kv, D, variant;
    bool causal, bias;
    int masked;                 // keys of the masked range
    int64_t bh() const { return (int64_t)B * H; }
    int64_t tiles() const { return (kv + kTileKV - 1) / kTileKV; }
    int64_t items() const { const int rows = D > 128 ? 128 : 256; return bh() * ((Nq + rows - 1) / rows); }
    int v() const { return variant == 0 ? 0 : 1; }
    int d() const { return D == 64 ? 0 : D == 128 ? 1 : 2; }
};

// alone: whether the forms without the main kernel may do everything
Choice choose(const Problem& s, const FormCost* c, float q_main, float launch, bool two_runs, bool alone = true) {
    const int64_t items = s.items(), whole = items / s.units * s.units;
    // (past a round of row tiles the two-run form does what the main kernel's whole rounds leave: that is ahead of
    // it doing everything, or level)
    Choice best = alone ? best_small(c, s.Nq, s.bh(), s.D, s.variant, s.kv, s.units, two_runs && (s.causal || whole == 0 || whole == items))
                        : Choice{1e30f, AttnPlan{items, 0, 0}};
    const float main = c[MAIN].of(items, s.tiles(), s.units) + q_main;
    if (main <= best.t) best = Choice{main, AttnPlan{items, 0, 0}};
    if (!s.causal && whole > 0 && whole < items) {
        // (a masked range: 3 us of the two-run form that the short form does not know, and the main kernel has either way)
        const float range = s.masked > 0 ? 3.0f : 0.0f;
        const Choice rest = best_small(c, s.D > 128 ? 128 : 256, items - whole, s.D, s.variant, s.kv, s.units, two_runs, range);
        const float t = c[MAIN].of(whole, s.tiles(), s.units) + q_main + launch + rest.t - (rest.p.two_runs ? range : 0.0f);
        if (t < best.t) best = Choice{t, AttnPlan{whole, rest.p.short_kw, 0, rest.p.two_runs}};
    }
    return best;
}

float q_cost(const Problem& s) {
    const int blkq = s.variant == 0 ? 128 : 32;
    const int64_t alone = quant_short_workgroups(s.B, s.H, s.Nq, s.kv, s.D, blkq, 64, false);
    const int64_t with_q = alone > 0 ? quant_short_workgroups(s.B, s.H, s.Nq, s.kv, s.D, blkq, 64, true) : 0;
    return std::max(s.Nq > 2 * s.kv ? kQCost[s.d()][s.v()][0] : 0.0f, alone > 0 && (with_q == 0 || with_q > s.units) ? kQCost[s.d()][s.v()][1] : 0.0f);
}

const FormCost* by_length(const Problem& s) { return s.D == 64 && s.v() == 0 && s.tiles() > 48 ? kCost64Long : kCostLong[s.d()][s.v()]; }

// What the split schedule is compared with: main kernel and short form by the figures for all lengths.
Choice main_or_short(const Problem& s) { return choose(s, by_length(s), q_cost(s), 0.0f, false); }
bool split_ahead(const Problem& s, int split, const Choice& other) {
    return !s.causal && split > 0 && s.D <= 128 && kSplitCost[s.d()][0] + kSplitCost[s.d()][1] * (float)(s.items() * s.tiles()) / 256.0f < other.t;
}
}  // namespace

static AttnPlan plan_by_shape(const Problem& s, int split) {
    if (split > 0 && split_ahead(s, split, main_or_short(s))) return AttnPlan{s.items(), 0, split};
    if (const int runs = fused_runs(s.units, s.B, s.H, s.Nq, s.kv, s.D, s.variant)) return AttnPlan{0, runs, 0};
    // (figures that were fitted to differences have not got what a second launch costs)
    const float launch = s.d() == 0 && s.v() == 0 ? 0.0f : 3.0f;
    // (two key tiles or fewer leave a run nothing to gain, e4m3 [1,926 x 89,30,128] 21.2 us by the main kernel, 23.0 so)
    const bool two_runs = s.D <= 128 && s.tiles() > 2 && pad_to(s.kv, kPadKV) <= kTwoRunKeys && !(s.bias && s.v() == 1);
    // (under a bias at 128 channels the short form alone is not ahead past a round: 1.07 to 2 times the main kernel's time in 53 such
    // calls.  A last row tile of a head that is hardly filled takes the main kernel less than the figures say: us, by the short
    // form -> so, [3,316 x 244,64,128] 53.7 -> 48.7, [3,855 x 52,64,128] 71.5 -> 48.3)
    if (s.D <= 128 && s.bias && s.v() == 0) return choose(s, kCostBias[s.d()], 0.0f, 3.0f, two_runs, s.D == 64 || s.items() <= s.units).p;
    if (s.D <= 128 && !s.bias && s.v() == 0 && s.items() <= s.units && (s.causal || s.masked > 0) && s.tiles() > 2 && s.tiles() <= 40) {
        Problem counted = s;
        counted.kv -= s.masked;
        return choose(counted, (s.causal ? kCostCausal : kCostRange)[s.d()], 0.0f, 0.0f, two_runs).p;
    }
    if (s.D == 256 && s.items() <= s.units && s.tiles() <= 64) {
        Problem counted = s;
        counted.kv -= s.masked;
        const FormCost* c = s.bias ? kCost256Bias[s.v()] : s.masked > 0 ? kCost256Range[s.v()] : s.v() == 1 ? kCost256E4m3[s.causal] : nullptr;
        if (c != nullptr) return choose(counted, c, 0.0f, 0.0f, false).p;
    }
    if (s.D <= 128 && !s.bias && s.tiles() <= 48) {
        const Choice best = choose(s, kCost[s.d()][s.v()], 0.0f, launch, two_runs);
        // Four waves: past a round of row tiles, but for the few that a second launch takes better (16 in 256).  Plain calls at 64
        // channels with fp16 P.V and 20 key tiles or more take it only where its own last round gives at most one workgroup to
        // a unit: that round is the shorter one then, 0.75 to 0.95 of the main kernel's time in 33 calls of 2 to 4 rounds; past it
        // 1.00 to 1.08 in 40 ([1,2602,40,64] 100.4 us against 96.1).  Not so with a range or causal ([2,1921,30,64] 62.9 against 74.1).
        const int64_t items = s.items(), whole = items / s.units * s.units, wgs = s.bh() * ((s.Nq + 127) / 128);
        const int64_t last = (wgs - 1) % (2 * s.units) + 1;
        const bool over = items > s.units && (s.tiles() <= 4 || (items - whole) * 16 > s.units || items == whole) &&
                          !(s.D == 64 && s.v() == 0 && !s.causal && s.masked == 0 && s.tiles() >= 20 && last > s.units);
        const float four = kCostFour[s.d()][s.v()].of(wgs, s.tiles(), 2 * s.units);
        return over && four < best.t ? AttnPlan{items, 0, 0, false, true} : best.p;
    }
    return choose(s, by_length(s), q_cost(s), 0.0f, two_runs).p;
}

void attn_short_override(int mode) { g_short_mode.store(mode); }

int64_t attn_main_items_on(int units, int B, int H, int Nq, int kv_valid, int D, int variant) {
    return plan_by_shape(Problem{units, B, H, Nq, kv_valid, D, variant, false, false, 0}, 0).main_items;
}

// Asked of the device once.  (256 where there is none to ask.)
int compute_units() {
    static std::atomic<int> known[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    int n = known[dev].load();
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        known[dev].store(n);
    }
    return n;
}

AttnPlan attn_plan(int B, int H, int Nq, int kv_valid, int D, int variant, bool causal, bool bias, int masked) {
    const int mode = g_short_mode.load(), rows = D > 128 ? 128 : 256;
    const bool two_runs_fit = D <= 128 && pad_to(kv_valid, kPadKV) <= kTwoRunKeys && !(bias && variant != 0);
    if (mode == 2 && two_runs_fit) return AttnPlan{0, 0, 0, true};
    if (mode == 3 && two_runs_fit && !bias) return AttnPlan{(int64_t)B * H * ((Nq + rows - 1) / rows), 0, 0, false, true};
    if (mode == 2 || mode == 3) return AttnPlan{(int64_t)B * H * ((Nq + rows - 1) / rows), 0, 0};
    if (mode > 0) return AttnPlan{0, D == 256 ? 4 : mode, 0};
    const int split = causal ? 0 : attn_split_workgroups(B, H, Nq, kv_valid, D, variant);
    if (mode < 0 || attn_split_override_mode() != 0)      // (a schedule of the main kernel was asked for)
        return AttnPlan{(int64_t)B * H * ((Nq + rows - 1) / rows), 0, split};
    return plan_by_shape(Problem{compute_units(), B, H, Nq, kv_valid, D, variant, causal, bias, masked}, split);
}

bool attn_q8_only(const AttnPlan& p, int B, int H, int Nq, int kv_valid, int D, int variant) {
    const int split = attn_split_workgroups(B, H, Nq, kv_valid, D, variant);
    if (split <= 0) return false;
    if (g_short_mode.load() != 0 || attn_split_override_mode() != 0) return p.main_items > 0;
    const Problem s{compute_units(), B, H, Nq, kv_valid, D, variant, false, false, 0};
    const Choice other = main_or_short(s);
    return split_ahead(s, split, other) || other.p.main_items > 0;
}

}  // namespace sage
