// sage_api.hip — the C ABI of libmi355_sage.so (declared in include/mi355_sage.h).
// Host-side only: argument checks, workspace carving, kernel sequencing.
#include "../../include/mi355_sage.h"
#include "../../include/mi355_sage_test.h"
#include "sage_internal.h"

#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <mutex>
#include <vector>

using namespace sage;

// Scratch of mi355_sage_sdpa_bf16_static: device memory that belongs to the loaded library, so
// that entry point never allocates.  Each GPU the library runs on holds its own copy of the
// array, at its own address, until the process ends.  In host code the array's NAME is only a
// handle for hipGetSymbolAddress; the address that call returns is what kernels are given.
constexpr size_t kStaticScratchBytes = 16u << 20;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

namespace {

constexpr size_t kAlign = 256;
inline size_t align_up(size_t x) { return (x + kAlign - 1) / kAlign * kAlign; }

#define SAGE_LOG(...)                              \
    do {                                           \
        std::fprintf(stderr, "[mi355_sage] ");     \
        std::fprintf(stderr, __VA_ARGS__);         \
        std::fprintf(stderr, "\n");                \
    } while (0)

#define SAGE_HIP(expr)                                                              \
    do {                                                                            \
        hipError_t e_ = (expr);                                                     \
        if (e_ != hipSuccess) {                                                     \
            SAGE_LOG("%s failed: %s", #expr, hipGetErrorString(e_));                \
            return (int)e_;                                                         \
        }                                                                           \
    } while (0)

// Forward: 64, 128 and (four-wave workgroups, no fused pre-ops) 256 channels per head; backward: 64, 128.
bool dims_ok(int D) { return D == 64 || D == 128 || D == 256; }
bool bwd_dims_ok(int D) { return D == 64 || D == 128; }

// Row starts must be 16-byte aligned and the head dim contiguous.
int check_view(const char* name, const void* p, const int64_t* s, int64_t off, int esz = 2) {
    if (s[3] != 1) {
        SAGE_LOG("%s: innermost stride %lld != 1", name, (long long)s[3]);
        return MI355_SAGE_EUNSUPPORTED;
    }
    const uintptr_t a = reinterpret_cast<uintptr_t>(p) + (uintptr_t)(off * esz);
    if ((a & 15) || (s[0] & 7) || (s[1] & 7) || (s[2] & 7)) {
        SAGE_LOG("%s: rows are not 16-byte aligned", name);
        return MI355_SAGE_EUNSUPPORTED;
    }
    return 0;
}

View make_view(const void* p, const int64_t* s, int64_t off) {
    return View{static_cast<const uint16_t*>(p) + off, s[0], s[1], s[2]};
}

bool blk_ok(int blk) { return blk == 32 || blk == 64 || blk == 128; }

// The attention kernel keeps one head's K scales in LDS.
int check_kv_len(int N_kv, int blkk, int D) {
    (void)blkk;
    if (pad_to(N_kv, kPadKV) > max_keys(D)) {
        SAGE_LOG("N_kv=%d exceeds the %d keys per head the attention kernel takes", N_kv, max_keys(D));
        return MI355_SAGE_EUNSUPPORTED;
    }
    return 0;
}

// Workspace layout of the one-shot calls.
struct Carve {
    size_t q8, k8, vq, qscale, kscale, kmean, qmul, kmul, vscale, kpart_sum, kpart_mm, vpart, qshift, rowinv_q, rowinv_k, split, total;
};

Carve carve(int B, int H, int Nq, int Nkv, int D, int variant) {
    const size_t bh = (size_t)B * H;
    const size_t nqp = (size_t)pad_to(Nq, kTileQ), nkp = (size_t)pad_to(Nkv, kPadKV);
    const size_t ng = (size_t)((Nkv + kGroup - 1) / kGroup);
    Carve c{};
    size_t off = 0;
    auto take = [&](size_t bytes) { size_t o = off; off += align_up(bytes); return o; };
    c.q8 = take(bh * nqp * D);
    c.k8 = take(bh * nkp * D);
    c.vq = take(bh * nkp * D * (variant == MI355_SAGE_PV_FP16 ? 2 : 1));
    c.qscale = take(bh * (nqp / 32) * sizeof(float));      // smallest block is 32 tokens
    c.kscale = take(bh * (nkp / 32) * sizeof(float));
    c.kmean = take(bh * D * sizeof(float));
    c.qmul = take(bh * D * sizeof(float));
    c.kmul = take(bh * D * sizeof(float));
    c.vscale = take(bh * D * sizeof(float));
    c.kpart_sum = take(bh * ng * D * sizeof(double));
    c.kpart_mm = take(bh * ng * D * 2 * sizeof(float));
    c.vpart = take(variant == MI355_SAGE_PV_FP16 ? 0 : bh * ng * D * sizeof(float));
    c.qshift = take(bh * nqp * sizeof(float));
    c.rowinv_q = take((size_t)B * Nq * sizeof(float));        // whole-row RMSNorm statistic per token (optional pre-op)
    c.rowinv_k = take((size_t)B * Nkv * sizeof(float));
    // hand-over slots of the attention kernel's split scheduling, for the shapes that qualify
    c.split = take(attn_split_bytes(attn_split_rule(B, H, Nq, Nkv, D, variant), D));
    c.total = off;
    return c;
}

// Scratch of the stage quantizers: K group sums and minima / maxima, V group maxima.
struct ScratchCarve {
    size_t kpart_sum, kpart_mm, vpart, rowinv_q, rowinv_k, total;
};
ScratchCarve scratch_carve(int B, int H, int Nkv, int D) {
    const size_t n = (size_t)B * H * ((Nkv + kGroup - 1) / kGroup) * D;
    ScratchCarve c{};
    c.kpart_sum = 0;
    c.kpart_mm = align_up(n * sizeof(double));
    c.vpart = c.kpart_mm + align_up(n * 2 * sizeof(float));
    // whole-row RMSNorm statistics (that pre-op needs N_q == N_kv)
    c.rowinv_q = c.vpart + align_up(n * sizeof(float));
    c.rowinv_k = c.rowinv_q + align_up((size_t)B * Nkv * sizeof(float));
    c.total = c.rowinv_k + align_up((size_t)B * Nkv * sizeof(float));
    return c;
}

// Internal workspaces (workspace == NULL): one buffer per (device, stream), so calls on
// different streams never share one.  A buffer that has become too small is replaced by a
// larger one and kept allocated until the process ends: work queued earlier may still be
// using it, and waiting for that work would make the call synchronise.  Sizes at least double,
// so the retired buffers of a stream add up to less than its current one.  Allocation is not
// possible while the stream is being captured into a graph: such a call fails with
// MI355_SAGE_EWORKSPACE unless the buffer is already large enough.
std::mutex g_ws_mutex;
struct StreamWs { int dev; hipStream_t stream; void* p; size_t bytes; };
std::vector<StreamWs> g_ws;          // one-shot calls
std::vector<StreamWs> g_split_ws;    // hand-over slots of mi355_sage_attn_fwd, which takes no workspace

int internal_workspace(std::vector<StreamWs>& registry, size_t need, hipStream_t stream, void** out) {
    int dev = 0;
    SAGE_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(g_ws_mutex);
    StreamWs* w = nullptr;
    for (auto& e : registry)
        if (e.dev == dev && e.stream == stream) { w = &e; break; }
    if (w == nullptr || w->bytes < need) {
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(stream, &cs) == hipSuccess && cs != hipStreamCaptureStatusNone) {
            SAGE_LOG("the internal workspace would have to grow to %zu bytes while the stream is being captured; "
                     "pass a workspace or run the call once before capturing", need);
            return MI355_SAGE_EWORKSPACE;
        }
        const size_t bytes = w ? (need > 2 * w->bytes ? need : 2 * w->bytes) : need;
        void* p = nullptr;
        SAGE_HIP(hipMalloc(&p, bytes));
        if (w == nullptr) {
            registry.push_back(StreamWs{dev, stream, p, bytes});
            w = &registry.back();
        } else {
            w->p = p;              // the old buffer stays allocated (see above)
            w->bytes = bytes;
        }
    }
    *out = w->p;
    return 0;
}

// A call's launches go out together: threads that call on one stream share its workspace (the library's own, or the
// host path's), which is safe in stream order only if no other call's launches fall between them.  One mutex per
// stream, by hash (streams that share one wait for each other's few microseconds of submission); uncontended ~20 ns.
std::mutex& launch_mutex(hipStream_t stream) {
    static std::mutex m[64];
    return m[(reinterpret_cast<uintptr_t>(stream) * 0x9E3779B97F4A7C15ull) >> 58];
}

// The optional ops in front of the quantizers (RMSNorm + interleaved RoPE of Q and of K).
struct Pre {
    PreOp q{}, k{};
    bool full_row = false;      // RMSNorm over all H*D channels of a token (gains of H*D entries)
};

// q_gain / k_gain null together = nothing to do.  Tables are optional on top of the gains.
int make_pre(const void* q_gain, const void* k_gain, float eps, const void* rope_cos, const void* rope_sin,
             int64_t rope_batch_rows, int rope_layout, Pre* out) {
    *out = Pre{};
    if (!q_gain && !k_gain && !rope_cos && !rope_sin) return 0;
    if (!q_gain || !k_gain) { SAGE_LOG("RMSNorm gains must be given for both Q and K"); return MI355_SAGE_EINVAL; }
    if ((rope_cos == nullptr) != (rope_sin == nullptr)) return MI355_SAGE_EINVAL;
    if (!(eps >= 0.0f) || rope_batch_rows < 0) return MI355_SAGE_EINVAL;
    if (rope_layout & ~(MI355_SAGE_ROPE_HALFSPLIT | MI355_SAGE_ROPE_TABLES_BF16 | MI355_SAGE_NORM_FULL_ROW)) return MI355_SAGE_EINVAL;
    const uintptr_t bits = reinterpret_cast<uintptr_t>(q_gain) | reinterpret_cast<uintptr_t>(k_gain) |
                           reinterpret_cast<uintptr_t>(rope_cos) | reinterpret_cast<uintptr_t>(rope_sin);
    if (bits & 15) { SAGE_LOG("gains and RoPE tables must be 16-byte aligned"); return MI355_SAGE_EUNSUPPORTED; }
    out->q = PreOp{static_cast<const uint16_t*>(q_gain), eps, static_cast<const float*>(rope_cos),
                   static_cast<const float*>(rope_sin), rope_batch_rows, (rope_layout & MI355_SAGE_ROPE_HALFSPLIT) ? 1 : 0,
                   (rope_layout & MI355_SAGE_ROPE_TABLES_BF16) ? 1 : 0, nullptr, 0};
    out->full_row = (rope_layout & MI355_SAGE_NORM_FULL_ROW) != 0;
    out->k = out->q;
    out->k.gain = static_cast<const uint16_t*>(k_gain);
    return 0;
}

// Device address of `scratch` on the current device, looked up once per device.
std::mutex g_static_mutex;
void* g_static_ptr[64] = {};

int static_scratch(void** out) {
    int dev = 0;
    SAGE_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= 64) return MI355_SAGE_EUNSUPPORTED;
    std::lock_guard<std::mutex> lock(g_static_mutex);
    if (g_static_ptr[dev] == nullptr) {
        void* p = nullptr;
        SAGE_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (p == nullptr || (reinterpret_cast<uintptr_t>(p) & (kAlign - 1))) return MI355_SAGE_EUNSUPPORTED;
        g_static_ptr[dev] = p;
    }
    *out = g_static_ptr[dev];
    return 0;
}

float cmul_of(float scale) { return (float)((double)scale * 1.4426950408889634074); }   // scale*log2(e), rounded once

// Clips the masked key range to [0, n) and counts the keys that remain.
int clip_mask(int n, int mask_lo, int mask_hi, KeyMask* km) {
    int lo = mask_lo < 0 ? 0 : mask_lo, hi = mask_hi > n ? n : mask_hi;
    if (hi <= lo) lo = hi = 0;
    *km = KeyMask{lo, hi};
    return n - (hi - lo);
}

struct QuantOut {
    int8_t* q8; float* qscale; int8_t* k8; float* kscale;
    float *kmean, *qmul, *kmul;
    double* kpart_sum; float* kpart_mm;
    float* rowdot;
    float *rowinv_q, *rowinv_k;       // whole-row RMSNorm statistics (only with that pre-op)
    uint64_t* flags;                  // room for the hand-over of the one-launch stage, null: the launches
    size_t flag_bytes;
    int once_polls;                   // tests: that form, with so many looks at a flag (< 0: and no flag raised); 0: by the rule
};

// A number for the flags of one call: no two calls of a process share one (SplitMix64's finalizer, a bijection of the counter), and memory that
// other work has filled does not hold it but for a chance of 2^-64 a word.
uint64_t call_tag() {
    static std::atomic<uint64_t> n{(uint64_t)std::chrono::steady_clock::now().time_since_epoch().count() << 20};
    uint64_t z = n.fetch_add(1, std::memory_order_relaxed) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// Looks (0.27 us each) at the other workgroups' flags before a workgroup computes what is missing itself: twice what any takes on a device with
// nothing else on it (16 without the pre-ops, 32 and a few with them: [1,8192,30,128] with norm + RoPE has 61 groups computed twice at 32, none
// at 64), and less than computing a head's groups takes (14 us for five, 60 for 18).  Behind another stream's kernel: see quant_once_kernel.
constexpr int kOncePolls = 64;

bool capturing(hipStream_t st) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &cs) != hipSuccess) {
        (void)hipGetLastError();               // (or the launches that follow would report it as theirs)
        return true;
    }
    return cs != hipStreamCaptureStatusNone;
}

// K statistics + Q / K encoders (+ the V passes when vq is given): launches 1-3, or one launch.
int quantize(const View& q, const View& k, const View* v, int B, int H, int Nq, int Nkv, int D, float scale,
             int blkq, int blkk, int k_flags, const KeyMask& km, int kept, const QuantOut& o,
             int variant, void* vq, float* vscale, float* vpart, const Pre& pre_in, hipStream_t st) {
    Pre pre = pre_in;
    if (pre.full_row) {
        SAGE_HIP(launch_row_inv(q, k, B, H, Nq, Nkv, D, pre.q.eps, o.rowinv_q, o.rowinv_k, st));
        pre.q.row_inv = o.rowinv_q; pre.q.row_n = Nq;
        pre.k.row_inv = o.rowinv_k; pre.k.row_n = Nkv;
    }
    const float cmul = cmul_of(scale);
    const int64_t nqp = pad_to(Nq, kTileQ), nkp = pad_to(Nkv, kPadKV);
    const bool kstats = (k_flags & 3) != 0;
    const bool v_fp8 = v != nullptr && variant != MI355_SAGE_PV_FP16;

    FinalArgs f{};
    f.total = (int64_t)B * H * D; f.D = D; f.ngroups = (Nkv + kGroup - 1) / kGroup; f.kept = kept;
    f.flags = k_flags; f.cmul = cmul;
    f.kpart_sum = kstats ? o.kpart_sum : nullptr; f.kpart_mm = o.kpart_mm;
    f.kmean = o.kmean; f.qmul = o.qmul; f.kmul = o.kmul;
    f.vpart = vpart; f.vscale = v_fp8 ? vscale : nullptr;

    QuantArgs a{};
    a.q = q; a.k = k; a.H = H; a.Nq = Nq; a.Nkv = Nkv; a.nq_pad = nqp; a.nkv_pad = nkp; a.km = km;
    a.blkq = blkq; a.blkk = blkk; a.cmul = cmul;
    a.kmean = o.kmean; a.qmul = o.qmul; a.kmul = o.kmul; a.vscale = vscale;
    a.q8 = o.q8; a.qscale = o.qscale; a.rowdot = o.rowdot; a.k8 = o.k8; a.kscale = o.kscale;
    if (v_fp8) { a.v = *v; a.v8 = static_cast<uint8_t*>(vq); }
    else if (v != nullptr) { a.v = *v; a.v16 = static_cast<uint16_t*>(vq); }
    a.pre_q = pre.q; a.pre_k = pre.k;
    const bool forced = o.once_polls != 0, short_form = v != nullptr && quant_short_workgroups(a, B, D) > 0;
    if (forced || (v != nullptr && o.flags != nullptr &&
                   quant_once_rule(B, H, Nkv, D, blkk, k_flags, v_fp8, a.pre_k.gain != nullptr, pre.full_row, short_form) &&
                   (size_t)quant_once_flag_words(B, H, Nkv, v_fp8) * sizeof(uint64_t) <= o.flag_bytes && !capturing(st))) {
        OnceArgs w{};
        w.q = a; w.f = f;
        w.flags = o.flags; w.tag = call_tag();
        w.polls = forced ? abs(o.once_polls) : kOncePolls;
        w.raise = o.once_polls >= 0;
        SAGE_HIP(launch_quant_once(w, B, D, st));
        return 0;
    }
    if (!forced && short_form) {
        SAGE_HIP(launch_quant_short(a, f, B, D, st));
        return 0;
    }

    PrepArgs p{};
    p.k = k; p.H = H; p.Nkv = Nkv; p.nkv_pad = nkp; p.km = km; p.pre_k = pre.k;
    p.vmode = 2;
    if (v_fp8) {
        p.v = *v;
        p.vmode = 1;                       // (the fp16 repack needs no statistics: it goes with launch 3)
        p.vpart = vpart;
    }
    p.kpart_sum = kstats ? o.kpart_sum : nullptr;
    p.kpart_mm = o.kpart_mm;
    SAGE_HIP(launch_prep(p, B, D, st));
    const bool adds_up = f.kmean != nullptr && quant_adds_up(a);
    if (!adds_up) SAGE_HIP(launch_stats_final(f, st));
    SAGE_HIP(launch_quant(a, adds_up ? &f : nullptr, B, D, st));
    return 0;
}

struct MaskArgs {
    int lo = 0, hi = 0;                // keys lo <= s < hi are masked
    const void* add = nullptr;         // additive bias, bf16, logical [B,H,N_q,N_kv]
    const int64_t* add_strides = nullptr;
    int64_t add_off = 0;
    bool any_row_start = false;        // rows of the bias may start at any even byte address
};

// The bytes from a view's first element to its last, for whether two may share memory.
struct Bytes { uintptr_t lo, hi; };
Bytes view_bytes(const void* p, const int64_t* s, int64_t off, int B, int H, int N, int D) {
    int64_t lo = off, hi = off + D;
    const int64_t last[3] = {(B - 1) * s[0], (H - 1) * s[1], (N - 1) * s[2]};
    for (int64_t x : last) (x < 0 ? lo : hi) += x;
    const uintptr_t base = reinterpret_cast<uintptr_t>(p);
    return Bytes{base + (uintptr_t)(lo * 2), base + (uintptr_t)(hi * 2)};
}
bool meet(const Bytes& a, const Bytes& b) { return a.lo < b.hi && b.lo < a.hi; }

int sdpa_impl(const void* Q, const void* K, const void* V, void* O, void* Stats,
              int B, int H, int N_q, int N_kv, int D, float scale,
              const int64_t* qs, const int64_t* ks, const int64_t* vs, const int64_t* os,
              int64_t q_off, int64_t k_off, int64_t v_off, int64_t o_off, int64_t stats_off,
              int causal, int real_N_kv, void* stream,
              int variant, int blkq, int blkk, int k_flags, void* workspace, size_t workspace_bytes,
              const Pre& pre = Pre{}, const MaskArgs& mask = MaskArgs{}) {
    // argument checks in the order of serenitymojo/ops/cshim/cudnn_sdpa.cpp:391-393
    if (!Q || !K || !V || !O) return MI355_SAGE_EINVAL;
    if (B <= 0 || H <= 0 || N_q <= 0 || N_kv <= 0 || D <= 0) return MI355_SAGE_EINVAL;
    if (!qs || !ks || !vs || !os) return MI355_SAGE_EINVAL;
    if (!dims_ok(D)) { SAGE_LOG("head dim %d not supported (64, 128 or 256)", D); return MI355_SAGE_EUNSUPPORTED; }
    if (D == 256 && pre.q.gain != nullptr) { SAGE_LOG("the fused RMSNorm / RoPE are built for head dims 64 and 128"); return MI355_SAGE_EUNSUPPORTED; }
    if (variant != MI355_SAGE_PV_FP16 && variant != MI355_SAGE_PV_FP8) return MI355_SAGE_EUNSUPPORTED;
    if (!blk_ok(blkq) || !blk_ok(blkk)) { SAGE_LOG("block sizes must be 32, 64 or 128"); return MI355_SAGE_EUNSUPPORTED; }
    if (k_flags & ~3) return MI355_SAGE_EUNSUPPORTED;
    int rc;
    if ((rc = check_kv_len(N_kv, blkk, D))) return rc;
    if ((rc = check_view("Q", Q, qs, q_off)) || (rc = check_view("K", K, ks, k_off)) ||
        (rc = check_view("V", V, vs, v_off)) || (rc = check_view("O", O, os, o_off)))
        return rc;
    if (pre.q.gain != nullptr && (pre.q.cos != nullptr || pre.full_row) && N_q != N_kv) {
        SAGE_LOG("fused RoPE / whole-row RMSNorm are self-attention pre-ops: N_q must equal N_kv");
        return MI355_SAGE_EUNSUPPORTED;
    }
    if (mask.add != nullptr) {
        const int64_t* ms = mask.add_strides;
        if (!ms) return MI355_SAGE_EINVAL;
        const uintptr_t a = reinterpret_cast<uintptr_t>(mask.add) + (uintptr_t)(mask.add_off * 2);
        if (ms[3] != 1 || (!mask.any_row_start && ((a & 7) || (ms[0] & 3) || (ms[1] & 3) || (ms[2] & 3)))) {
            SAGE_LOG("mask: key stride must be 1 and every row 8-byte aligned");
            return MI355_SAGE_EUNSUPPORTED;
        }
    }
    // Keys past the real length are excluded from the statistics and the scores alike:
    // the quantizers see only the first kv tokens.
    const int kv = (real_N_kv > 0 && real_N_kv < N_kv) ? real_N_kv : N_kv;
    KeyMask km;
    const int kept = clip_mask(kv, mask.lo, mask.hi, &km);
    if (kept <= 0) { SAGE_LOG("every key is masked"); return MI355_SAGE_EINVAL; }

    hipStream_t st = static_cast<hipStream_t>(stream);
    std::lock_guard<std::mutex> together(launch_mutex(st));
    const Carve c = carve(B, H, N_q, kv, D, variant);
    uint8_t* ws = static_cast<uint8_t*>(workspace);
    if (ws) {
        if (workspace_bytes < c.total) {
            SAGE_LOG("workspace too small: %zu < %zu", workspace_bytes, c.total);
            return MI355_SAGE_EWORKSPACE;
        }
        if (reinterpret_cast<uintptr_t>(ws) & (kAlign - 1)) return MI355_SAGE_EUNSUPPORTED;
    } else {
        void* p = nullptr;
        if ((rc = internal_workspace(g_ws, c.total, st, &p))) return rc;
        ws = static_cast<uint8_t*>(p);
    }
    // (one decision for carving and launching; slots the caller's workspace was not sized for — a
    // forced schedule of the test switch — come from the library's per-stream buffer)
    const AttnPlan plan = attn_plan(B, H, N_q, kv, D, variant, causal != 0, mask.add != nullptr, km.hi - km.lo);
    // The plain forward leaves Q to the attention kernel, which encodes its own rows (same codes and
    // scales): the quantize stage then neither reads Q nor writes its codes.
    // Not where the encoders have room for it and a prologue is on the path of the whole call — the main kernel does
    // everything in one round that leaves compute units without a workgroup (us with Q in the kernel -> in the
    // encoders, with the stage in one launch by hand-over wherever the call makes it that: [1,700,24,128] 28.5 -> 26.5, [1,1153,24,128] 38.0 -> 34.4,
    // [1,2000,12,128] 42.2 -> 40.2; level at two rounds, [1,2304,24,128] 67.0; [1,4608,24,128] 206.8 -> 209.3) — nor, with e4m3 P.V, whose scale blocks
    // are single waves' and whose prologue costs more, where the short form does all or part of it ([1,256,30,128] 15.7 -> 14.6; the line was drawn where the stage was
    // two launches, [1,1153,24,128] 49.8 -> 46.6, and that call is now 35.4 -> 37.0) or the main kernel fills at most five eighths of the chip
    // (128 of them, [2,320,32,128], 31.1 -> 30.7, where the last of these rules speaks against it; but 240, [1,1497,40,128], 53.3 -> 60.3, 256, [2,1995,16,128], 63.6 -> 71.3, 960, [2,2822,40,128],
    // 285.9 -> 290.1), up to 8192 tokens of 128 channels, 4096 of 64.  Many queries on few keys keep it ([1,3840 x 333,32,128] fp16
    // 43.4 -> 47.3, e4m3 44.0 -> 60.0), and so does a K that takes quant_short_kernel alone and the launches, or more than a
    // workgroup per compute unit, with Q ([1,2048 x 512,32,64] 21.5 -> 26.5, e4m3 [1,512,24,128] 20.4 -> 24.3).
    auto one_launch = [&](bool with_q) { return quant_short_workgroups(B, H, N_q, kv, D, blkq, blkk, with_q); };
    const int units = compute_units();
    // (row tiles of the main kernel's loop in one round or less; of both its forms together where it takes more)
    const int64_t loop_items = plan.two_runs && plan.main_items == 0 ? (int64_t)B * H * ((N_q + kTileQ - 1) / kTileQ) : plan.main_items;
    const bool room = variant == MI355_SAGE_PV_FP8 ? (plan.short_kw > 0 || loop_items * 8 <= units * 5) && (int64_t)N_q * 64 <= (int64_t)4096 * D
                                                   : loop_items > 0 && plan.short_kw == 0 && loop_items < units;
    bool q_in_encoders = room && N_q <= 2 * N_kv;
    if (q_in_encoders && one_launch(false) > 0) {
        const int64_t wgs = one_launch(true);
        q_in_encoders = wgs > 0 && wgs <= units;
    }
    // Outputs that lie over Q, K or V: all three are read by the quantizers' launches then, before the attention kernel
    // writes anything.  (O in Q's own rows needs that in the short form only: elsewhere a workgroup that encodes Q has whole
    // scale blocks, which it reads before it writes.)
    bool over_q = false, over_kv = false;
    {
        const Bytes q = view_bytes(Q, qs, q_off, B, H, N_q, D), k = view_bytes(K, ks, k_off, B, H, N_kv, D), v = view_bytes(V, vs, v_off, B, H, N_kv, D);
        const uintptr_t st0 = reinterpret_cast<uintptr_t>(Stats) + (uintptr_t)(stats_off * 4);
        const Bytes outs[2] = {view_bytes(O, os, o_off, B, H, N_q, D), Stats ? Bytes{st0, st0 + (uintptr_t)((int64_t)B * H * N_q * 4)} : Bytes{0, 0}};
        for (const Bytes& x : outs) {
            const bool own_rows = &x == outs && plan.short_kw == 0 && x.lo == q.lo && os[0] == qs[0] && os[1] == qs[1] && os[2] == qs[2];
            over_q = over_q || (meet(x, q) && !own_rows);
            over_kv = over_kv || meet(x, k) || meet(x, v);
        }
    }
    const bool q_in_kernel = Stats == nullptr && mask.add == nullptr && pre.q.gain == nullptr && (D <= 128 || plan.main_items == 0) &&
                             plan.split_wgs == 0 && !q_in_encoders && !over_q;
    if (pre.q.gain == nullptr && !over_q && !over_kv && attn_fused_rule(plan, B, H, N_q, kv, D, variant, blkq, blkk)) {
        const View q = make_view(Q, qs, q_off);
        AttnArgs a{};
        a.blkq = blkq; a.blkk = blkk; a.variant = variant; a.km = km;
        a.B = B; a.H = H; a.Nq = N_q; a.Nkv = kv; a.kv_valid = kv; a.D = D;
        a.causal = causal ? 1 : 0;
        a.nq_pad = pad_to(N_q, kTileQ); a.nkv_pad = pad_to(kv, kPadKV);
        a.o = static_cast<uint16_t*>(O) + o_off; a.osb = os[0]; a.osh = os[1]; a.osn = os[2];
        a.stats = Stats ? static_cast<float*>(Stats) + stats_off : nullptr;
        if (mask.add != nullptr) {
            a.amask = static_cast<const uint16_t*>(mask.add) + mask.add_off;
            a.amb = mask.add_strides[0]; a.amh = mask.add_strides[1]; a.amn = mask.add_strides[2];
        }
        a.q_src = q.p; a.qsb = q.sb; a.qsh = q.sh; a.qsn = q.sn;
        a.short_kw = plan.short_kw;
        SAGE_HIP(launch_attn_fused(a, FuseArgs{make_view(K, ks, k_off), make_view(V, vs, v_off), kept, k_flags, cmul_of(scale)}, st));
        return MI355_SAGE_OK;
    }
    QuantOut o{};
    o.q8 = q_in_kernel ? nullptr : reinterpret_cast<int8_t*>(ws + c.q8);
    o.k8 = reinterpret_cast<int8_t*>(ws + c.k8);
    o.qscale = reinterpret_cast<float*>(ws + c.qscale);
    o.kscale = reinterpret_cast<float*>(ws + c.kscale);
    o.kmean = reinterpret_cast<float*>(ws + c.kmean);
    o.qmul = reinterpret_cast<float*>(ws + c.qmul);
    o.kmul = reinterpret_cast<float*>(ws + c.kmul);
    o.kpart_sum = reinterpret_cast<double*>(ws + c.kpart_sum);
    o.kpart_mm = reinterpret_cast<float*>(ws + c.kpart_mm);
    o.rowinv_q = reinterpret_cast<float*>(ws + c.rowinv_q);
    o.rowinv_k = reinterpret_cast<float*>(ws + c.rowinv_k);
    // (the flags lie where the whole-row statistics would)
    if (!pre.full_row) { o.flags = reinterpret_cast<uint64_t*>(ws + c.rowinv_q); o.flag_bytes = c.split - c.rowinv_q; }
    // Stats needs <q, kmean> per row: K smoothing lowers every score of a row by it
    float* qshift = (Stats && (k_flags & MI355_SAGE_K_SMOOTH)) ? reinterpret_cast<float*>(ws + c.qshift) : nullptr;
    o.rowdot = qshift;
    void* vq = ws + c.vq;
    float* vscale = reinterpret_cast<float*>(ws + c.vscale);
    float* vpart = reinterpret_cast<float*>(ws + c.vpart);

    const View q = make_view(Q, qs, q_off), k = make_view(K, ks, k_off), v = make_view(V, vs, v_off);
    if ((rc = quantize(q, k, &v, B, H, N_q, kv, D, scale, blkq, blkk, k_flags, km, kept, o, variant, vq, vscale,
                       vpart, pre, st)))
        return rc;

    AttnArgs a{};
    a.q8 = o.q8; a.qscale = o.qscale; a.blkq = blkq;
    a.k8 = o.k8; a.kscale = o.kscale; a.blkk = blkk;
    a.vq = vq; a.vscale = vscale; a.qshift = qshift;
    a.variant = variant;
    a.km = km;
    a.B = B; a.H = H; a.Nq = N_q; a.Nkv = kv; a.kv_valid = kv; a.D = D;
    a.causal = causal ? 1 : 0;
    a.nq_pad = pad_to(N_q, kTileQ); a.nkv_pad = pad_to(kv, kPadKV);
    a.o = static_cast<uint16_t*>(O) + o_off; a.osb = os[0]; a.osh = os[1]; a.osn = os[2];
    a.stats = Stats ? static_cast<float*>(Stats) + stats_off : nullptr;
    if (mask.add != nullptr) {
        a.amask = static_cast<const uint16_t*>(mask.add) + mask.add_off;
        a.amb = mask.add_strides[0]; a.amh = mask.add_strides[1]; a.amn = mask.add_strides[2];
    }
    if (q_in_kernel) {
        a.q_src = q.p; a.qsb = q.sb; a.qsh = q.sh; a.qsn = q.sn;
        a.qmul = o.qmul;
    }
    a.main_items = plan.main_items;
    a.short_kw = plan.short_kw;
    a.two_runs = plan.two_runs; a.four_waves = plan.four_waves;
    a.split_wgs = plan.split_wgs;
    if (a.split_wgs > 0) {
        if (attn_split_bytes(a.split_wgs, D) <= attn_split_bytes(attn_split_rule(B, H, N_q, kv, D, variant), D)) a.split = ws + c.split;
        else if ((rc = internal_workspace(g_split_ws, attn_split_bytes(a.split_wgs, D), st, &a.split))) return rc;
    }
    SAGE_HIP(launch_attn(a, st));
    return MI355_SAGE_OK;
}

int default_blkq(int variant) { return variant == MI355_SAGE_PV_FP8 ? 32 : 128; }
constexpr int kDefaultFlags = MI355_SAGE_K_SMOOTH | MI355_SAGE_K_BALANCE;

}  // namespace

extern "C" {

const char* mi355_sage_version(void) { return "mi355_sage 0.2 gfx950"; }

int64_t mi355_sage_pad_q(int64_t n) { return pad_to(n, kTileQ); }
int64_t mi355_sage_pad_kv(int64_t n) { return pad_to(n, kPadKV); }

int mi355_sage_v_slot(int key_in_tile, int variant) {
    if (key_in_tile < 0 || key_in_tile >= kTileKV) return -1;
    return variant == MI355_SAGE_PV_FP16 ? v_slot_f16(key_in_tile) : v_slot_fp8(key_in_tile);
}

size_t mi355_sage_workspace_bytes(int B, int H, int N_q, int N_kv, int D, int variant) {
    if (B <= 0 || H <= 0 || N_q <= 0 || N_kv <= 0 || !dims_ok(D)) return 0;
    if (variant != MI355_SAGE_PV_FP16 && variant != MI355_SAGE_PV_FP8) return 0;
    return carve(B, H, N_q, N_kv, D, variant).total;
}

size_t mi355_sage_quant_scratch_bytes(int B, int H, int N_kv, int D) {
    if (B <= 0 || H <= 0 || N_kv <= 0 || D <= 0) return 0;
    return scratch_carve(B, H, N_kv, D).total;
}

int mi355_sage_sdpa_bf16(const void* Q, const void* K, const void* V, void* O,
                         int B, int H, int N_q, int N_kv, int D, float scale,
                         const int64_t* q_strides, const int64_t* k_strides,
                         const int64_t* v_strides, const int64_t* o_strides,
                         int64_t q_off, int64_t k_off, int64_t v_off, int64_t o_off,
                         int causal, void* stream,
                         int variant, void* workspace, size_t workspace_bytes) {
    return sdpa_impl(Q, K, V, O, nullptr, B, H, N_q, N_kv, D, scale, q_strides, k_strides, v_strides,
                     o_strides, q_off, k_off, v_off, o_off, 0, causal, 0, stream, variant, default_blkq(variant), 64,
                     kDefaultFlags, workspace, workspace_bytes);
}

int mi355_sage_sdpa_bf16_static(const void* Q, const void* K, const void* V, void* O,
                                int B, int H, int N_q, int N_kv, int D, float scale,
                                const int64_t* q_strides, const int64_t* k_strides,
                                const int64_t* v_strides, const int64_t* o_strides,
                                int64_t q_off, int64_t k_off, int64_t v_off, int64_t o_off,
                                int causal, void* stream, int variant) {
    if (B <= 0 || H <= 0 || N_q <= 0 || N_kv <= 0 || D <= 0) return MI355_SAGE_EINVAL;
    if (!dims_ok(D) || (variant != MI355_SAGE_PV_FP16 && variant != MI355_SAGE_PV_FP8)) return MI355_SAGE_EUNSUPPORTED;
    const size_t need = carve(B, H, N_q, N_kv, D, variant).total;
    if (need > kStaticScratchBytes) {
        SAGE_LOG("mi355_sage_sdpa_bf16_static: this problem needs %zu bytes of scratch, the built-in buffer holds %zu; "
                 "use mi355_sage_sdpa_bf16 with a workspace", need, kStaticScratchBytes);
        return MI355_SAGE_EWORKSPACE;
    }
    // Nothing in the buffer has to start at zero: every byte a kernel of the path reads was
    // written by an earlier kernel of the same call (pad rows and pad blocks included).
    void* p = nullptr;
    int rc;
    if ((rc = static_scratch(&p))) return rc;
    return sdpa_impl(Q, K, V, O, nullptr, B, H, N_q, N_kv, D, scale, q_strides, k_strides, v_strides,
                     o_strides, q_off, k_off, v_off, o_off, 0, causal, 0, stream, variant, default_blkq(variant), 64,
                     kDefaultFlags, p, kStaticScratchBytes);
}

size_t mi355_sage_static_scratch_bytes(void) { return kStaticScratchBytes; }

int mi355_sage_sdpa_bf16_ex(const void* Q, const void* K, const void* V, void* O,
                            int B, int H, int N_q, int N_kv, int D, float scale,
                            const int64_t* q_strides, const int64_t* k_strides,
                            const int64_t* v_strides, const int64_t* o_strides,
                            int64_t q_off, int64_t k_off, int64_t v_off, int64_t o_off,
                            int causal, void* stream,
                            int variant, int blkq, int blkk, int k_flags,
                            void* workspace, size_t workspace_bytes) {
    return sdpa_impl(Q, K, V, O, nullptr, B, H, N_q, N_kv, D, scale, q_strides, k_strides, v_strides,
                     o_strides, q_off, k_off, v_off, o_off, 0, causal, 0, stream, variant, blkq, blkk,
                     k_flags, workspace, workspace_bytes);
}

int mi355_sage_sdpa_bf16_train_fwd(const void* Q, const void* K, const void* V, void* O, void* Stats,
                                   int B, int H, int N_q, int N_kv, int D, float scale,
                                   const int64_t* q_strides, const int64_t* k_strides,
                                   const int64_t* v_strides, const int64_t* o_strides,
                                   int64_t q_off, int64_t k_off, int64_t v_off, int64_t o_off,
                                   int64_t stats_off, int causal, int real_N_q, int real_N_kv,
                                   void* stream, int variant, void* workspace, size_t workspace_bytes) {
    if (!Stats) return MI355_SAGE_EINVAL;              // cudnn_sdpa.cpp:485
    (void)real_N_q;                                    // padded query rows are computed and ignored
    return sdpa_impl(Q, K, V, O, Stats, B, H, N_q, N_kv, D, scale, q_strides, k_strides, v_strides,
                     o_strides, q_off, k_off, v_off, o_off, stats_off, causal, real_N_kv, stream, variant,
                     default_blkq(variant), 64, kDefaultFlags, workspace, workspace_bytes);
}

int mi355_sage_sdpa_bf16_keymask(const void* Q, const void* K, const void* V, void* O, void* Stats,
                                 int B, int H, int N_q, int N_kv, int D, float scale,
                                 const int64_t* q_strides, const int64_t* k_strides,
                                 const int64_t* v_strides, const int64_t* o_strides,
                                 int64_t q_off, int64_t k_off, int64_t v_off, int64_t o_off,
                                 int64_t stats_off, int mask_lo, int mask_hi,
                                 void* stream, int variant, void* workspace, size_t workspace_bytes) {
    if (mask_lo < 0 || mask_hi < mask_lo || mask_hi > N_kv) return MI355_SAGE_EINVAL;
    MaskArgs m;
    m.lo = mask_lo; m.hi = mask_hi;
    return sdpa_impl(Q, K, V, O, Stats, B, H, N_q, N_kv, D, scale, q_strides, k_strides, v_strides,
                     o_strides, q_off, k_off, v_off, o_off, stats_off, 0, 0, stream, variant,
                     default_blkq(variant), 64, kDefaultFlags, workspace, workspace_bytes, Pre{}, m);
}

static int sdpa_mask_entry(const void* Q, const void* K, const void* V, const void* Mask, void* O,
                           int B, int H, int N_q, int N_kv, int D, float scale,
                           const int64_t* q_strides, const int64_t* k_strides,
                           const int64_t* v_strides, const int64_t* mask_strides, const int64_t* o_strides,
                           int64_t q_off, int64_t k_off, int64_t v_off, int64_t mask_off, int64_t o_off,
                           void* stream, int variant, void* workspace, size_t workspace_bytes, bool any_row_start) {
    if (!Mask || !mask_strides) return MI355_SAGE_EINVAL;
    MaskArgs m;
    m.add = Mask; m.add_strides = mask_strides; m.add_off = mask_off; m.any_row_start = any_row_start;
    return sdpa_impl(Q, K, V, O, nullptr, B, H, N_q, N_kv, D, scale, q_strides, k_strides, v_strides,
                     o_strides, q_off, k_off, v_off, o_off, 0, 0, 0, stream, variant,
                     default_blkq(variant), 64, kDefaultFlags, workspace, workspace_bytes, Pre{}, m);
}

int mi355_sage_sdpa_bf16_mask(const void* Q, const void* K, const void* V, const void* Mask, void* O,
                              int B, int H, int N_q, int N_kv, int D, float scale,
                              const int64_t* q_strides, const int64_t* k_strides,
                              const int64_t* v_strides, const int64_t* mask_strides, const int64_t* o_strides,
                              int64_t q_off, int64_t k_off, int64_t v_off, int64_t mask_off, int64_t o_off,
                              void* stream, int variant, void* workspace, size_t workspace_bytes) {
    return sdpa_mask_entry(Q, K, V, Mask, O, B, H, N_q, N_kv, D, scale, q_strides, k_strides, v_strides, mask_strides, o_strides,
                           q_off, k_off, v_off, mask_off, o_off, stream, variant, workspace, workspace_bytes, false);
}

int mi355_sage_sdpa_bf16_mask_any(const void* Q, const void* K, const void* V, const void* Mask, void* O,
                                  int B, int H, int N_q, int N_kv, int D, float scale,
                                  const int64_t* q_strides, const int64_t* k_strides,
                                  const int64_t* v_strides, const int64_t* mask_strides, const int64_t* o_strides,
                                  int64_t q_off, int64_t k_off, int64_t v_off, int64_t mask_off, int64_t o_off,
                                  void* stream, int variant, void* workspace, size_t workspace_bytes) {
    return sdpa_mask_entry(Q, K, V, Mask, O, B, H, N_q, N_kv, D, scale, q_strides, k_strides, v_strides, mask_strides, o_strides,
                           q_off, k_off, v_off, mask_off, o_off, stream, variant, workspace, workspace_bytes, true);
}

static int quant_qk_entry(const void* Q, const void* K, int B, int H, int N_q, int N_kv, int D,
                          float scale, const int64_t* q_strides, const int64_t* k_strides,
                          int64_t q_off, int64_t k_off, const Pre& pre, int blkq, int blkk, int k_flags,
                          int mask_lo, int mask_hi,
                          void* q8, void* qscale, void* k8, void* kscale, void* kmean, void* qmul, void* kmul,
                          void* scratch, size_t scratch_bytes, void* stream) {
    if (!Q || !K || !q8 || !qscale || !k8 || !kscale || !kmean || !qmul || !kmul) return MI355_SAGE_EINVAL;
    if (B <= 0 || H <= 0 || N_q <= 0 || N_kv <= 0 || D <= 0) return MI355_SAGE_EINVAL;
    if (!q_strides || !k_strides) return MI355_SAGE_EINVAL;
    if ((k_flags & 3) && !scratch) return MI355_SAGE_EINVAL;
    if (!dims_ok(D) || !blk_ok(blkq) || !blk_ok(blkk) || (k_flags & ~3)) return MI355_SAGE_EUNSUPPORTED;
    if (D == 256 && pre.q.gain != nullptr) return MI355_SAGE_EUNSUPPORTED;
    const ScratchCarve sc = scratch_carve(B, H, N_kv, D);
    if ((k_flags & 3) && scratch_bytes < sc.total) return MI355_SAGE_EWORKSPACE;
    if (pre.q.gain != nullptr && (pre.q.cos != nullptr || pre.full_row) && N_q != N_kv) return MI355_SAGE_EUNSUPPORTED;
    if (pre.full_row && (!scratch || scratch_bytes < sc.total)) return MI355_SAGE_EWORKSPACE;
    int rc;
    if ((rc = check_view("Q", Q, q_strides, q_off)) || (rc = check_view("K", K, k_strides, k_off))) return rc;
    KeyMask km;
    const int kept = clip_mask(N_kv, mask_lo, mask_hi, &km);
    if (kept <= 0) return MI355_SAGE_EINVAL;
    QuantOut o{};
    o.q8 = static_cast<int8_t*>(q8); o.qscale = static_cast<float*>(qscale);
    o.k8 = static_cast<int8_t*>(k8); o.kscale = static_cast<float*>(kscale);
    o.kmean = static_cast<float*>(kmean); o.qmul = static_cast<float*>(qmul); o.kmul = static_cast<float*>(kmul);
    o.kpart_sum = reinterpret_cast<double*>(static_cast<uint8_t*>(scratch) + sc.kpart_sum);
    o.kpart_mm = reinterpret_cast<float*>(static_cast<uint8_t*>(scratch) + sc.kpart_mm);
    o.rowinv_q = reinterpret_cast<float*>(static_cast<uint8_t*>(scratch) + sc.rowinv_q);
    o.rowinv_k = reinterpret_cast<float*>(static_cast<uint8_t*>(scratch) + sc.rowinv_k);
    return quantize(make_view(Q, q_strides, q_off), make_view(K, k_strides, k_off), nullptr, B, H, N_q, N_kv, D,
                    scale, blkq, blkk, k_flags, km, kept, o, 0, nullptr, nullptr, nullptr, pre,
                    static_cast<hipStream_t>(stream));
}

int mi355_sage_quant_qk_bf16(const void* Q, const void* K, int B, int H, int N_q, int N_kv, int D,
                             float scale, const int64_t* q_strides, const int64_t* k_strides,
                             int64_t q_off, int64_t k_off, int blkq, int blkk, int k_flags,
                             int mask_lo, int mask_hi,
                             void* q8, void* qscale, void* k8, void* kscale, void* kmean, void* qmul, void* kmul,
                             void* scratch, size_t scratch_bytes, void* stream) {
    return quant_qk_entry(Q, K, B, H, N_q, N_kv, D, scale, q_strides, k_strides, q_off, k_off, Pre{}, blkq, blkk,
                          k_flags, mask_lo, mask_hi, q8, qscale, k8, kscale, kmean, qmul, kmul, scratch,
                          scratch_bytes, stream);
}

int mi355_sage_quant_qk_norm_rope_bf16(const void* Q, const void* K, int B, int H, int N_q, int N_kv, int D,
                                       float scale, const int64_t* q_strides, const int64_t* k_strides,
                                       int64_t q_off, int64_t k_off,
                                       const void* q_gain, const void* k_gain, float eps,
                                       const void* rope_cos, const void* rope_sin, int64_t rope_batch_rows, int rope_layout,
                                       int blkq, int blkk, int k_flags,
                                       void* q8, void* qscale, void* k8, void* kscale,
                                       void* kmean, void* qmul, void* kmul,
                                       void* scratch, size_t scratch_bytes, void* stream) {
    Pre pre;
    int rc;
    if ((rc = make_pre(q_gain, k_gain, eps, rope_cos, rope_sin, rope_batch_rows, rope_layout, &pre))) return rc;
    if (!pre.q.gain) return MI355_SAGE_EINVAL;
    return quant_qk_entry(Q, K, B, H, N_q, N_kv, D, scale, q_strides, k_strides, q_off, k_off, pre, blkq, blkk,
                          k_flags, 0, 0, q8, qscale, k8, kscale, kmean, qmul, kmul, scratch, scratch_bytes, stream);
}

int mi355_sage_sdpa_bf16_norm_rope(const void* Q, const void* K, const void* V, void* O,
                                   int B, int H, int N_q, int N_kv, int D, float scale,
                                   const int64_t* q_strides, const int64_t* k_strides,
                                   const int64_t* v_strides, const int64_t* o_strides,
                                   int64_t q_off, int64_t k_off, int64_t v_off, int64_t o_off,
                                   int causal, void* stream,
                                   int variant, int blkq, int blkk, int k_flags,
                                   const void* q_gain, const void* k_gain, float eps,
                                   const void* rope_cos, const void* rope_sin, int64_t rope_batch_rows, int rope_layout,
                                   void* workspace, size_t workspace_bytes) {
    Pre pre;
    int rc;
    if ((rc = make_pre(q_gain, k_gain, eps, rope_cos, rope_sin, rope_batch_rows, rope_layout, &pre))) return rc;
    if (!pre.q.gain) return MI355_SAGE_EINVAL;
    return sdpa_impl(Q, K, V, O, nullptr, B, H, N_q, N_kv, D, scale, q_strides, k_strides, v_strides,
                     o_strides, q_off, k_off, v_off, o_off, 0, causal, 0, stream, variant, blkq, blkk,
                     k_flags, workspace, workspace_bytes, pre);
}

int mi355_sage_sdpa_bf16_norm_rope_train_fwd(const void* Q, const void* K, const void* V, void* O, void* Stats,
                                             int B, int H, int N_q, int N_kv, int D, float scale,
                                             const int64_t* q_strides, const int64_t* k_strides,
                                             const int64_t* v_strides, const int64_t* o_strides,
                                             int64_t q_off, int64_t k_off, int64_t v_off, int64_t o_off,
                                             int64_t stats_off, int causal, int real_N_q, int real_N_kv,
                                             void* stream, int variant,
                                             const void* q_gain, const void* k_gain, float eps,
                                             const void* rope_cos, const void* rope_sin, int64_t rope_batch_rows, int rope_layout,
                                             void* workspace, size_t workspace_bytes) {
    if (!Stats) return MI355_SAGE_EINVAL;
    (void)real_N_q;
    Pre pre;
    int rc;
    if ((rc = make_pre(q_gain, k_gain, eps, rope_cos, rope_sin, rope_batch_rows, rope_layout, &pre))) return rc;
    if (!pre.q.gain) return MI355_SAGE_EINVAL;
    return sdpa_impl(Q, K, V, O, Stats, B, H, N_q, N_kv, D, scale, q_strides, k_strides, v_strides,
                     o_strides, q_off, k_off, v_off, o_off, stats_off, causal, real_N_kv, stream, variant,
                     default_blkq(variant), 64, kDefaultFlags, workspace, workspace_bytes, pre);
}

static int quant_qkv_entry(const void* Q, const void* K, const void* V, int B, int H, int N_q, int N_kv, int D,
                              float scale, const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides,
                              int64_t q_off, int64_t k_off, int64_t v_off,
                              int variant, int blkq, int blkk, int k_flags, int mask_lo, int mask_hi,
                              void* q8, void* qscale, void* k8, void* kscale, void* kmean, void* qmul, void* kmul,
                              void* vq, void* vscale, void* scratch, size_t scratch_bytes, void* stream, const Pre& pre, int once_polls) {
    if (!Q || !K || !V || !k8 || !kscale || !kmean || !qmul || !kmul || !vq || !scratch) return MI355_SAGE_EINVAL;
    if ((q8 == nullptr) != (qscale == nullptr)) return MI355_SAGE_EINVAL;      // both NULL: Q is left to mi355_sage_attn_fwd_q16
    if (B <= 0 || H <= 0 || N_q <= 0 || N_kv <= 0 || D <= 0) return MI355_SAGE_EINVAL;
    if (!q_strides || !k_strides || !v_strides) return MI355_SAGE_EINVAL;
    if (variant != MI355_SAGE_PV_FP16 && variant != MI355_SAGE_PV_FP8) return MI355_SAGE_EUNSUPPORTED;
    if (variant == MI355_SAGE_PV_FP8 && !vscale) return MI355_SAGE_EINVAL;
    if (!dims_ok(D) || !blk_ok(blkq) || !blk_ok(blkk) || (k_flags & ~3)) return MI355_SAGE_EUNSUPPORTED;
    const ScratchCarve sc = scratch_carve(B, H, N_kv, D);
    if (scratch_bytes < sc.total) return MI355_SAGE_EWORKSPACE;
    int rc;
    if ((rc = check_view("Q", Q, q_strides, q_off)) || (rc = check_view("K", K, k_strides, k_off)) ||
        (rc = check_view("V", V, v_strides, v_off)))
        return rc;
    KeyMask km;
    const int kept = clip_mask(N_kv, mask_lo, mask_hi, &km);
    if (kept <= 0) return MI355_SAGE_EINVAL;
    uint8_t* scr = static_cast<uint8_t*>(scratch);
    QuantOut o{};
    o.q8 = static_cast<int8_t*>(q8); o.qscale = static_cast<float*>(qscale);
    o.k8 = static_cast<int8_t*>(k8); o.kscale = static_cast<float*>(kscale);
    o.kmean = static_cast<float*>(kmean); o.qmul = static_cast<float*>(qmul); o.kmul = static_cast<float*>(kmul);
    o.kpart_sum = reinterpret_cast<double*>(scr + sc.kpart_sum);
    o.kpart_mm = reinterpret_cast<float*>(scr + sc.kpart_mm);
    o.rowinv_q = reinterpret_cast<float*>(scr + sc.rowinv_q);
    o.rowinv_k = reinterpret_cast<float*>(scr + sc.rowinv_k);
    if (once_polls != 0) {
        const bool v_fp8 = variant != MI355_SAGE_PV_FP16;
        if (D > 128 || blkk != 64 || !(k_flags & 3) || pre.full_row || (pre.q.cos != nullptr && N_q != N_kv)) return MI355_SAGE_EUNSUPPORTED;
        o.flags = reinterpret_cast<uint64_t*>(scr + sc.total);
        if (scratch_bytes < sc.total + (size_t)quant_once_flag_words(B, H, N_kv, v_fp8) * sizeof(uint64_t)) return MI355_SAGE_EWORKSPACE;
        o.once_polls = once_polls;
    }
    const View v = make_view(V, v_strides, v_off);
    return quantize(make_view(Q, q_strides, q_off), make_view(K, k_strides, k_off), &v, B, H, N_q, N_kv, D, scale,
                    blkq, blkk, k_flags, km, kept, o, variant, vq, static_cast<float*>(vscale),
                    reinterpret_cast<float*>(scr + sc.vpart), pre, static_cast<hipStream_t>(stream));
}

int mi355_sage_quant_qkv_bf16(const void* Q, const void* K, const void* V, int B, int H, int N_q, int N_kv, int D,
                              float scale, const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides,
                              int64_t q_off, int64_t k_off, int64_t v_off,
                              int variant, int blkq, int blkk, int k_flags, int mask_lo, int mask_hi,
                              void* q8, void* qscale, void* k8, void* kscale, void* kmean, void* qmul, void* kmul,
                              void* vq, void* vscale, void* scratch, size_t scratch_bytes, void* stream) {
    return quant_qkv_entry(Q, K, V, B, H, N_q, N_kv, D, scale, q_strides, k_strides, v_strides, q_off, k_off, v_off, variant, blkq, blkk, k_flags,
                           mask_lo, mask_hi, q8, qscale, k8, kscale, kmean, qmul, kmul, vq, vscale, scratch, scratch_bytes, stream, Pre{}, 0);
}

int mi355_sage_quant_once(const void* Q, const void* K, const void* V, int B, int H, int N_q, int N_kv, int D, float scale,
                          const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides, int variant, int blkq,
                          int mask_lo, int mask_hi, const void* q_gain, const void* k_gain, float eps, const void* rope_cos,
                          const void* rope_sin, int rope_layout, void* q8, void* qscale, void* k8, void* kscale, void* kmean, void* qmul,
                          void* kmul, void* vq, void* vscale, void* scratch, size_t scratch_bytes, int polls, void* stream) {
    if (polls == 0) return MI355_SAGE_EINVAL;
    Pre pre;
    int rc;
    if ((rc = make_pre(q_gain, k_gain, eps, rope_cos, rope_sin, 0, rope_layout, &pre))) return rc;
    return quant_qkv_entry(Q, K, V, B, H, N_q, N_kv, D, scale, q_strides, k_strides, v_strides, 0, 0, 0, variant, blkq, 64, kDefaultFlags,
                           mask_lo, mask_hi, q8, qscale, k8, kscale, kmean, qmul, kmul, vq, vscale, scratch, scratch_bytes, stream, pre, polls);
}

int mi355_sage_quant_v_f16(const void* V, int B, int H, int N_kv, int D, const int64_t* v_strides,
                           int64_t v_off, int mask_lo, int mask_hi, void* v16, void* stream) {
    if (!V || !v16 || !v_strides) return MI355_SAGE_EINVAL;
    if (B <= 0 || H <= 0 || N_kv <= 0 || D <= 0) return MI355_SAGE_EINVAL;
    if (!dims_ok(D)) return MI355_SAGE_EUNSUPPORTED;
    int rc;
    if ((rc = check_view("V", V, v_strides, v_off))) return rc;
    PrepArgs p{};
    p.v = make_view(V, v_strides, v_off); p.H = H; p.Nkv = N_kv; p.nkv_pad = pad_to(N_kv, kPadKV);
    clip_mask(N_kv, mask_lo, mask_hi, &p.km);
    p.vmode = 0; p.v16 = static_cast<uint16_t*>(v16);
    SAGE_HIP(launch_prep(p, B, D, static_cast<hipStream_t>(stream)));
    return MI355_SAGE_OK;
}

int mi355_sage_quant_v_fp8(const void* V, int B, int H, int N_kv, int D, const int64_t* v_strides,
                           int64_t v_off, int mask_lo, int mask_hi, void* v8, void* vscale,
                           void* scratch, size_t scratch_bytes, void* stream) {
    if (!V || !v8 || !vscale || !v_strides || !scratch) return MI355_SAGE_EINVAL;
    if (B <= 0 || H <= 0 || N_kv <= 0 || D <= 0) return MI355_SAGE_EINVAL;
    if (!dims_ok(D)) return MI355_SAGE_EUNSUPPORTED;
    const ScratchCarve sc = scratch_carve(B, H, N_kv, D);
    if (scratch_bytes < sc.total) return MI355_SAGE_EWORKSPACE;
    int rc;
    if ((rc = check_view("V", V, v_strides, v_off))) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    PrepArgs p{};
    p.v = make_view(V, v_strides, v_off); p.H = H; p.Nkv = N_kv; p.nkv_pad = pad_to(N_kv, kPadKV);
    if (clip_mask(N_kv, mask_lo, mask_hi, &p.km) <= 0) return MI355_SAGE_EINVAL;
    p.vmode = 1; p.vpart = reinterpret_cast<float*>(static_cast<uint8_t*>(scratch) + sc.vpart);
    SAGE_HIP(launch_prep(p, B, D, st));
    FinalArgs f{};
    f.total = (int64_t)B * H * D; f.D = D; f.ngroups = (N_kv + kGroup - 1) / kGroup;
    f.vpart = p.vpart; f.vscale = static_cast<float*>(vscale);
    SAGE_HIP(launch_stats_final(f, st));
    QuantArgs a{};
    a.v = p.v; a.H = H; a.Nkv = N_kv; a.nkv_pad = p.nkv_pad; a.km = p.km; a.blkq = 32; a.blkk = 32;
    a.vscale = f.vscale; a.v8 = static_cast<uint8_t*>(v8);
    SAGE_HIP(launch_quant(a, nullptr, B, D, st));
    return MI355_SAGE_OK;
}

int mi355_sage_attn_fwd(const void* q8, const void* qscale, int blkq, const void* k8, const void* kscale,
                        int blkk, const void* vq, const void* vscale, int variant, int B, int H, int N_q,
                        int N_kv, int kv_valid, int mask_lo, int mask_hi, int D,
                        void* O, const int64_t* o_strides, int64_t o_off,
                        const void* qshift, void* stats, void* stream) {
    if (!q8 || !qscale || !k8 || !kscale || !vq || !O || !o_strides) return MI355_SAGE_EINVAL;
    if (B <= 0 || H <= 0 || N_q <= 0 || N_kv <= 0 || D <= 0) return MI355_SAGE_EINVAL;
    if (kv_valid <= 0 || kv_valid > N_kv) return MI355_SAGE_EINVAL;
    if (variant == MI355_SAGE_PV_FP8 && !vscale) return MI355_SAGE_EINVAL;
    if (variant != MI355_SAGE_PV_FP16 && variant != MI355_SAGE_PV_FP8) return MI355_SAGE_EUNSUPPORTED;
    if (!dims_ok(D) || !blk_ok(blkq) || !blk_ok(blkk)) return MI355_SAGE_EUNSUPPORTED;
    int rc;
    if ((rc = check_kv_len(N_kv, blkk, D))) return rc;
    if ((rc = check_view("O", O, o_strides, o_off))) return rc;
    AttnArgs a{};
    a.q8 = static_cast<const int8_t*>(q8); a.qscale = static_cast<const float*>(qscale); a.blkq = blkq;
    a.k8 = static_cast<const int8_t*>(k8); a.kscale = static_cast<const float*>(kscale); a.blkk = blkk;
    a.vq = vq; a.vscale = static_cast<const float*>(vscale); a.qshift = static_cast<const float*>(qshift);
    a.variant = variant;
    if (clip_mask(kv_valid, mask_lo, mask_hi, &a.km) <= 0) return MI355_SAGE_EINVAL;
    a.B = B; a.H = H; a.Nq = N_q; a.Nkv = N_kv; a.kv_valid = kv_valid; a.D = D;
    a.nq_pad = pad_to(N_q, kTileQ); a.nkv_pad = pad_to(N_kv, kPadKV);
    a.o = static_cast<uint16_t*>(O) + o_off; a.osb = o_strides[0]; a.osh = o_strides[1]; a.osn = o_strides[2];
    a.stats = static_cast<float*>(stats);
    // Same scheduling, hence the same bits, as the one-shot calls: shapes that are split over a
    // fixed number of workgroups need hand-over slots, kept per (device, stream) by the library.
    const AttnPlan plan = attn_plan(B, H, N_q, kv_valid, D, variant, false, false, a.km.hi - a.km.lo);
    a.main_items = plan.main_items; a.short_kw = plan.short_kw; a.split_wgs = plan.split_wgs; a.two_runs = plan.two_runs; a.four_waves = plan.four_waves;
    std::lock_guard<std::mutex> together(launch_mutex(static_cast<hipStream_t>(stream)));
    const size_t split_bytes = attn_split_bytes(a.split_wgs, D);
    if (split_bytes > 0 && (rc = internal_workspace(g_split_ws, split_bytes, static_cast<hipStream_t>(stream), &a.split))) return rc;
    SAGE_HIP(launch_attn(a, static_cast<hipStream_t>(stream)));
    return MI355_SAGE_OK;
}

int mi355_sage_attn_fwd_q16(const void* Q, const int64_t* q_strides, int64_t q_off, const void* qmul, int blkq,
                            const void* k8, const void* kscale, int blkk, const void* vq, const void* vscale, int variant,
                            int B, int H, int N_q, int N_kv, int kv_valid, int mask_lo, int mask_hi, int D,
                            void* O, const int64_t* o_strides, int64_t o_off, void* stream) {
    if (!Q || !q_strides || !qmul || !k8 || !kscale || !vq || !O || !o_strides) return MI355_SAGE_EINVAL;
    if (B <= 0 || H <= 0 || N_q <= 0 || N_kv <= 0 || D <= 0) return MI355_SAGE_EINVAL;
    if (kv_valid <= 0 || kv_valid > N_kv) return MI355_SAGE_EINVAL;
    if (variant == MI355_SAGE_PV_FP8 && !vscale) return MI355_SAGE_EINVAL;
    if (variant != MI355_SAGE_PV_FP16 && variant != MI355_SAGE_PV_FP8) return MI355_SAGE_EUNSUPPORTED;
    if (!dims_ok(D) || D > 128 || !blk_ok(blkq) || !blk_ok(blkk)) return MI355_SAGE_EUNSUPPORTED;
    int rc;
    if ((rc = check_kv_len(N_kv, blkk, D))) return rc;
    if ((rc = check_view("Q", Q, q_strides, q_off)) || (rc = check_view("O", O, o_strides, o_off))) return rc;
    AttnArgs a{};
    const bool keys = clip_mask(kv_valid, mask_lo, mask_hi, &a.km) > 0;
    const AttnPlan plan = attn_plan(B, H, N_q, kv_valid, D, variant, false, false, a.km.hi - a.km.lo);
    if (attn_q8_only(plan, B, H, N_q, kv_valid, D, variant)) return MI355_SAGE_EUNSUPPORTED;
    a.main_items = plan.main_items; a.short_kw = plan.short_kw; a.two_runs = plan.two_runs; a.four_waves = plan.four_waves;
    const View q = make_view(Q, q_strides, q_off);
    a.q_src = q.p; a.qsb = q.sb; a.qsh = q.sh; a.qsn = q.sn; a.qmul = static_cast<const float*>(qmul); a.blkq = blkq;
    a.k8 = static_cast<const int8_t*>(k8); a.kscale = static_cast<const float*>(kscale); a.blkk = blkk;
    a.vq = vq; a.vscale = static_cast<const float*>(vscale);
    a.variant = variant;
    if (!keys) return MI355_SAGE_EINVAL;
    a.B = B; a.H = H; a.Nq = N_q; a.Nkv = N_kv; a.kv_valid = kv_valid; a.D = D;
    a.nq_pad = pad_to(N_q, kTileQ); a.nkv_pad = pad_to(N_kv, kPadKV);
    a.o = static_cast<uint16_t*>(O) + o_off; a.osb = o_strides[0]; a.osh = o_strides[1]; a.osn = o_strides[2];
    SAGE_HIP(launch_attn(a, static_cast<hipStream_t>(stream)));
    return MI355_SAGE_OK;
}

int mi355_sage_attn_split_faults(int reset) { return attn_split_faults(reset); }
int mi355_sage_quant_once_helps(int reset) { return quant_once_helps(reset); }
int mi355_sage_quant_once_takes(int B, int H, int N_q, int N_kv, int D, int variant, int blkq, int blkk, int k_flags, int with_q) {
    if (B <= 0 || H <= 0 || N_q <= 0 || N_kv <= 0 || !dims_ok(D) || !blk_ok(blkq) || !blk_ok(blkk)) return MI355_SAGE_EINVAL;
    const bool v_fp8 = variant != MI355_SAGE_PV_FP16;
    const Carve c = carve(B, H, N_q, N_kv, D, variant);
    return quant_once_rule(B, H, N_kv, D, blkk, k_flags, v_fp8, false, false, quant_short_workgroups(B, H, N_q, N_kv, D, blkq, blkk, with_q != 0) > 0) &&
           (size_t)quant_once_flag_words(B, H, N_kv, v_fp8) * sizeof(uint64_t) <= c.split - c.rowinv_q;
}

// (declared in include/mi355_sage_test.h: switches for the library's own tests)
int mi355_sage_attn_split_rule(int B, int H, int N_q, int N_kv, int D, int variant) {
    if (B <= 0 || H <= 0 || N_q <= 0 || N_kv <= 0) return 0;
    return attn_split_rule(B, H, N_q, N_kv, D, variant);
}

int mi355_sage_set_attn_split(int mode) {
    if (mode < -1 || mode > kSplitMaxWorkgroups || (mode > 0 && (mode & 7))) return MI355_SAGE_EINVAL;
    attn_split_override(mode);
    return MI355_SAGE_OK;
}

int mi355_sage_set_attn_short(int mode) {
    if (mode != -1 && mode != 0 && mode != 2 && mode != 3 && mode != 4 && mode != 8) return MI355_SAGE_EINVAL;
    attn_short_override(mode);
    return MI355_SAGE_OK;
}

int mi355_sage_attn_plan(int B, int H, int N_q, int N_kv, int D, int variant, int causal, int bias, int masked, int64_t* out) {
    if (B <= 0 || H <= 0 || N_q <= 0 || N_kv <= 0 || masked < 0 || masked >= N_kv || !dims_ok(D) || !out) return MI355_SAGE_EINVAL;
    const AttnPlan p = attn_plan(B, H, N_q, N_kv, D, variant, causal != 0, bias != 0, masked);
    out[0] = p.main_items; out[1] = p.short_kw; out[2] = p.two_runs; out[3] = p.four_waves; out[4] = p.split_wgs;
    out[5] = attn_fused_rule(p, B, H, N_q, N_kv, D, variant, default_blkq(variant), 64);
    return MI355_SAGE_OK;
}

int64_t mi355_sage_attn_main_items(int B, int H, int N_q, int N_kv, int D, int variant) {
    if (B <= 0 || H <= 0 || N_q <= 0 || N_kv <= 0) return 0;
    return attn_plan(B, H, N_q, N_kv, D, variant, false).main_items;
}

int64_t mi355_sage_attn_main_items_on(int units, int B, int H, int N_q, int N_kv, int D, int variant) {
    if (units <= 0 || B <= 0 || H <= 0 || N_q <= 0 || N_kv <= 0 || !dims_ok(D)) return 0;
    return attn_main_items_on(units, B, H, N_q, N_kv, D, variant);
}

int mi355_sage_set_attn_split_wait(int polls) {
    if (polls < -(1 << 24) || polls > (1 << 24)) return MI355_SAGE_EINVAL;
    attn_split_wait(polls);
    return MI355_SAGE_OK;
}

int mi355_sage_cast(int count, const void* const* src, void* const* dst, const int64_t* n, int to_bf16, void* stream) {
    if (count < 1 || count > 4 || !src || !dst || !n) return MI355_SAGE_EINVAL;
    CastArgs a{};
    a.count = count;
    for (int t = 0; t < count; t++) {
        if (n[t] < 0 || (n[t] > 0 && (!src[t] || !dst[t]))) return MI355_SAGE_EINVAL;
        if ((reinterpret_cast<uintptr_t>(src[t]) | reinterpret_cast<uintptr_t>(dst[t])) & 15) {
            SAGE_LOG("cast: tensors must be 16-byte aligned");
            return MI355_SAGE_EUNSUPPORTED;
        }
        a.src[t] = src[t]; a.dst[t] = dst[t]; a.n[t] = n[t];
    }
    SAGE_HIP(launch_cast(a, to_bf16 != 0, static_cast<hipStream_t>(stream)));
    return MI355_SAGE_OK;
}

// ---- backward ---------------------------------------------------------------------------------
struct BwdCarve { size_t lse2, delta, kcen, total; };
static BwdCarve bwd_carve(int B, int H, int Nq, int D) {
    const size_t bh = (size_t)B * H;
    const size_t nqp = (size_t)pad_to(Nq, 64);
    BwdCarve c{};
    size_t off = 0;
    auto take = [&](size_t bytes) { size_t o = off; off += align_up(bytes); return o; };
    c.lse2 = take(bh * nqp * sizeof(float));
    c.delta = take(bh * nqp * sizeof(float));
    c.kcen = take(bh * D * sizeof(float));
    c.total = off;
    return c;
}

size_t mi355_sage_bwd_workspace_bytes(int B, int H, int N_q, int N_kv, int D) {
    if (B <= 0 || H <= 0 || N_q <= 0 || N_kv <= 0 || !bwd_dims_ok(D)) return 0;
    return bwd_carve(B, H, N_q, D).total;
}

static int bwd_impl(bool f32, const void* Q, const void* K, const void* V, const void* O, const void* dO, void* dO_bf16,
                             const void* Stats, void* dQ, void* dK, void* dV,
                             int B, int H, int N_q, int N_kv, int D, float scale,
                             const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides,
                             const int64_t* o_strides, const int64_t* do_strides, const int64_t* dq_strides,
                             const int64_t* dk_strides, const int64_t* dv_strides,
                             int64_t q_off, int64_t k_off, int64_t v_off, int64_t o_off, int64_t do_off,
                             int64_t stats_off, int64_t dq_off, int64_t dk_off, int64_t dv_off,
                             int causal, int real_N_q, int real_N_kv, void* stream,
                             void* workspace, size_t workspace_bytes) {
    // same order as serenitymojo/ops/cshim/cudnn_sdpa_bwd.cpp:348-352
    if (!Q || !K || !V || !O || !dO || !Stats) return MI355_SAGE_EINVAL;
    if (!dQ || !dK || !dV || (f32 && !dO_bf16)) return MI355_SAGE_EINVAL;
    if (B <= 0 || H <= 0 || N_q <= 0 || N_kv <= 0 || D <= 0) return MI355_SAGE_EINVAL;
    if (!q_strides || !k_strides || !v_strides || !o_strides || !do_strides || !dq_strides || !dk_strides || !dv_strides)
        return MI355_SAGE_EINVAL;
    if (causal) { SAGE_LOG("causal attention is not supported"); return MI355_SAGE_EUNSUPPORTED; }
    if (!bwd_dims_ok(D)) { SAGE_LOG("backward: head dim %d is not supported (64 or 128)", D); return MI355_SAGE_EUNSUPPORTED; }
    const int esz = f32 ? 4 : 2;
    int rc;
    if ((rc = check_view("Q", Q, q_strides, q_off)) || (rc = check_view("K", K, k_strides, k_off)) ||
        (rc = check_view("V", V, v_strides, v_off)) || (rc = check_view("O", O, o_strides, o_off)) ||
        (rc = check_view("dO", dO, do_strides, do_off, esz)) || (rc = check_view("dQ", dQ, dq_strides, dq_off, esz)) ||
        (rc = check_view("dK", dK, dk_strides, dk_off, esz)) || (rc = check_view("dV", dV, dv_strides, dv_off, esz)) ||
        (f32 && (rc = check_view("dO_bf16", dO_bf16, do_strides, do_off))))
        return rc;
    // the tile copies address a head's rows with 32-bit byte offsets
    auto span_ok = [&](const char* name, int N, const int64_t* s) {
        if (s[2] < 0 || (uint64_t)(N - 1) * (uint64_t)s[2] * 2 + (uint64_t)D * 2 > 0xFFFFFFFFull) {
            SAGE_LOG("%s: a head's rows span more than 4 GiB (or the row stride is negative)", name);
            return false;
        }
        return true;
    };
    if (!span_ok("Q", N_q, q_strides) || !span_ok("dO", N_q, do_strides) || !span_ok("K", N_kv, k_strides) ||
        !span_ok("V", N_kv, v_strides))
        return MI355_SAGE_EUNSUPPORTED;

    const BwdCarve c = bwd_carve(B, H, N_q, D);
    hipStream_t st = static_cast<hipStream_t>(stream);
    std::lock_guard<std::mutex> together(launch_mutex(st));
    if (workspace == nullptr) {
        if ((rc = internal_workspace(g_ws, c.total, st, &workspace))) return rc;
    } else if (workspace_bytes < c.total || (reinterpret_cast<uintptr_t>(workspace) & (kAlign - 1))) {
        SAGE_LOG("backward workspace: %zu bytes at a 256-byte boundary needed, %zu given", c.total, workspace_bytes);
        return MI355_SAGE_EWORKSPACE;
    }
    uint8_t* ws = static_cast<uint8_t*>(workspace);
    BwdArgs a{};
    a.q = make_view(Q, q_strides, q_off);
    a.k = make_view(K, k_strides, k_off);
    a.v = make_view(V, v_strides, v_off);
    a.o = make_view(O, o_strides, o_off);
    a.dout = make_view(f32 ? dO_bf16 : dO, do_strides, do_off);
    a.dout32 = f32 ? static_cast<const float*>(dO) + do_off : nullptr;
    a.out32 = f32;
    a.stats = static_cast<const float*>(Stats) + stats_off;
    auto out = [&](void* p, int64_t off) { return reinterpret_cast<uint16_t*>(static_cast<uint8_t*>(p) + off * esz); };
    a.dq = out(dQ, dq_off); a.dq_sb = dq_strides[0]; a.dq_sh = dq_strides[1]; a.dq_sn = dq_strides[2];
    a.dk = out(dK, dk_off); a.dk_sb = dk_strides[0]; a.dk_sh = dk_strides[1]; a.dk_sn = dk_strides[2];
    a.dv = out(dV, dv_off); a.dv_sb = dv_strides[0]; a.dv_sh = dv_strides[1]; a.dv_sn = dv_strides[2];
    a.B = B; a.H = H; a.Nq = N_q; a.Nkv = N_kv; a.D = D;
    a.valid_q = real_N_q > 0 && real_N_q < N_q ? real_N_q : N_q;          // cudnn_sdpa_bwd.cpp:362-363
    a.valid_kv = real_N_kv > 0 && real_N_kv < N_kv ? real_N_kv : N_kv;
    a.scale = scale;
    a.lse2 = reinterpret_cast<float*>(ws + c.lse2);
    a.ndelta = reinterpret_cast<float*>(ws + c.delta);
    a.kcen = reinterpret_cast<float*>(ws + c.kcen);
    a.nq_pad = pad_to(N_q, 64);
    SAGE_HIP(launch_bwd(a, st));
    return 0;
}

#define SAGE_BWD_PARAMS                                                                                                          \
    int B, int H, int N_q, int N_kv, int D, float scale, const int64_t *q_strides, const int64_t *k_strides,                     \
        const int64_t *v_strides, const int64_t *o_strides, const int64_t *do_strides, const int64_t *dq_strides,                \
        const int64_t *dk_strides, const int64_t *dv_strides, int64_t q_off, int64_t k_off, int64_t v_off, int64_t o_off,        \
        int64_t do_off, int64_t stats_off, int64_t dq_off, int64_t dk_off, int64_t dv_off, int causal, int real_N_q,             \
        int real_N_kv, void *stream, void *workspace, size_t workspace_bytes
#define SAGE_BWD_ARGS                                                                                                            \
    B, H, N_q, N_kv, D, scale, q_strides, k_strides, v_strides, o_strides, do_strides, dq_strides, dk_strides, dv_strides,       \
        q_off, k_off, v_off, o_off, do_off, stats_off, dq_off, dk_off, dv_off, causal, real_N_q, real_N_kv, stream, workspace,   \
        workspace_bytes
int mi355_sage_sdpa_bwd_bf16(const void* Q, const void* K, const void* V, const void* O, const void* dO, const void* Stats, void* dQ,
                             void* dK, void* dV, SAGE_BWD_PARAMS) {
    return bwd_impl(false, Q, K, V, O, dO, nullptr, Stats, dQ, dK, dV, SAGE_BWD_ARGS);
}
int mi355_sage_sdpa_bwd_f32_grads(const void* Q, const void* K, const void* V, const void* O, const void* dO, void* dO_bf16,
                                  const void* Stats, void* dQ, void* dK, void* dV, SAGE_BWD_PARAMS) {
    return bwd_impl(true, Q, K, V, O, dO, dO_bf16, Stats, dQ, dK, dV, SAGE_BWD_ARGS);
}
#undef SAGE_BWD_PARAMS
#undef SAGE_BWD_ARGS

}  // extern "C"
