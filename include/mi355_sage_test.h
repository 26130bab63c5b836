/* mi355_sage_test.h — switches of libmi355_sage.so that exist for its own tests and measurements.
 * Not part of the interface a caller binds (include/mi355_sage.h); process-wide, not thread-safe
 * against calls in flight. */
#ifndef MI355_SAGE_TEST_H
#define MI355_SAGE_TEST_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Attention scheduling.  mode 0: by shape and device (default); -1: one 256-row workgroup per row tile
 * whatever the shape (never split, never the short form below); n > 0 (multiple
 * of 8, <= 1024): always split over n workgroups (fp16 variant, head dim up to 128; hand-over slots
 * a caller's workspace does not hold come from a library-owned per-stream buffer).  Returns 0, or -1
 * for a mode outside these. */
int mi355_sage_set_attn_split(int mode);

/* How long a workgroup of the split schedule polls for another workgroup's partial result before
 * it gives up, writes NaN into its rows and counts a fault.  polls > 0: that many polls of about a
 * microsecond (default 262144; the longest wait that can legitimately occur is one row tile's worth
 * of work, a few milliseconds); 0: back to the default; polls < 0: no workgroup announces its
 * result and every waiting one gives up after -polls polls, which is how the give-up path is
 * exercised without a hang. */
int mi355_sage_set_attn_split_wait(int polls);

/* Workgroups the split schedule would use for this shape on a device that supports it (256), or 0
 * where it is not considered: the rule that sizes the workspace, whatever the switch above and the
 * device say.  Whether it is taken is decided by the predicted costs of the forms. */
int mi355_sage_attn_split_rule(int B, int H, int N_q, int N_kv, int D, int variant);

/* The short form of the attention kernel (32 or 64 query rows per workgroup, keys split over its
 * waves).  mode 0: by shape (default); -1: never; 8 or 4: always, with that many key runs per row
 * block (head dim 256: always 4); 2: the two-run form of the main kernel instead (128 rows, the keys split over two halves
 * of the waves), where it exists (not at head dim 256, under a bias with e4m3, or past 32768 keys); 3: the main kernel in
 * workgroups of four waves, where they exist (not under any bias either).  2, 3, 4 and 8 take
 * precedence over the switch above, which otherwise keeps the short and the two-run form out when it is set.  Returns 0, or -1 for
 * a mode outside these. */
int mi355_sage_set_attn_short(int mode);

/* The forms that a one-shot call of this shape takes (default blocks, no pre-ops) on the current device and under the
 * current switches, six numbers: row tiles of the main kernel; key runs of the short form, which does the rest (or
 * everything), 0 without it; 1: the two-run form does the rest (or everything); 1: the main kernel's row tiles in
 * workgroups of four waves; workgroups of the split schedule, 0 without it; 1: the short form quantizes K and V
 * itself (one launch).  causal and bias: whether the call has that mask; masked: keys of a
 * masked range.  Returns 0, or -1 for a bad shape. */
int mi355_sage_attn_plan(int B, int H, int N_q, int N_kv, int D, int variant, int causal, int bias, int masked, int64_t* out);

/* Row tiles (256 rows of a head; 128 at head dim 256) the main kernel would do for this shape on the current
 * device and under the current switches; the short or the two-run form does the others. */
int64_t mi355_sage_attn_main_items(int B, int H, int N_q, int N_kv, int D, int variant);

/* The same by the shape alone, on a device of that many compute units and without the split schedule. */
int64_t mi355_sage_attn_main_items_on(int units, int B, int H, int N_q, int N_kv, int D, int variant);

/* The quantize stage as the one launch whose workgroups hand their statistics to each other, whatever the shape (head
 * dims 64 and 128, K blocks of 64 keys, both K flags): outputs as mi355_sage_quant_qkv_bf16's, bit for bit, with the pre-ops of
 * mi355_sage_quant_qk_norm_rope_bf16 where q_gain is given.  scratch: mi355_sage_quant_scratch_bytes and 16 bytes
 * more per head and group of 256 keys, with any contents: behind mi355_sage_quant_scratch_bytes lie the flags, 8 bytes each, by head those of K's
 * groups and, with e4m3, of V's.  polls > 0: looks at the flags before a workgroup computes the groups that are missing
 * itself; polls < 0: no workgroup raises a flag, and every one computes all groups after -polls looks. */
int mi355_sage_quant_once(const void* Q, const void* K, const void* V, int B, int H, int N_q, int N_kv, int D, float scale,
                          const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides, int variant, int blkq,
                          int mask_lo, int mask_hi, const void* q_gain, const void* k_gain, float eps, const void* rope_cos,
                          const void* rope_sin, int rope_layout, void* q8, void* qscale, void* k8, void* kscale, void* kmean, void* qmul,
                          void* kmul, void* vq, void* vscale, void* scratch, size_t scratch_bytes, int polls, void* stream);

/* Groups that workgroups of that launch, in any call on the current device, computed after they had waited for them, since the last
 * reset (< 0: a HIP error).  Asked after the caller's own synchronisation. */
int mi355_sage_quant_once_helps(int reset);
/* 1 where a one-shot call of that shape without pre-ops, not under capture, makes its quantize stage that launch (with_q: Q's codes in it). */
int mi355_sage_quant_once_takes(int B, int H, int N_q, int N_kv, int D, int variant, int blkq, int blkk, int k_flags, int with_q);

#ifdef __cplusplus
}
#endif
#endif
