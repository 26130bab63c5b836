"""Timed cases of the attention library: the calls its users make, over the sizes they make them at.

Every case goes through the public host surface (mojodiffusion_amd.attention_sage,
mojodiffusion_amd.model_dispatch) as a sampler or trainer does.  A case is a dict:

  kind     which call:
             nomask     sdpa_nomask: a DiT sampler's self-attention (joint text + image tokens)
             cross      ltx2_sdpa_product_fwd_rect: rectangular cross-attention (video / audio / text)
             keymask    sdpa_qwen_keymask: joint attention with padded text keys left out
             bias       sdpa: an additive score bias of shape [B,H,S,S]
             norm_rope  qk_norm_rope_sdpa_nomask: QK RMSNorm + RoPE + attention from the projections
             dh256      ideogram4_sdpa_product_fwd: head dim 256
             train      sdpa_flash_train_fwd followed by sdpa_flash_backward: a trainer's step, BF16
             autograd   record_sdpa on F32 activations and torch.autograd.grad through it
  B, H, Sq, Skv, D   batch, heads, query tokens, key tokens, head dim
  fp8      False: INT8 QK^T with FP16 P.V; True: INT8 QK^T with FP8-e4m3 P.V
  n_txt, real_txt    text tokens in front, and how many of them are real (keymask, bias)
"""
import torch

from mojodiffusion_amd import attention_sage as A
from mojodiffusion_amd import model_dispatch as M


def _case(kind, B, H, Sq, Skv, D, fp8=False, n_txt=0, real_txt=0):
    return {"kind": kind, "B": B, "H": H, "Sq": Sq, "Skv": Skv, "D": D, "fp8": fp8, "n_txt": n_txt, "real_txt": real_txt}


def listed():
    named = {
        # the text refiner of a DiT: a couple of hundred tokens, launches and host time are what counts
        "refiner_256": _case("nomask", 1, 30, 256, 256, 128),
        # the small self-attention of the library's first workload, head dim 64
        "small_dh64": _case("nomask", 1, 8, 1024, 1024, 64),
        # cross-attention of a video block onto its text tokens: many queries, few keys, odd lengths
        "cross_text": _case("cross", 1, 32, 3840, 333, 128),
        # joint text + image attention of a 1024x1024 sampler step (512 + 4096 tokens): the headline shape
        "joint_4608": _case("nomask", 1, 24, 4608, 4608, 128),
        # 2048x2048 sampler step with FP8 P.V
        "sampler_16896_fp8": _case("nomask", 1, 24, 16896, 16896, 128, fp8=True),
        # a video sampler's full self-attention, the longest sequence of the workloads
        "video_32760_fp8": _case("nomask", 1, 40, 32760, 32760, 128, fp8=True),
        # joint attention with padded text keys, ragged length
        "keymask_4429": _case("keymask", 1, 24, 4429, 4429, 128, n_txt=333, real_txt=141),
        # additive mask (padded text keys as -1e4), odd length
        "bias_1153": _case("bias", 1, 24, 1153, 1153, 128, n_txt=129, real_txt=57),
        # the block's attention from the projections on, two images per batch (256 + 4096 tokens)
        "norm_rope_4352": _case("norm_rope", 2, 30, 4352, 4352, 128),
        # head dim 256, odd length
        "dh256_1153": _case("dh256", 1, 18, 1153, 1153, 256),
        # a LoRA trainer's step at 512x512, two images: forward with statistics, then the backward
        "train_1248": _case("train", 2, 30, 1248, 1248, 128),
        # F32 activations through the autograd node, head dim 64
        "autograd_2304_dh64": _case("autograd", 1, 12, 2304, 2304, 64),
    }
    return [dict(c, name=n) for n, c in named.items()]


_MOST = 4 * 40 * 32760 ** 2 * 128          # operations of the largest listed case


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    """One more case: the same calls, heads, batches and lengths over the whole range, odd ones among them."""
    while True:
        kind = rng.choice(["nomask", "nomask", "nomask", "cross", "keymask", "bias", "norm_rope", "dh256", "train", "train", "autograd"])
        B, H, fp8 = rng.choice([1, 1, 2]), rng.choice([4, 8, 12, 16, 19, 24, 30, 32, 40]), rng.random() < 0.35
        D = 256 if kind == "dh256" else rng.choice([64, 128, 128])
        lo, hi = {"nomask": (64, 24576), "cross": (256, 12288), "keymask": (256, 9216), "bias": (128, 2304), "norm_rope": (128, 9216),
                  "dh256": (128, 4608), "train": (128, 4608), "autograd": (128, 4608)}[kind]
        Sq = _log_int(rng, lo, hi)
        if rng.random() < 0.5:
            Sq = max(64, Sq // 64 * 64)
        Skv = _log_int(rng, 16, 2048) if kind == "cross" else Sq
        n_txt = real = 0
        if kind in ("keymask", "bias"):
            n_txt = max(2, int(Sq * rng.uniform(0.05, 0.5)))
            real = rng.randint(1, n_txt)
        if kind in ("train", "autograd", "bias"):
            fp8 = False                     # (trainers and masked callers keep FP16 P.V)
        c = _case(kind, B, H, Sq, Skv, D, fp8, n_txt, real)
        if work(c)["flops"] <= _MOST:
            return c


def prepare(case, seed):
    B, H, Sq, Skv, D = (case[n] for n in ("B", "H", "Sq", "Skv", "D"))
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))

    def normal(shape, dtype=torch.bfloat16):
        return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).to(dtype)

    kind = case["kind"]
    s = {"kind": kind, "scale": D ** -0.5, "variant": A.PV_FP8 if case["fp8"] else A.PV_FP16}
    act = torch.float32 if kind == "autograd" else torch.bfloat16
    s["q"], s["v"] = normal((B, Sq, H, D), act), normal((B, Skv, H, D), act)
    k = torch.randn((B, Skv, H, D), generator=g, device="cuda", dtype=torch.float32)
    if kind in ("nomask", "cross", "keymask"):
        # keys of a trained model carry a large offset per channel
        k += 4.0 * torch.randn((B, 1, H, D), generator=g, device="cuda", dtype=torch.float32)
    s["k"] = k.to(act)
    if kind == "keymask":
        s["n_txt"], s["real_txt"] = case["n_txt"], case["real_txt"]
    if kind == "bias":
        # padded text keys far below the rest, a small score bias elsewhere
        mask = (0.5 * torch.randn((B, H, Sq, Skv), generator=g, device="cuda", dtype=torch.float32))
        mask[..., case["real_txt"]:case["n_txt"]] = -1e4
        s["mask"] = mask.to(torch.bfloat16)
    if kind == "norm_rope":
        s["q_norm"], s["k_norm"] = ((1.0 + 0.1 * torch.randn((D,), generator=g, device="cuda")).to(torch.bfloat16) for _ in range(2))
        freq = 10000.0 ** (-torch.arange(D // 2, device="cuda", dtype=torch.float32) / (D // 2))
        angle = torch.arange(Sq, device="cuda", dtype=torch.float32)[:, None] * freq
        s["cos"], s["sin"] = (t.repeat_interleave(H, dim=0).contiguous() for t in (angle.cos(), angle.sin()))   # row = token * H + head
    if kind in ("train", "autograd"):
        s["d_out"] = normal((B, Sq, H, D), act)
    if kind == "autograd":
        for n in ("q", "k", "v"):
            s[n].requires_grad_(True)
    return s


def run(s):
    kind, q, k, v, scale, variant = s["kind"], s["q"], s["k"], s["v"], s["scale"], s["variant"]
    if kind == "nomask":
        return A.sdpa_nomask(q, k, v, scale, variant)
    if kind == "cross":
        return M.ltx2_sdpa_product_fwd_rect(q, k, v, scale, variant)
    if kind == "keymask":
        return A.sdpa_qwen_keymask(q, k, v, s["n_txt"], s["real_txt"], scale, variant)
    if kind == "bias":
        return A.sdpa(q, k, v, s["mask"], scale, variant)
    if kind == "norm_rope":
        return A.qk_norm_rope_sdpa_nomask(q, k, v, s["q_norm"], s["k_norm"], 1e-6, s["cos"], s["sin"], scale, variant)
    if kind == "dh256":
        return M.ideogram4_sdpa_product_fwd(q, k, v, scale, variant)
    if kind == "train":
        fwd = A.sdpa_flash_train_fwd(q, k, v, scale, variant)
        grads = A.sdpa_flash_backward(fwd, s["d_out"], scale)
        return fwd.o, fwd.stats, grads.d_q, grads.d_k, grads.d_v
    if kind == "autograd":
        att = A.record_sdpa(q, k, v, scale, variant)
        return (att.detach(),) + tuple(torch.autograd.grad(att, (q, k, v), s["d_out"]))
    raise ValueError(kind)


def work(case):
    B, H, Sq, Skv, D, kind = (case[n] for n in ("B", "H", "Sq", "Skv", "D", "kind"))
    kept = Skv - (case["n_txt"] - case["real_txt"] if kind == "keymask" else 0)
    flops = 4 * B * H * Sq * kept * D                                # Q K^T and P V
    size = 4 if kind == "autograd" else 2
    data = B * H * D * size * (2 * Sq + 2 * kept)                    # q and o, k and v
    if kind == "bias":
        data += 2 * B * H * Sq * Skv
    if kind == "norm_rope":
        data += 2 * 4 * Sq * H * (D // 2)                            # the cos and sin tables
    if kind in ("train", "autograd"):
        flops += 10 * B * H * Sq * Skv * D                           # the backward's five products
        data += B * H * D * size * (2 * Sq + 2 * Skv)                # d_out and d_q, d_k and d_v
    if kind == "train":
        data += 4 * B * H * Sq                                       # Stats
    return {"bytes": data, "flops": flops}


def tolerance(case):
    # results are bf16, from INT8 / FP16 or bf16 matrix operands; e4m3 probabilities carry 2^-4 each, and another
    # correct implementation may round them against another reference maximum
    return {"rel": 2e-2 if case["fp8"] else 1e-2}
