"""Rows whose maximum rises along the keys, in the main kernel's main loop (test_reference_maximum_keeps_rising has rises
so steep, on a problem so short, that the short form and the loop's careful bodies take it): the optimistic steps that
are done again (fp16), the reference that is raised inside a trip (e4m3), and the rescaled accumulators, sums and Stats.
What the inputs make happen is counted on the host, from the oracle's codes and scales."""
import numpy as np
import pytest

from mojodiffusion_amd import _lib
from mojodiffusion_amd.workloads import bf16_bits_to_f32, f32_to_bf16_bits

pytestmark = pytest.mark.gpu

EXACT_BIAS, MAGIC_F, MAGIC_UNIT = 4096.0, 0.15915494309189532, 2.0 ** 26        # csrc/sage_attn_common.h


def _inputs(S, H, D, rise, seed):
    """Even queries lie along one direction and odd ones against it; the keys' share of it grows by `rise` powers of two of
    the score per 64 keys.  One key per tile is ahead of the rest of its tile by a tile's rise: its place goes through the
    four combinations of half-wave (key bit 2) and 32-key block."""
    rng = np.random.default_rng(seed)
    u = rng.choice([-1.0, 1.0], (1, 1, H, D))
    q, k, v = (rng.standard_normal((1, S, H, D)) for _ in range(3))
    q = 0.2 * q + 1.4 * u * np.where(np.arange(S) % 2 == 0, 1.0, -1.0)[None, :, None, None]
    tile = np.arange(S) // 64
    level = tile - 1.0
    for t in range(S // 64):
        level[t * 64 + 9 + 4 * (t & 1) + 32 * (t >> 1 & 1)] = t
    per_unit = 1.4 * D * D ** -0.5 * np.log2(np.e)           # score (log2) per unit of the keys' share
    k = 0.2 * k + (u * ((level - tile[-1] / 2) * rise / per_unit)[None, :, None, None])
    return [f32_to_bf16_bits(x.astype(np.float32)) for x in (q, k, v)]


def _what_happens(oracle, q, k, scale, variant, blkq, mask):
    """Steps of the main loop at which a wave of 32 rows raises its reference, as a share of those steps, per wave; and the
    largest accumulator bias times score scale."""
    import gpu_harness as G
    S = k.shape[1]
    g = G.oracle_quant_qk(oracle, q, k, scale, blkq, 64, True, True, mask)
    qs, ks = np.repeat(g["qscale"], blkq, -1)[..., :S], np.repeat(g["kscale"], 64, -1)[..., :S]
    s = np.einsum("bhid,bhjd->bhij", g["q8"][:, :, :S].astype(np.float32), g["k8"][:, :, :S].astype(np.float32)) * qs[..., None] * ks[:, :, None, :]
    s[..., mask[0]:mask[1]] = -np.inf
    step = 32 if variant == 0 else 64
    n = S // step - 8 * (64 // step)                          # (the last tiles go through the general bodies)
    waves = s[..., :S // 32 * 32, :].reshape(s.shape[0], s.shape[1], -1, 32, S)
    ref = waves[..., :step].max(-1)
    if variant == 1:
        ref = np.ceil(ref)
    raised = np.zeros(waves.shape[:3])
    for h in range(1, n):
        x = waves[..., h * step:(h + 1) * step]
        top = x.max(-1)
        if variant == 0:
            with np.errstate(over="ignore"):
                again = (np.exp2(np.minimum(x - ref[..., None], 100)).sum(-1) > 8192).any(-1)     # (one lane has half of a row's keys)
            new = np.maximum(ref, top)
        else:
            again = (top > ref + 1).any(-1)
            new = np.ceil(np.maximum(ref, top))
        raised += again
        ref = np.where(again[..., None], new, ref)
    kept = np.r_[0:mask[0], mask[1]:S]                        # (blocks without any key that counts have scale 1)
    return raised / n, MAGIC_F * MAGIC_UNIT * float(qs.max()) * float(ks[..., kept].max())


@pytest.mark.parametrize("form", [-1, 4])
@pytest.mark.parametrize("call", ["plain", "stats", "range"])
@pytest.mark.parametrize("variant,D,S,rise", [(0, 128, 1600, 8.0), (0, 64, 1601, 8.0), (0, 128, 959, 14.0), (0, 64, 2047, 3.0),
                                              (1, 128, 1600, 1.7), (1, 64, 1601, 1.7), (1, 128, 959, 3.0), (1, 64, 2047, 2.2)])
def test_rising_reference(oracle, form, call, variant, D, S, rise):
    import gpu_harness as G
    from mojodiffusion_amd import attention_sage as A
    scale, blkq = D ** -0.5, 128 if variant == 0 else 32
    q, k, v = _inputs(S, 2, D, rise, S + D)
    lo, hi = (150, 150 + 3 * 64) if call == "range" else (0, 0)
    raised, bias = _what_happens(oracle, q, k, scale, variant, blkq, (lo, hi))
    assert raised.min() >= 0.1 and (variant == 0 or bias <= EXACT_BIAS), (raised.min(), bias)
    qd, kd, vd = (G.dev_bf16(x) for x in (q, k, v))
    assert _lib.lib().mi355_sage_set_attn_short(form) == 0
    try:
        if call == "stats":
            fwd = A.sdpa_flash_train_fwd(qd, kd, vd, scale, variant)
            got, stats = fwd.o.float().cpu().numpy(), fwd.stats.cpu().numpy()[..., 0]
        elif call == "range":
            got = A.sdpa_qwen_keymask(qd, kd, vd, hi, lo, scale, variant).float().cpu().numpy()
        else:
            got = A.sdpa_nomask(qd, kd, vd, scale, variant).float().cpu().numpy()
    finally:
        _lib.lib().mi355_sage_set_attn_short(0)
    _, want, want_stats = oracle.sdpa_bf16(q, k, v, scale, variant=variant, blkq=blkq, blkk=64, mask_lo=lo, mask_hi=hi, want_stats=True)
    assert np.isfinite(got).all()
    cos, mx = G.cos_maxabs(got, want)
    assert mx <= 2e-2 and cos >= 0.9999, (cos, mx)            # (the bars of every O test; seen: 0.012 and 0.999997)
    if call == "stats":
        np.testing.assert_allclose(stats, want_stats, atol=2e-3 if variant == 0 else 1e-2)
