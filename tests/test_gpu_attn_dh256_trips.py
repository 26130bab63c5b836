"""GPU tests of the main loop at 256 channels, whose trips run over rings of three (fp16 P.V) or four (e4m3) slots:
key counts around the first trips and their remainders, a masked range in front of, inside and behind a trip,
and the causal end.  Bars of the other forward tests: max-abs 2e-2 and cosine 0.9999 against the CPU checker."""
import numpy as np
import pytest

from mojodiffusion_amd import _lib
from mojodiffusion_amd.workloads import f32_to_bf16_bits

pytestmark = pytest.mark.gpu
D = 256


def _check(oracle, variant, Sq, Skv, lo=0, hi=0, seed=0):
    import torch
    import gpu_harness as G
    from mojodiffusion_amd import attention_sage as A
    rng = np.random.default_rng(seed)
    q, k, v = (f32_to_bf16_bits(rng.standard_normal((1, n, 2, D)).astype(np.float32)) for n in (Sq, Skv, Skv))
    scale = 1.0 / float(np.sqrt(D))
    qd, kd, vd = (G.dev_bf16(x) for x in (q, k, v))
    lib = _lib.lib()
    assert lib.mi355_sage_set_attn_short(-1) == 0
    try:
        if hi > lo:
            got = A.sdpa_qwen_keymask(qd, kd, vd, hi, lo, scale, variant)
        else:
            got = A.sdpa_cross_nomask(qd, kd, vd, scale, variant)
        torch.cuda.synchronize()
    finally:
        lib.mi355_sage_set_attn_short(0)
    _, want = oracle.sdpa_bf16(q, k, v, scale, variant=variant, blkq=128 if variant == 0 else 32, blkk=64, mask_lo=lo, mask_hi=hi)
    cos, mx = G.cos_maxabs(got.float().cpu().numpy(), want)
    assert mx <= 2e-2 and cos >= 0.9999, (variant, Sq, Skv, lo, hi, cos, mx)


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("tiles", range(3, 14))
def test_key_counts_around_the_trips(oracle, variant, tiles):
    for ragged in (0, 1, 33):
        _check(oracle, variant, 131, tiles * 64 - ragged, seed=tiles * 10 + ragged)


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("lo,hi", [(1, 70), (60, 500), (257, 259), (320, 704), (500, 1270), (1, 1279)])
def test_masked_range_around_the_trips(oracle, variant, lo, hi):
    _check(oracle, variant, 1280, 1280, lo, hi, seed=lo)


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("Sq,Skv", [(130, 130), (700, 700), (300, 1025), (1025, 300)])
def test_causal_end(oracle, variant, Sq, Skv):
    """Against the checker given the mask as a bias.  (e4m3: a probability next to a rounding boundary may lie 2^-3 of itself off the
    checker's, and in the first rows a key's probability is most of the row's: 2^-3 * 0.8 of |v - o| < 5, which leaves the cosine to
    hold the rest.)"""
    import gpu_harness as G
    from mojodiffusion_amd.workloads import bf16_bits_to_f32
    from test_gpu_attn_causal import _bias, _causal_call
    rng = np.random.default_rng(Sq + Skv)
    q, k, v = (f32_to_bf16_bits(rng.standard_normal((1, n, 2, D)).astype(np.float32)) for n in (Sq, Skv, Skv))
    lib = _lib.lib()
    assert lib.mi355_sage_set_attn_short(-1) == 0
    try:
        got, _ = _causal_call(q, k, v, float(D ** -0.5), variant, 128 if variant == 0 else 32)
    finally:
        lib.mi355_sage_set_attn_short(0)
    _, want = oracle.sdpa_bf16(q, k, v, float(D ** -0.5), variant=variant, blkq=128 if variant == 0 else 32, blkk=64, addmask=_bias(1, 2, Sq, Skv))
    cos, mx = G.cos_maxabs(bf16_bits_to_f32(got), want)
    assert mx <= (2e-2 if variant == 0 else 0.5) and cos >= 0.9999, (cos, mx)
