"""GPU tests of the main kernel's two-run form: 128 query rows per workgroup, the keys of a tile split over the two halves
of its waves, whose results meet in LDS at the end.  Against the CPU checker (max-abs 2e-2, cosine 0.9999, the bars of the
other forward tests) at key counts around a tile, where a run has few keys or none, and under every kind of mask: a range, a
bias, causal."""
import numpy as np
import pytest

from mojodiffusion_amd import _lib
from mojodiffusion_amd.workloads import f32_to_bf16_bits

pytestmark = pytest.mark.gpu


@pytest.fixture
def two_runs():
    L = _lib.lib()
    assert L.mi355_sage_set_attn_short(2) == 0
    yield
    L.mi355_sage_set_attn_short(0)


def _inputs(B, Sq, Skv, H, D, seed):
    rng = np.random.default_rng(seed)
    return [f32_to_bf16_bits(rng.standard_normal((B, n, H, D)).astype(np.float32)) for n in (Sq, Skv, Skv)]


def _close(got, want, what, bar=2e-2):
    import gpu_harness as G
    cos, mx = G.cos_maxabs(got, want)
    assert mx <= bar and cos >= 0.9999, (what, cos, mx)


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Skv", [1, 32, 33, 64, 65, 127, 129, 256, 320, 385, 700, 1025])
def test_key_counts(oracle, two_runs, variant, D, Skv):
    import torch
    import gpu_harness as G
    from mojodiffusion_amd import attention_sage as A
    Sq, scale = 129 + Skv % 3 * 64, float(D ** -0.5)
    q, k, v = _inputs(2, Sq, Skv, 3, D, 7 * Skv + D)
    dev = [G.dev_bf16(x) for x in (q, k, v)]
    plain = A.sdpa_cross_nomask(*dev, scale, variant)
    fwd = A.sdpa_flash_train_fwd_rect(*dev, scale, variant)
    torch.cuda.synchronize()
    _, want, stats = oracle.sdpa_bf16(q, k, v, scale, variant=variant, blkq=128 if variant == 0 else 32, blkk=64, want_stats=True)
    # An e4m3 probability next to a rounding boundary may lie one step, 2^-3 of it, off the checker's.  A key's share of the row
    # moves the output by its probability times |v - o|, below 4 + 1; of n keys of N(0, 1) scores the largest has below
    # exp(3.5) / (n exp(0.5)) = 20 / n of the row, or all but a fifth of it where that bounds nothing; one key has all of it, exactly.
    bar = 2e-2 if variant == 0 or Skv == 1 else max(2e-2, 0.125 * 5.0 * min(0.8, 20.0 / Skv))
    _close(plain.float().cpu().numpy(), want, ("plain", Skv), bar)
    _close(fwd.o.float().cpu().numpy(), want, ("stats", Skv), bar)
    # (the plain schedule rounds alike)
    assert _lib.lib().mi355_sage_set_attn_short(-1) == 0
    whole, whole_fwd = A.sdpa_cross_nomask(*dev, scale, variant), A.sdpa_flash_train_fwd_rect(*dev, scale, variant)
    for what, a, b in (("plain", plain, whole), ("stats", fwd.o, whole_fwd.o)):
        _close(a.float().cpu().numpy(), b.float().cpu().numpy(), ("against the plain schedule", what, Skv))
    np.testing.assert_allclose(fwd.stats.cpu().numpy()[..., 0], stats, atol=2e-3 if variant == 0 else 2e-2)


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("S,lo,hi", [(333, 3, 300), (700, 0, 64), (1025, 120, 1000), (200, 32, 64)])
def test_masks(oracle, two_runs, variant, D, S, lo, hi):
    import gpu_harness as G
    from mojodiffusion_amd import attention_sage as A
    q, k, v = _inputs(1, S, S, 2, D, S + D)
    scale, blkq = float(D ** -0.5), 128 if variant == 0 else 32
    qd, kd, vd = (G.dev_bf16(x) for x in (q, k, v))
    got = A.sdpa_qwen_keymask(qd, kd, vd, hi, lo, scale, variant).float().cpu().numpy()
    _close(got, oracle.sdpa_bf16(q, k, v, scale, variant=variant, blkq=blkq, blkk=64, mask_lo=lo, mask_hi=hi)[1], "range")
    bias = f32_to_bf16_bits((1.5 * np.random.default_rng(S).standard_normal((1, 2, S, S))).astype(np.float32))
    got = A.sdpa(qd, kd, vd, G.dev_bf16(bias), scale, variant).float().cpu().numpy()
    _close(got, oracle.sdpa_bf16(q, k, v, scale, variant=variant, blkq=blkq, blkk=64, addmask=oracle.bf16_to_f32(bias))[1], "bias")


# (lengths on either side of a row block and of a trip, more keys than queries and fewer)
@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Sq,Skv", [(1, 77), (129, 129), (700, 700), (1100, 1100), (300, 1025), (1025, 300)])
def test_causal(oracle, two_runs, variant, D, Sq, Skv):
    from mojodiffusion_amd.workloads import bf16_bits_to_f32
    from test_gpu_attn_causal import _bias, _causal_call
    q, k, v = _inputs(1, Sq, Skv, 2, D, Sq + Skv + D)
    scale, blkq = float(D ** -0.5), 128 if variant == 0 else 32
    got = [_causal_call(q, k, v, scale, variant, blkq, want_stats=w) for w in (False, True)]
    assert _lib.lib().mi355_sage_set_attn_short(-1) == 0
    plain, plain_stats = _causal_call(q, k, v, scale, variant, blkq, want_stats=True)
    _, want, stats = oracle.sdpa_bf16(q, k, v, scale, variant=variant, blkq=blkq, blkk=64, addmask=_bias(1, 2, Sq, Skv), want_stats=True)
    for o, st in got:
        _close(bf16_bits_to_f32(o), want, "checker", 2e-2 if variant == 0 else 0.125 * 5.0 * 0.8)      # (see test_key_counts: rows of a few keys)
        _close(bf16_bits_to_f32(o), bf16_bits_to_f32(plain), "against the plain schedule")
        if st is not None:
            np.testing.assert_allclose(st, plain_stats, atol=1e-4 if variant == 0 else 2e-2)
            np.testing.assert_allclose(st, stats, atol=2e-3 if variant == 0 else 2e-2)


# (fp16 P.V at 64 channels gives what is left of a round to four waves or the short form up to 3072 keys)
@pytest.mark.parametrize("variant,D,B,H,S,Skv", [(0, 128, 1, 84, 900, 900), (0, 128, 1, 66, 1100, 1100), (1, 128, 1, 88, 900, 900), (1, 128, 1, 66, 1200, 1000),
                                                 (1, 64, 1, 66, 1100, 1100), (1, 64, 1, 84, 900, 1000), (0, 64, 2, 82, 300, 3200)])
def test_behind_full_rounds_of_the_main_kernel(variant, D, B, H, S, Skv):
    """More row tiles than 256, the last of a head at most half full (its second piece is empty) or not: the whole rounds keep the
    bits of the plain schedule, the two-run form does the rest.  Q from the encoders (Stats), Q in the kernel, and a masked
    range."""
    import torch
    import gpu_harness as G
    from mojodiffusion_amd import attention_sage as A
    from test_abi_exports import attn_plan
    L = _lib.lib()
    per_head, lo, hi = (S + 255) // 256, Skv // 4, Skv // 4 + Skv // 3
    assert attn_plan(B, H, S, Skv, D, variant) == "main + two runs"
    q, k, v = (G.dev_bf16(x) for x in _inputs(B, S, Skv, H, D, S))
    ranged = S == Skv and attn_plan(B, H, S, S, D, variant, masked=hi - lo) == "main + two runs"
    assert ranged or S != Skv

    def calls():
        fwd = A.sdpa_flash_train_fwd_rect(q, k, v, D ** -0.5, variant)
        return [fwd.o, A.sdpa_cross_nomask(q, k, v, D ** -0.5, variant)] + ([A.sdpa_qwen_keymask(q, k, v, hi, lo, D ** -0.5, variant)] if ranged else []), fwd.stats

    got, stats = calls()
    assert L.mi355_sage_set_attn_split(-1) == 0
    try:
        plain, plain_stats = calls()
    finally:
        L.mi355_sage_set_attn_split(0)
    torch.cuda.synchronize()
    tiles = lambda t: torch.nn.functional.pad(t.permute(0, 2, 1, 3).reshape(B * H, S, -1).float(), (0, 0, 0, per_head * 256 - S)).reshape(B * H * per_head, 256, -1)
    main = B * H * per_head // 256 * 256
    for x, y in zip(got, plain):
        a, b = tiles(x), tiles(y)
        assert torch.equal(a[:main], b[:main])
        _close(a[main:].cpu().numpy(), b[main:].cpu().numpy(), main)
    assert torch.equal(got[0], got[1])
    assert float((stats - plain_stats).abs().max()) <= (1e-4 if variant == 0 else 2e-2)
