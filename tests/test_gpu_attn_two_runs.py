"""GPU tests of the main kernel's two-run form: 128 query rows per workgroup, the keys of a tile split over the two halves
of its waves, whose results meet in LDS at the end.  Against the CPU checker (max-abs 2e-2, cosine 0.9999, the bars of the
other forward tests) at key counts around a tile, where a run has few keys or none, and under every kind of mask."""
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
    # An e4m3 probability next to a rounding boundary may lie one step, 2^-3 of it, off the checker's: with n keys of N(0, 1)
    # scores the largest is below exp(3.5) / (n exp(0.5)) = 20 / n, and |v - o| below 4, so 10 / n.  The plain schedule
    # rounds it alike.
    bar = 2e-2 if variant == 0 else max(2e-2, 10.0 / Skv)
    _close(plain.float().cpu().numpy(), want, ("plain", Skv), bar)
    _close(fwd.o.float().cpu().numpy(), want, ("stats", Skv), bar)
    assert _lib.lib().mi355_sage_set_attn_short(-1) == 0
    whole = A.sdpa_cross_nomask(*dev, scale, variant)
    _close(plain.float().cpu().numpy(), whole.float().cpu().numpy(), ("against the plain schedule", Skv))
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


@pytest.mark.parametrize("variant,D,B,H,S,Skv", [(0, 128, 1, 80, 1000, 1500), (1, 128, 1, 80, 850, 1500), (0, 64, 1, 68, 1000, 1500), (1, 64, 1, 66, 1100, 1500)])
def test_behind_full_rounds_of_the_main_kernel(variant, D, B, H, S, Skv):
    """More row tiles than 256, the last of a head at most half full: the whole rounds keep the bits of the plain schedule,
    whatever form does the rest."""
    import torch
    import gpu_harness as G
    from mojodiffusion_amd import attention_sage as A
    L = _lib.lib()
    main = L.mi355_sage_attn_main_items(B, H, S, Skv, D, variant)
    assert main == 256 < B * H * ((S + 255) // 256)
    q, k, v = (G.dev_bf16(x) for x in _inputs(B, S, Skv, H, D, S))
    got = A.sdpa_flash_train_fwd_rect(q, k, v, D ** -0.5, variant)
    assert L.mi355_sage_set_attn_split(-1) == 0
    try:
        plain = A.sdpa_flash_train_fwd_rect(q, k, v, D ** -0.5, variant)
    finally:
        L.mi355_sage_set_attn_split(0)
    torch.cuda.synchronize()
    per_head = (S + 255) // 256
    tiles = lambda t: torch.nn.functional.pad(t.permute(0, 2, 1, 3).reshape(B * H, S, -1).float(), (0, 0, 0, per_head * 256 - S)).reshape(B * H * per_head, 256, -1)
    a, b = tiles(got.o), tiles(plain.o)
    assert torch.equal(a[:main], b[:main])
    _close(a[main:].cpu().numpy(), b[main:].cpu().numpy(), main)
    assert float((got.stats - plain.stats).abs().max()) <= (1e-4 if variant == 0 else 2e-2)
