"""GPU tests of the attention kernel's short form (32 or 64 query rows per workgroup, keys split over its
waves, partial results merged in LDS), forced at the sizes where it can go wrong: fewer key steps than
waves, one step more than a multiple, row blocks with one row, lengths next to the tile sizes.  Bars as
for the other forms: max-abs <= 2e-2 against the CPU checker, cosine >= 0.999 against the fp32 referee."""
import numpy as np
import pytest

from mojodiffusion_amd import _lib
from mojodiffusion_amd.workloads import WORKLOADS, make_inputs, bf16_bits_to_f32

pytestmark = pytest.mark.gpu


@pytest.fixture
def short():
    L = _lib.lib()

    def set_mode(mode):
        assert L.mi355_sage_set_attn_short(mode) == 0
    yield set_mode
    L.mi355_sage_set_attn_short(0)


@pytest.mark.parametrize("variant,D,runs,Sq,Skv", [
    (0, 128, 8, 1, 1), (0, 128, 8, 33, 257), (0, 128, 4, 65, 129), (0, 128, 8, 300, 2049), (0, 64, 8, 31, 63), (0, 64, 4, 129, 513),
    (0, 256, 4, 33, 97), (0, 256, 4, 96, 640), (1, 128, 8, 32, 64), (1, 128, 4, 63, 577), (1, 64, 8, 257, 1000), (1, 256, 4, 40, 333)])
def test_short_form_against_checker_and_referee(oracle, short, variant, D, runs, Sq, Skv):
    """Plain (Q encoded by the kernel) and with Stats (Q encoded by the quantize stage): the same bits."""
    import torch
    import gpu_harness as H
    from mojodiffusion_amd import attention_sage as A
    w = WORKLOADS[1 if D == 64 else 2].scaled(B=2, H=3, S=max(Sq, Skv), D=D)
    q, k, v = make_inputs(w)
    q, k, v = (np.ascontiguousarray(x[:, :n]) for x, n in ((q, Sq), (k, Skv), (v, Skv)))
    qd, kd, vd = H.dev_bf16(q), H.dev_bf16(k), H.dev_bf16(v)
    short(runs)
    o = A.sdpa_cross_nomask(qd, kd, vd, w.scale, variant)
    fwd = A.sdpa_flash_train_fwd_rect(qd, kd, vd, w.scale, variant)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(H.to_bits(o), H.to_bits(fwd.o))
    got = o.float().cpu().numpy()
    _, want, stats = oracle.sdpa_bf16(q, k, v, w.scale, variant=variant, blkq=32 if variant else 128, blkk=64, want_stats=True)
    cos, mx = H.cos_maxabs(got, want)
    assert mx <= 2e-2 and cos >= 0.9999, (cos, mx)
    assert np.abs(fwd.stats.cpu().numpy()[..., 0] - stats).max() <= 2e-2
    ref = oracle.sdpa_f32(bf16_bits_to_f32(q), bf16_bits_to_f32(k), bf16_bits_to_f32(v), w.scale)
    assert H.cos_maxabs(got, ref)[0] >= 0.999


@pytest.mark.parametrize("variant,D,runs", [(0, 128, 8), (0, 64, 4), (1, 128, 4), (0, 256, 4)])
def test_short_form_masks_and_causal(oracle, short, variant, D, runs):
    """A masked key range that empties whole key runs, an additive mask, causal: against the checker."""
    import torch
    import gpu_harness as H
    from mojodiffusion_amd import attention_sage as A
    from test_gpu_attn_causal import _bias, _causal_call
    w = WORKLOADS[1 if D == 64 else 2].scaled(B=1, H=2, S=452, D=D)
    q, k, v = make_inputs(w)
    qd, kd, vd = H.dev_bf16(q), H.dev_bf16(k), H.dev_bf16(v)
    blkq = 32 if variant else 128
    bias = oracle.f32_to_bf16((np.random.default_rng(7).standard_normal((1, 2, 452, 452)) * 1.5).astype(np.float32))
    short(runs)
    keymask = A.sdpa_qwen_keymask(qd, kd, vd, 300, 3, w.scale, variant).float().cpu().numpy()
    added = A.sdpa(qd, kd, vd, H.dev_bf16(bias), w.scale, variant).float().cpu().numpy()
    causal = bf16_bits_to_f32(_causal_call(q, k, v, w.scale, variant, blkq)[0])
    for got, kw in ((keymask, dict(mask_lo=3, mask_hi=300)), (added, dict(addmask=oracle.bf16_to_f32(bias))),
                    (causal, dict(addmask=_bias(1, 2, 452, 452)))):
        _, want = oracle.sdpa_bf16(q, k, v, w.scale, variant=variant, blkq=blkq, blkk=64, **kw)
        cos, mx = H.cos_maxabs(got, want)
        assert mx <= 2e-2 and cos >= 0.9999, (kw.keys(), cos, mx)


@pytest.mark.parametrize("variant,D,B,H,Sq,Skv", [(0, 64, 1, 87, 600, 520), (0, 128, 3, 43, 300, 2000), (1, 128, 2, 65, 511, 700), (1, 64, 1, 89, 700, 1000)])
def test_full_rounds_by_the_main_kernel_and_the_rest_by_the_short_form(variant, D, B, H, Sq, Skv):
    """A few row tiles more than 256, the last tile of a head ragged (pieces of it empty): the tiles of the
    main kernel keep the bits of the plain schedule, the others agree with it to the rounding of the
    probabilities, Stats to 1e-4 (the same sums in another order; e4m3: 2^-4 of the largest probability left out of one)."""
    import torch
    import gpu_harness as G
    from mojodiffusion_amd import attention_sage as A
    L = _lib.lib()
    items, per_head = B * H * ((Sq + 255) // 256), (Sq + 255) // 256
    assert L.mi355_sage_attn_main_items(B, H, Sq, Skv, D, variant) == 256 < items
    w = WORKLOADS[1 if D == 64 else 2].scaled(B=B, H=H, S=max(Sq, Skv), D=D)
    from mojodiffusion_amd.workloads import device_inputs
    q, k, v = device_inputs(w, 3)
    q, k, v = q[:, :Sq].contiguous(), k[:, :Skv].contiguous(), v[:, :Skv].contiguous()
    o = A.sdpa_cross_nomask(q, k, v, w.scale, variant)
    fwd = A.sdpa_flash_train_fwd_rect(q, k, v, w.scale, variant)
    assert L.mi355_sage_set_attn_split(-1) == 0
    try:
        plain = A.sdpa_flash_train_fwd_rect(q, k, v, w.scale, variant)
    finally:
        L.mi355_sage_set_attn_split(0)
    torch.cuda.synchronize()
    assert torch.equal(o, fwd.o)
    tiles = lambda t: torch.nn.functional.pad(t.permute(0, 2, 1, 3).reshape(B * H, Sq, -1).float(), (0, 0, 0, per_head * 256 - Sq)).reshape(items, 256, -1)
    a, b = tiles(fwd.o), tiles(plain.o)
    assert torch.equal(a[:256], b[:256])
    # (e4m3 probabilities round alike whatever whole-number reference a wave holds: its bits may well agree)
    assert variant == 1 or not torch.equal(a[256:], b[256:])
    cos, mx = G.cos_maxabs(a[256:].cpu().numpy(), b[256:].cpu().numpy())
    assert cos >= 0.9999 and mx <= 2e-2, (cos, mx)
    assert float((fwd.stats - plain.stats).abs().max()) <= (1e-4 if variant == 0 else 2e-2)


def test_short_form_rule():
    """By shape: small problems take it, problems that fill the chip with 256-row workgroups do not; a
    forced schedule of those workgroups keeps it out."""
    from test_abi_exports import attn_plan
    L = _lib.lib()
    assert attn_plan(1, 30, 256, 256, 128, 0) == "one launch" and attn_plan(1, 8, 1024, 1024, 64, 0) == "short8"
    assert attn_plan(1, 1, 1, 1, 128, 1) in ("short4", "short8")
    assert not any("short" in attn_plan(*x) for x in ((1, 24, 4608, 4608, 128, 0), (2, 30, 1248, 1248, 128, 0)))
    assert L.mi355_sage_set_attn_split(-1) == 0
    try:
        assert attn_plan(1, 30, 256, 256, 128, 0) == attn_plan(1, 8, 1024, 1024, 64, 0) == "main"
    finally:
        L.mi355_sage_set_attn_split(0)
    assert L.mi355_sage_set_attn_short(5) == -1
