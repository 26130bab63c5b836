"""The additive bias at the edges of its chunks of eight keys and steps of 32: rows anywhere in memory with NaN between
them (nothing past a row's end is read into a result), biases of the type's lowest value, both forms of the kernel."""
import ctypes

import numpy as np
import pytest

from mojodiffusion_amd import _lib
from mojodiffusion_amd.workloads import WORKLOADS, make_inputs, bf16_bits_to_f32, f32_to_bf16_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", [-1, 4])
@pytest.mark.parametrize("variant,D,Sq,Skv,gap", [
    (0, 128, 33, 1, 0), (0, 128, 5, 7, 1), (0, 128, 257, 8, 3), (0, 64, 64, 9, 0), (0, 128, 40, 31, 2), (0, 64, 300, 33, 5),
    (0, 128, 65, 63, 8), (0, 128, 130, 65, 1), (0, 64, 31, 95, 0), (0, 128, 290, 577, 1), (0, 256, 70, 41, 1),
    (1, 128, 40, 7, 1), (1, 128, 130, 129, 0), (1, 64, 33, 333, 2)])
def test_bias_rows(oracle, form, variant, D, Sq, Skv, gap):
    import torch
    import gpu_harness as G
    w = WORKLOADS[1 if D == 64 else 2].scaled(B=2, H=2, S=max(Sq, Skv), D=D)
    q, k, v = make_inputs(w)
    q, k, v = (np.ascontiguousarray(x[:, :n]) for x, n in ((q, Sq), (k, Skv), (v, Skv)))
    rng = np.random.default_rng(Sq * Skv + D)
    bias = f32_to_bf16_bits(rng.standard_normal((w.B, w.H, Sq, Skv)).astype(np.float32) * 1.5)
    if Skv > 8:
        bias[..., 3:6] = 0xFF7F                              # the lowest finite bf16
        bias[0, :, :, :Skv - 2] = 0xFF7F                     # ... in everything but the last two keys
    row = Skv + gap
    wide = torch.full((w.B, w.H, Sq, row), float("nan"), dtype=torch.bfloat16, device="cuda")
    wide[..., :Skv] = G.dev_bf16(bias)
    qd, kd, vd = G.dev_bf16(q), G.dev_bf16(k), G.dev_bf16(v)
    o = torch.zeros_like(qd)
    L = _lib.lib()
    qs, ks = _lib.strides_bhnd(Sq, w.H, D), _lib.strides_bhnd(Skv, w.H, D)
    ms = (ctypes.c_int64 * 4)(w.H * Sq * row, Sq * row, row, 1)
    assert L.mi355_sage_set_attn_short(form) == 0
    try:
        rc = L.mi355_sage_sdpa_bf16_mask_any(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), wide.data_ptr(), o.data_ptr(), w.B, w.H, Sq, Skv, D,
                                             w.scale, qs, ks, ks, ms, qs, 0, 0, 0, 0, 0, G.stream(), variant, None, 0)
        torch.cuda.synchronize()
    finally:
        L.mi355_sage_set_attn_short(0)
    assert rc == 0, rc
    _, want = oracle.sdpa_bf16(q, k, v, w.scale, variant=variant, blkq=128 if variant == 0 else 32, blkk=64, addmask=bf16_bits_to_f32(bias))
    got = o.float().cpu().numpy()
    assert np.isfinite(got).all()
    cos, mx = G.cos_maxabs(got, want)
    assert mx <= 2e-2 and cos >= 0.9999, (cos, mx)            # (the bars of every O test: one bf16 step at |O| ~ 4)


@pytest.mark.parametrize("form", [-1, 4])
@pytest.mark.parametrize("variant,D,value", [(0, 128, -1e9), (0, 128, -2e38), (0, 64, -1e9), (0, 64, -1e30), (0, 256, -1e9), (1, 128, -1e9), (1, 64, -1e30)])
def test_bias_beyond_the_scores_precision(oracle, form, variant, D, value):
    """Whole steps of keys, and whole rows, at a bias whose rounding is larger than any score: such keys weigh nothing
    where a row has others, and are alike where it has none."""
    import torch
    import gpu_harness as G
    S = 290
    w = WORKLOADS[1 if D == 64 else 2].scaled(B=1, H=2, S=S, D=D)
    q, k, v = make_inputs(w)
    bias = np.zeros((w.B, w.H, S, S), np.float32)
    bias[:, 0, :, :130] = value                              # the first steps
    bias[:, 1, :, 70:] = value                               # the later ones
    bias[:, :, 40:75] = value                                # rows with nothing else
    bias = f32_to_bf16_bits(bias)
    qd, kd, vd, md = (G.dev_bf16(x) for x in (q, k, v, bias))
    o = torch.zeros_like(qd)
    L = _lib.lib()
    qs, ms = _lib.strides_bhnd(S, w.H, D), (ctypes.c_int64 * 4)(w.H * S * S, S * S, S, 1)
    assert L.mi355_sage_set_attn_short(form) == 0
    try:
        rc = L.mi355_sage_sdpa_bf16_mask_any(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), md.data_ptr(), o.data_ptr(), w.B, w.H, S, S, D,
                                             w.scale, qs, qs, qs, ms, qs, 0, 0, 0, 0, 0, G.stream(), variant, None, 0)
        torch.cuda.synchronize()
    finally:
        L.mi355_sage_set_attn_short(0)
    assert rc == 0, rc
    _, want = oracle.sdpa_bf16(q, k, v, w.scale, variant=variant, blkq=128 if variant == 0 else 32, blkk=64, addmask=bf16_bits_to_f32(bias))
    got = o.float().cpu().numpy()
    assert np.isfinite(got).all()
    cos, mx = G.cos_maxabs(got, want)
    assert mx <= 2e-2 and cos >= 0.9999, (cos, mx)            # (the bars of every O test: one bf16 step at |O| ~ 4)
