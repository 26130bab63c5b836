"""GPU test: the scale entries of blocks without a row or key that counts — rows past N_q, the second half of the last 128
keys, blocks inside a masked range — are read by the attention kernel and must not matter.  (The quantizers write
1 there, far above any real scale; the e4m3 kernel takes steps outside its main loop for waves with very large scales.)"""
import numpy as np
import pytest

from mojodiffusion_amd.workloads import WORKLOADS, make_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("wid,Sq,Skv,mask", [(2, 300, 700, (0, 0)), (1, 1000, 1090, (0, 0)), (2, 1000, 1090, (128, 512)), (1, 270, 1280, (64, 200))])
def test_scales_of_padding_do_not_matter(variant, wid, Sq, Skv, mask):
    import torch
    import gpu_harness as H
    from mojodiffusion_amd import _lib
    w = WORKLOADS[wid].scaled(B=1, H=2, S=Skv)
    q, k, v = make_inputs(w)
    q = np.ascontiguousarray(q[:, :Sq])
    blkq = 128 if variant == 0 else 32
    g = H.quant_qk(q, k, w.scale, blkq, 64, True, mask=mask)["dev"]
    gv = H.quant_v(v, variant, mask=mask)["dev"]
    L = _lib.lib()
    assert L.mi355_sage_set_attn_split(-1) == 0             # the main kernel, whatever the size
    try:
        out = []
        for value in (1.0, 1e-6):
            qs, ks = g["qscale"].clone(), g["kscale"].clone()
            qs[..., (Sq + blkq - 1) // blkq:] = value
            ks[..., (Skv + 63) // 64:] = value
            ks[..., (mask[0] + 63) // 64:mask[1] // 64] = value
            out.append(H.attn_fwd(g["q8"], qs, blkq, g["k8"], ks, 64, gv["vq"], gv.get("vscale"), variant, Sq, Skv, mask=mask)[0])
    finally:
        L.mi355_sage_set_attn_split(0)
    assert torch.isfinite(torch.from_numpy(out[0].astype(np.int32) << 16).view(torch.float32)).all()
    np.testing.assert_array_equal(out[0], out[1])


@pytest.mark.parametrize("variant,D", [(1, 64), (1, 128), (1, 256), (0, 128)])
@pytest.mark.parametrize("kv_valid", [1, 64, 100, 128, 150, 300, 449, 577])
def test_nothing_past_the_last_key_matters(oracle, variant, D, kv_valid):
    """One to ten key tiles, odd and even, of operands that go on behind them: V of the tiles behind as NaN, their scales as
    NaN.  The main kernel's bits are those of operands that end there; both meet the checker's bar."""
    import torch
    import gpu_harness as H
    from mojodiffusion_amd import _lib
    from mojodiffusion_amd.workloads import bf16_bits_to_f32
    w = WORKLOADS[2].scaled(B=1, H=2, S=640)
    Sq, blkq = 300, 128 if variant == 0 else 32
    rng = np.random.default_rng(kv_valid + D)
    q, k, v = (np.ascontiguousarray((rng.standard_normal((1, n, 2, D)).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16))
               for n in (Sq, kv_valid, kv_valid))
    scale = D ** -0.5
    g = H.quant_qk(q, k, scale, blkq, 64, True)["dev"]
    gv = H.quant_v(v, variant)["dev"]
    n = (kv_valid + 63) // 64                                       # key tiles that hold a key
    k8 = torch.full((1, 2, 640, D), 99, dtype=torch.int8, device="cuda")
    k8[:, :, :n * 64] = g["k8"][:, :, :n * 64]
    ks = torch.full((1, 2, 10), float("nan"), device="cuda")
    ks[..., :n] = g["kscale"][..., :n]
    vq = torch.full((1, 2, 10, D, 64), 0x7E00 if variant == 0 else 0x7F, dtype=gv["vq"].dtype, device="cuda")
    vq[:, :, :n] = gv["vq"].view(1, 2, -1, D, 64)[:, :, :n]
    L = _lib.lib()
    assert L.mi355_sage_set_attn_split(-1) == 0                     # the main kernel, whatever the size
    try:
        want, ws = H.attn_fwd(g["q8"], g["qscale"], blkq, g["k8"], g["kscale"], 64, gv["vq"], gv.get("vscale"), variant, Sq, kv_valid, want_stats=True)
        got, gs = H.attn_fwd(g["q8"], g["qscale"], blkq, k8, ks, 64, vq, gv.get("vscale"), variant, Sq, 640, kv_valid=kv_valid, want_stats=True)
    finally:
        L.mi355_sage_set_attn_split(0)
    np.testing.assert_array_equal(got, want)
    np.testing.assert_array_equal(gs, ws)
    _, ref = oracle.sdpa_bf16(q, k, v, scale, variant=variant, blkq=blkq, blkk=64)
    assert np.isfinite(bf16_bits_to_f32(got)).all() and np.abs(bf16_bits_to_f32(got) - ref).max() <= 2e-2


@pytest.mark.parametrize("form", ["main", "short"])
@pytest.mark.parametrize("variant,D", [(0, 64), (0, 128), (1, 64), (1, 128), (1, 256)])
@pytest.mark.parametrize("Skv", [192, 256, 300])
def test_score_scales_that_underflow_to_zero(form, variant, D, Skv):
    """Inputs so small that the score scale is zero in F32: every key counts alike, and a masked score (-inf) times that
    scale must not become NaN.  The result is the mean of V over the keys; V is within 1, so 2e-2 bounds its
    storage (e4m3: 2^-4 relative, averaged) and the rounding of O."""
    import torch
    from mojodiffusion_amd import _lib, model_dispatch as M
    g = torch.Generator().manual_seed(Skv + D)
    q, k = (1e-25 * torch.randn((1, n, 2, D), generator=g) for n in (300, Skv))
    v = torch.rand((1, Skv, 2, D), generator=g).bfloat16()
    L = _lib.lib()
    assert L.mi355_sage_set_attn_split(-1 if form == "main" else 0) == 0
    assert L.mi355_sage_set_attn_short(0 if form == "main" else 4) == 0
    try:
        o = M.ltx2_sdpa_product_fwd_rect(q.bfloat16().cuda(), k.bfloat16().cuda(), v.cuda(), D ** -0.5, variant)
    finally:
        L.mi355_sage_set_attn_split(0)
        L.mi355_sage_set_attn_short(0)
    want = v.double().mean(dim=1, keepdim=True)
    assert float((o.cpu().double() - want).abs().max()) <= 2e-2
