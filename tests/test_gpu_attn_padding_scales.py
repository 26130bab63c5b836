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
