"""GPU test of the masked key range in the main kernel's loop: key tiles inside the range are left out (in pairs),
the main loop stops in front of the range and goes on behind it.  Ranges at the start, across tile and trip
boundaries, of less than a tile, of nearly everything, up to the ragged end; 256-row workgroups forced, and the
form the shape takes by itself.  Bar: max-abs 2e-2 against the CPU checker given the same range."""
import numpy as np
import pytest

from mojodiffusion_amd import _lib
from mojodiffusion_amd.workloads import WORKLOADS, make_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant,D", [(0, 128), (1, 128), (0, 64), (0, 256)])
def test_masked_ranges(oracle, variant, D):
    import torch
    import gpu_harness as H
    from mojodiffusion_amd import attention_sage as A
    S = 1530
    w = WORKLOADS[1 if D == 64 else 2].scaled(B=1, H=2, S=S, D=D)
    q, k, v = make_inputs(w)
    qd, kd, vd = H.dev_bf16(q), H.dev_bf16(k), H.dev_bf16(v)
    L = _lib.lib()
    for lo, hi in ((0, 64), (0, 1400), (1, 130), (130, 520), (500, 501), (640, 768), (64, 1441), (1300, S), (700, 1280)):
        _, want = oracle.sdpa_bf16(q, k, v, w.scale, variant=variant, blkq=32 if variant else 128, blkk=64, mask_lo=lo, mask_hi=hi)
        try:
            for mode in (-1, 0):
                assert L.mi355_sage_set_attn_split(mode) == 0
                got = A.sdpa_qwen_keymask(qd, kd, vd, hi, lo, w.scale, variant)
                torch.cuda.synchronize()
                g = got.float().cpu().numpy()
                assert np.isfinite(g).all(), (lo, hi, mode)
                cos, mx = H.cos_maxabs(g, want)
                assert cos >= 0.9999 and mx <= 2e-2, (lo, hi, mode, cos, mx)
        finally:
            L.mi355_sage_set_attn_split(0)
