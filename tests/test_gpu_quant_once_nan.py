"""NaNs among the keys of a one-shot call whose quantize stage is one launch: the scale of every block is that of the values, whatever
the extremes of a leaf of 16 keys come to — a signaling NaN takes an extreme's place in v_min3 / v_max3 — so that the call gives the bits of
the stage entry points' launches, with K smoothing or balancing alone as well (with smoothing, a NaN's channel has no mean and counts for nothing)."""
import numpy as np
import pytest

import gpu_harness as H
from mojodiffusion_amd import _lib
from mojodiffusion_amd.workloads import f32_to_bf16_bits

pytestmark = pytest.mark.gpu


def _one_shot(q, k, v, scale, flags):
    import torch
    L = _lib.lib()
    B, S, Hh, D = q.shape
    st = _lib.strides_bhnd(S, Hh, D)
    x = [H.dev_bf16(t) for t in (q, k, v)]
    o = torch.zeros((B, S, Hh, D), dtype=torch.bfloat16, device="cuda")
    n = L.mi355_sage_workspace_bytes(B, Hh, S, S, D, 0)
    ws = torch.full((n,), 0xAB, dtype=torch.uint8, device="cuda")
    rc = L.mi355_sage_sdpa_bf16_ex(*(t.data_ptr() for t in x), o.data_ptr(), B, Hh, S, S, D, scale, st, st, st, st, 0, 0, 0, 0, 0, H.stream(),
                                   0, 128, 64, flags, ws.data_ptr(), n)
    assert rc == 0, rc
    torch.cuda.synchronize()
    return H.to_bits(o)


@pytest.mark.parametrize("nan", [0x7F81, 0xFFBF, 0x7FC0])               # signaling, signaling and negative, quiet
@pytest.mark.parametrize("flags", [_lib.K_BALANCE, _lib.K_SMOOTH, _lib.K_SMOOTH | _lib.K_BALANCE])
@pytest.mark.parametrize("D,Hh,S", [(128, 24, 1157), (64, 70, 709), (128, 4, 1157)])      # groups encoded by their workgroups (two), blocks apart
def test_scales_behind_a_nan(D, Hh, S, flags, nan):
    rng = np.random.default_rng(S + D)
    q, k, v = (f32_to_bf16_bits(rng.standard_normal((1, S, Hh, D), dtype=np.float32)) for _ in range(3))
    big, small = f32_to_bf16_bits(np.array([50.0, -50.0], np.float32))
    last = S // 16 * 16                     # the leaf that the end cuts
    for h, leaf in ((0, 32), (1, last)):
        k[0, leaf, h, 3], k[0, leaf + 1, h, 3], k[0, leaf + 2, h, 3] = big, small, nan       # (behind the extremes)
        k[0, leaf + 1, h, 4], k[0, leaf + 3, h, 4] = nan, big                                # (in front of one)
    k[0, last + 4, 2, 5] = nan
    scale = D ** -0.5
    qk = H.quant_qk(q, k, scale, 128, 64, bool(flags & _lib.K_SMOOTH), balance=bool(flags & _lib.K_BALANCE))["dev"]
    vq = H.quant_v(v, 0)["dev"]["vq"]
    want, _ = H.attn_fwd(qk["q8"], qk["qscale"], 128, qk["k8"], qk["kscale"], 64, vq, None, 0, S, S)
    got = _one_shot(q, k, v, scale, flags)
    np.testing.assert_array_equal(got, want)
