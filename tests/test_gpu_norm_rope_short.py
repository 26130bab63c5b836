"""RMSNorm + RoPE in front of short self-attention, whose quantizers take two launches where those of plain rows take one: bits of
the same call on rows normed and rotated before."""
import numpy as np
import pytest

import gpu_harness as H
from mojodiffusion_amd import attention_sage as A
from mojodiffusion_amd.workloads import f32_to_bf16_bits
from test_gpu_norm_rope import _gains, _tables

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", [A.PV_FP16, A.PV_FP8])
@pytest.mark.parametrize("D,S", [(64, 512), (64, 513), (64, 1024), (128, 256), (128, 257), (128, 512)])
def test_short_calls_with_pre_ops(oracle, D, S, variant):
    import torch
    B, Hh, eps, scale = 1, 3, 1e-6, float(D ** -0.5)
    rng = np.random.default_rng(S + D)
    q, k, v = (f32_to_bf16_bits(rng.standard_normal((B, S, Hh, D), dtype=np.float32)) for _ in range(3))
    gq, gk = _gains(rng, D)
    cos, sin = _tables(rng, S * Hh, D)
    got = A.qk_norm_rope_sdpa_nomask(*map(H.dev_bf16, (q, k, v, gq, gk)), eps, torch.from_numpy(cos).cuda(), torch.from_numpy(sin).cuda(), scale, variant)
    qn, kn = (oracle.norm_rope_bf16(x, g, eps, cos, sin, 0) for x, g in ((q, gq), (k, gk)))
    want = A.sdpa_nomask(*map(H.dev_bf16, (qn, kn, v)), scale, variant)
    np.testing.assert_array_equal(H.to_bits(got), H.to_bits(want))
