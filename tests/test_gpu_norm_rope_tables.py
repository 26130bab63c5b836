"""Every layout of the rotation tables through the fused quantizers, at lengths on and next to the edges of a leaf
(16 tokens), a group (256) and a block: bits of the unfused pipeline."""
import numpy as np
import pytest

import gpu_harness as H
from mojodiffusion_amd.workloads import f32_to_bf16_bits
from test_gpu_norm_rope import _gains, _gpu_quant

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("full_row", [False, True])
@pytest.mark.parametrize("layout", ["none", "pairs_f32", "pairs_bf16", "half_f32", "half_bf16"])
@pytest.mark.parametrize("S", [1, 17, 255, 257])
def test_table_layouts_bit_exact(oracle, D, full_row, layout, S):
    rng = np.random.default_rng(S + D)
    B, Hh, eps, scale = 2, 3, 1e-6, float(D ** -0.5)
    q = f32_to_bf16_bits(rng.standard_normal((B, S, Hh, D)).astype(np.float32) * 2.0)
    k = f32_to_bf16_bits((rng.standard_normal((B, S, Hh, D)) + 1.5 * rng.standard_normal((B, 1, Hh, D))).astype(np.float32))
    q[1, S // 2] = 0                                           # an all-zero token
    gq, gk = _gains(rng, D * Hh if full_row else D)
    cos = sin = None
    if layout != "none":
        th = rng.uniform(-np.pi, np.pi, (S * Hh, D // 2))
        cos, sin = np.cos(th).astype(np.float32), np.sin(th).astype(np.float32)
        if layout.endswith("bf16"):
            cos, sin = f32_to_bf16_bits(cos), f32_to_bf16_bits(sin)
    half = layout.startswith("half")
    got = _gpu_quant(q, k, scale, 128, 64, True, gq, gk, eps, cos, sin, 0, halfsplit=half, full_row=full_row)
    qn, kn = (oracle.norm_rope_bf16(x, g, eps, cos, sin, 0, halfsplit=half, full_row=full_row) for x, g in ((q, gq), (k, gk)))
    want = H.oracle_quant_qk(oracle, qn, kn, scale, 128, 64, True, True)
    for name in ("kmean", "qmul", "kmul"):
        np.testing.assert_array_equal(got[name].view(np.uint32), want[name].view(np.uint32), err_msg=name)
    for name in ("qscale", "kscale"):
        n = want[name].shape[2]
        np.testing.assert_array_equal(got[name][:, :, :n].view(np.uint32), want[name].view(np.uint32), err_msg=name)
    for name in ("q8", "k8"):
        np.testing.assert_array_equal(got[name], want[name], err_msg=name)
