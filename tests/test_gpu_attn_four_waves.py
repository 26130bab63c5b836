"""GPU tests of the main kernel in workgroups of four waves (128 query rows, two workgroups to a compute unit): the loop and
the order of its sums are the eight-wave form's, so the results have its bits."""
import pytest

from mojodiffusion_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Sq,Skv", [(1, 1), (127, 31), (128, 64), (129, 65), (257, 190), (300, 333), (513, 700), (200, 1025)])
def test_bits_of_the_eight_wave_form(variant, D, Sq, Skv):
    import torch
    from mojodiffusion_amd import attention_sage as A
    L = _lib.lib()
    g = torch.Generator(device="cuda")
    g.manual_seed(Sq * 31 + Skv)
    q, k, v = (torch.randn((2, n, 3, D), generator=g, device="cuda").to(torch.bfloat16) for n in (Sq, Skv, Skv))
    scale = D ** -0.5
    got = {}
    for mode in (-1, 3):
        assert L.mi355_sage_set_attn_short(mode) == 0
        try:
            fwd = A.sdpa_flash_train_fwd_rect(q, k, v, scale, variant)
            got[mode] = [A.sdpa_cross_nomask(q, k, v, scale, variant), fwd.o, fwd.stats]
            if Skv > 2:
                got[mode].append(A.sdpa_qwen_keymask(k, k, v, Skv - 1, Skv // 3, scale, variant))
        finally:
            L.mi355_sage_set_attn_short(0)
    torch.cuda.synchronize()
    for a, b in zip(got[-1], got[3]):
        assert torch.isfinite(a.float()).all() and torch.equal(a, b)


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Sq,Skv", [(1, 77), (129, 129), (513, 700), (1100, 1100), (1025, 300)])
def test_causal_has_the_bits_of_the_eight_wave_form(variant, D, Sq, Skv):
    import numpy as np
    from mojodiffusion_amd.workloads import f32_to_bf16_bits
    from test_gpu_attn_causal import _causal_call
    L = _lib.lib()
    rng = np.random.default_rng(Sq + Skv)
    q, k, v = (f32_to_bf16_bits(rng.standard_normal((2, n, 3, D)).astype(np.float32)) for n in (Sq, Skv, Skv))
    got = {}
    for mode in (-1, 3):
        assert L.mi355_sage_set_attn_short(mode) == 0
        try:
            got[mode] = [_causal_call(q, k, v, float(D ** -0.5), variant, 128 if variant == 0 else 32, want_stats=w) for w in (False, True)]
        finally:
            L.mi355_sage_set_attn_short(0)
    for (a, sa), (b, sb) in zip(got[-1], got[3]):
        np.testing.assert_array_equal(a, b)
        if sa is not None:
            np.testing.assert_array_equal(sa, sb)


def test_a_shape_that_takes_it_by_itself(oracle):
    """Several rounds of few key tiles, against the checker: max-abs 2e-2, cosine 0.9999."""
    import numpy as np
    import gpu_harness as G
    from mojodiffusion_amd import attention_sage as A
    from mojodiffusion_amd.workloads import f32_to_bf16_bits
    from test_abi_exports import attn_plan
    assert attn_plan(1, 40, 2900, 333, 64, 0) == "four waves"
    rng = np.random.default_rng(3)
    q, k, v = (f32_to_bf16_bits(rng.standard_normal((1, n, 40, 64)).astype(np.float32)) for n in (2900, 333, 333))
    got = A.sdpa_cross_nomask(*(G.dev_bf16(x) for x in (q, k, v)), 0.125).float().cpu().numpy()
    _, want = oracle.sdpa_bf16(q, k, v, 0.125, variant=0, blkq=128, blkk=64)
    cos, mx = G.cos_maxabs(got, want)
    assert mx <= 2e-2 and cos >= 0.9999, (cos, mx)
