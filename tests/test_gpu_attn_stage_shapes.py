"""GPU tests of the attention stage's entry points where the choice of form meets their own arguments: key caches far longer
than the keys that count, and shapes around those that mi355_sage_attn_fwd_q16 leaves to the encoded-Q form."""
import pytest

from mojodiffusion_amd import _lib

pytestmark = pytest.mark.gpu


def _operands(H, Sq, Skv, D, variant, seed):
    """Random codes and scales in the device layouts, one batch."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    nq, nkv = -(-Sq // 256) * 256, -(-Skv // 128) * 128
    codes = lambda n: torch.randint(-127, 128, (1, H, n, D), generator=g, device="cuda", dtype=torch.int32).to(torch.int8)
    scales = lambda n: 0.008 + 0.002 * torch.rand((1, H, n), generator=g, device="cuda")
    if variant == 0:
        v, vs = torch.randn((1, H, nkv // 64, D, 64), generator=g, device="cuda").half(), None
    else:
        v = torch.randint(0, 0x70, (1, H, nkv // 64, D, 64), generator=g, device="cuda", dtype=torch.int32).to(torch.uint8)
        vs = torch.rand((1, H, D), generator=g, device="cuda") + 0.5
    return dict(q8=codes(nq), qs=scales(nq // 32), k8=codes(nkv), ks=scales(nkv // 64), v=v, vs=vs)


def _attn(x, Sq, Skv, kv_valid, variant, mask=(0, 0)):
    import torch
    import gpu_harness as G
    _, H, _, D = x["q8"].shape
    o = torch.zeros((1, Sq, H, D), dtype=torch.bfloat16, device="cuda")
    stats = torch.zeros((1, H, Sq), device="cuda")
    rc = _lib.lib().mi355_sage_attn_fwd(x["q8"].data_ptr(), x["qs"].data_ptr(), 32, x["k8"].data_ptr(), x["ks"].data_ptr(), 64, x["v"].data_ptr(),
                                        x["vs"].data_ptr() if variant else None, variant, 1, H, Sq, Skv, kv_valid, mask[0], mask[1], D,
                                        o.data_ptr(), _lib.strides_bhnd(Sq, H, D), 0, None, stats.data_ptr(), G.stream())
    assert rc == 0, rc
    torch.cuda.synchronize()
    return o, stats


# (mode 0: two runs, the main kernel's rounds and the rest, four waves, the short form; then every form at a few heads)
@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("mode,H,Sq,kv", [(0, 24, 1153, 1153), (0, 24, 4000, 2000), (0, 40, 2379, 333), (0, 4, 300, 300),
                                          (2, 2, 130, 65), (2, 2, 257, 1000), (3, 2, 257, 1000), (-1, 2, 257, 1000)])
def test_cache_past_the_keys_that_two_runs_and_four_waves_stage(variant, D, mode, H, Sq, kv):
    """A cache of 33 000 keys of which kv count has the bits of one that ends with them."""
    import torch
    cache = 33000
    x = _operands(H, Sq, cache, D, variant, kv + H)
    n = -(-kv // 128) * 128
    tight = dict(x, k8=x["k8"][:, :, :n].contiguous(), ks=x["ks"][:, :, :n // 64].contiguous(), v=x["v"][:, :, :n // 64].contiguous())
    L = _lib.lib()
    assert L.mi355_sage_set_attn_short(mode) == 0
    try:
        for mask in ((0, 0), (kv // 3, kv // 2)):
            for a, b in zip(_attn(x, Sq, cache, kv, variant, mask), _attn(tight, Sq, kv, kv, variant, mask)):
                assert torch.isfinite(a.float()).all() and torch.equal(a, b), mask
    finally:
        L.mi355_sage_set_attn_short(0)


@pytest.mark.parametrize("B,H,Sq,Skv,D,taken", [(3, 64, 257, 1770, 64, True), (4, 40, 311, 1084, 64, True), (3, 64, 285, 872, 64, True),
                                                (1, 33, 2048, 2048, 128, False)])
def test_shapes_that_the_stage_with_q_in_the_kernel_takes(B, H, Sq, Skv, D, taken):
    """Considered by the split schedule: taken where the short form is ahead of it and of the main kernel by the figures for
    all lengths, with the bits of the stage on encoded Q."""
    import numpy as np
    import gpu_harness as G
    if _lib.lib().mi355_sage_attn_split_rule(B, H, Sq, Skv, D, 0) == 0:
        pytest.skip("not a shape of the split schedule on this device")
    rng = np.random.default_rng(Sq)
    q, k, v = ((rng.standard_normal((B, n, H, D)).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16) for n in (Sq, Skv, Skv))
    g, gv = G.quant_qk(q, k, D ** -0.5, 128, 64, True)["dev"], G.quant_v(v, 0)["dev"]
    rc, got = G.attn_fwd_q16(q, g["qmul"], 128, g["k8"], g["kscale"], 64, gv["vq"], None, 0, Skv)
    assert rc == (0 if taken else -2)
    if taken:
        want, _ = G.attn_fwd(g["q8"], g["qscale"], 128, g["k8"], g["kscale"], 64, gv["vq"], None, 0, Sq, Skv)
        np.testing.assert_array_equal(got, want)
