"""GPU tests of the short form with the quantizers in it (one launch, fp16 P.V, up to 256 keys of 128 channels or 512 of
64): codes, scales and the order of every sum are those of the separate launches, so the results have their bits.  The
forced short form (8 or 4 key runs) goes through the separate launches."""
import pytest

from mojodiffusion_amd import _lib

pytestmark = pytest.mark.gpu


def _both(runs, call):
    import torch
    L = _lib.lib()
    one = call()
    assert L.mi355_sage_set_attn_short(runs) == 0
    try:
        apart = call()
    finally:
        L.mi355_sage_set_attn_short(0)
    torch.cuda.synchronize()
    for a, b in zip(one, apart):
        assert torch.isfinite(a.float()).all() and torch.equal(a, b), float((a.float() - b.float()).abs().max())


# (heads, queries) -> 8 key runs while there is a compute unit for every 32 rows, else 4
@pytest.mark.parametrize("H,Sq,runs", [(3, 1, 8), (2, 100, 8), (30, 256, 8), (60, 190, 4)])
@pytest.mark.parametrize("D,Skv", [(D, n) for D in (64, 128) for n in (1, 15, 16, 33, 64, 65, 127, 200, 255, 256)] + [(64, n) for n in (257, 400, 511, 512)])
def test_bits_of_the_separate_launches(D, Skv, H, Sq, runs):
    import torch
    from mojodiffusion_amd import attention_sage as A
    g = torch.Generator(device="cuda")
    g.manual_seed(Skv * 7 + Sq)
    q, k, v = (torch.randn((1, n, H, D), generator=g, device="cuda").to(torch.bfloat16) for n in (Sq, Skv, Skv))
    k += 3.0 * torch.randn((1, 1, H, D), generator=g, device="cuda").to(torch.bfloat16)
    bias = torch.randn((1, H, Sq, Skv), generator=g, device="cuda").to(torch.bfloat16)
    scale = D ** -0.5
    from test_abi_exports import attn_plan
    assert attn_plan(1, H, Sq, Skv, D, 0) == attn_plan(1, H, Sq, Skv, D, 0, bias=1) == "one launch"

    def call():
        fwd = A.sdpa_flash_train_fwd_rect(q, k, v, scale)
        out = [A.sdpa_cross_nomask(q, k, v, scale), fwd.o, fwd.stats, A.sdpa_cross_masked(q, k, v, bias, scale)]
        if Skv > 2 and Sq == 100:
            out.append(A.sdpa_qwen_keymask(k, k, v, Skv - 1, Skv // 3, scale))
        return out

    if Sq == 100 and Skv > 400:
        runs = 8
    _both(runs, call)


def test_values_that_take_the_careful_paths():
    """Infinities and NaN among K and V, values past fp16, rounding ties and a channel of zeros: as the separate launches."""
    import torch
    from mojodiffusion_amd import attention_sage as A
    L = _lib.lib()
    for D in (64, 128):
        g = torch.Generator(device="cuda")
        g.manual_seed(D)
        q, k, v = (torch.randn((1, 130, 4, D), generator=g, device="cuda").to(torch.bfloat16) for _ in range(3))
        k[:, :, 0] = (k[:, :, 0] * 8).round() / 8                     # many codes next to ties
        k[:, :, 1, 5] = 0.0
        v[0, 7, 2, 3] = float("inf")
        v[0, 9, 2, 4] = -1e30
        v[0, 11, 3, 1] = float("nan")
        k[0, 13, 3, 2] = 1e30
        one = A.sdpa_nomask(q, k, v, D ** -0.5)
        assert L.mi355_sage_set_attn_short(8) == 0
        try:
            apart = A.sdpa_nomask(q, k, v, D ** -0.5)
        finally:
            L.mi355_sage_set_attn_short(0)
        torch.cuda.synchronize()
        assert torch.equal(one.view(torch.int16), apart.view(torch.int16))
