"""The backward of callers with F32 activations (mi355_sage_sdpa_bwd_f32_grads): dO in F32 and gradients in F32 are the bf16
call's, for dO rounded to bf16, value for value."""
import pytest

from mojodiffusion_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Sq,Skv,real_q,real_kv", [(1, 1, 0, 0), (63, 130, 0, 0), (257, 257, 200, 129), (300, 64, 128, 1)])
def test_f32_gradients_hold_the_bf16_values(D, Sq, Skv, real_q, real_kv):
    import torch
    import gpu_harness as H
    L = _lib.lib()
    B, Hh = 2, 3
    g = torch.Generator(device="cuda").manual_seed(Sq + D)
    normal = lambda *s: torch.randn(s, generator=g, device="cuda", dtype=torch.float32)
    q, o = normal(B, Sq, Hh, D).bfloat16(), normal(B, Sq, Hh, D).bfloat16()
    k, v = normal(B, Skv, Hh, D).bfloat16(), normal(B, Skv, Hh, D).bfloat16()
    d = normal(B, Sq, Hh, D)
    for i, x in enumerate((1.00390625, 1.01171875, -1.00390625, 1e-41, -0.0)):       # ties to even, a subnormal, a zero's sign
        d.view(-1)[i] = x
    if real_q:
        d[:, real_q:] = float("nan")                                                 # what stands in padding rows never counts
    d16 = d.bfloat16()
    stats = normal(B, Hh, Sq) * 0.1 + 4.0
    sq, sk = _lib.strides_bhnd(Sq, Hh, D), _lib.strides_bhnd(Skv, Hh, D)
    ws = torch.empty(max(L.mi355_sage_bwd_workspace_bytes(B, Hh, Sq, Skv, D), 256), dtype=torch.uint8, device="cuda")
    tail = lambda: ((B, Hh, Sq, Skv, D, D ** -0.5, sq, sk, sk, sq, sq, sq, sk, sk) + (0,) * 9 + (0, real_q, real_kv, H.stream(), ws.data_ptr(), ws.numel()))
    grads = lambda dt: [torch.full_like(t, 7.0, dtype=dt) for t in (q, k, v)]
    want, got = grads(torch.bfloat16), grads(torch.float32)
    ptr = lambda *ts: tuple(t.data_ptr() for t in ts)
    assert L.mi355_sage_sdpa_bwd_bf16(*ptr(q, k, v, o, d16, stats, *want), *tail()) == 0
    scratch = torch.full_like(d16, float("nan"))
    assert L.mi355_sage_sdpa_bwd_f32_grads(*ptr(q, k, v, o, d, scratch, stats, *got), *tail()) == 0
    torch.cuda.synchronize()
    for name, a, b in zip(("dq", "dk", "dv"), got, want):
        assert torch.isfinite(a).all() and torch.equal(a, b.float()), name
    n = real_q or Sq
    assert torch.equal(scratch[:, :n].view(torch.int16), d16[:, :n].view(torch.int16))
    assert L.mi355_sage_sdpa_bwd_f32_grads(*ptr(q, k, v, o, d), None, *ptr(stats, *got), *tail()) == -1
