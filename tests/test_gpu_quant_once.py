"""The quantize stage as one launch whose workgroups hand their statistics to each other: the bits of the launches, in each
way it divides the work (K's blocks apart, K with its groups, fp16 V with them, heads in chunks), at ragged lengths, masked ranges and
pre-ops — and where no flag is ever raised, so that every workgroup computes what it waits for itself."""
import numpy as np
import pytest

import gpu_harness as H
from mojodiffusion_amd import _lib
from mojodiffusion_amd.workloads import f32_to_bf16_bits
from test_gpu_norm_rope import _gains, _gpu_quant, _tables

pytestmark = pytest.mark.gpu


def _once(q, k, v, scale, variant, blkq, mask, pre, polls):
    import torch
    L = _lib.lib()
    B, S, Hh, D = q.shape
    Skv = k.shape[1]
    st, sk = _lib.strides_bhnd(S, Hh, D), _lib.strides_bhnd(Skv, Hh, D)
    qd, kd, vd = H.dev_bf16(q), H.dev_bf16(k), H.dev_bf16(v)
    nqp, nkp = L.mi355_sage_pad_q(S), L.mi355_sage_pad_kv(Skv)
    out = dict(q8=torch.full((B, Hh, nqp, D), 77, dtype=torch.int8, device="cuda"), qscale=torch.full((B, Hh, nqp // blkq), -1.0, device="cuda"),
               k8=torch.full((B, Hh, nkp, D), 77, dtype=torch.int8, device="cuda"), kscale=torch.full((B, Hh, nkp // 64), -1.0, device="cuda"))
    for n in ("kmean", "qmul", "kmul"):
        out[n] = torch.full((B, Hh, D), -1.0, device="cuda")
    out["vq"] = torch.full((B, Hh, nkp // 64, D, 64), 0x7E, dtype=torch.int16 if variant == 0 else torch.uint8, device="cuda")
    out["vscale"] = torch.full((B, Hh, D), -1.0, device="cuda")
    groups = (Skv + 255) // 256
    scr = torch.full((L.mi355_sage_quant_scratch_bytes(B, Hh, Skv, D) + 16 * B * Hh * groups,), 0xAB, dtype=torch.uint8, device="cuda")
    p = [None, None, 0.0, None, None, 0]
    held = []
    if pre is not None:
        gq, gk, cos, sin, layout = pre
        held = [H.dev_bf16(gq), H.dev_bf16(gk), torch.from_numpy(cos).cuda(), torch.from_numpy(sin).cuda()]
        p = [held[0].data_ptr(), held[1].data_ptr(), 1e-6, held[2].data_ptr(), held[3].data_ptr(), layout]
    for _ in range(2):                    # (the second finds the first's flags in its scratch)
        rc = L.mi355_sage_quant_once(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), B, Hh, S, Skv, D, scale, st, sk, sk, variant, blkq, mask[0], mask[1],
                                     *p, *(t.data_ptr() for t in out.values()), scr.data_ptr(), scr.numel(), polls, H.stream())
        assert rc == 0, rc
    torch.cuda.synchronize()
    return {n: t.cpu().numpy() for n, t in out.items()}


@pytest.mark.parametrize("polls", [1024, -2])
@pytest.mark.parametrize("D,variant,B,Hh,Sq,Skv,mask,pre", [
    (128, 0, 1, 2, 1, 1, (0, 0), None), (64, 0, 1, 3, 257, 257, (0, 0), None), (128, 0, 2, 5, 700, 1153, (100, 400), None),       # K's blocks apart
    (64, 1, 1, 2, 63, 255, (0, 0), None), (128, 1, 2, 7, 300, 1300, (5, 900), None), (64, 1, 1, 3, 100, 8192, (0, 0), None),      # e4m3
    (128, 0, 1, 35, 130, 641, (0, 0), None), (64, 0, 1, 70, 64, 700, (17, 300), None),                                            # with the groups
    (128, 0, 1, 29, 64, 2305, (300, 900), None), (64, 0, 1, 90, 65, 600, (0, 0), None),                                           # V with them
    (64, 0, 1, 60, 64, 2310, (0, 0), None),                                                                                       # heads in chunks
    (128, 0, 1, 3, 513, 513, (0, 0), 0), (128, 0, 1, 3, 300, 300, (0, 0), 1), (64, 0, 2, 3, 1100, 1100, (0, 0), 0), (64, 1, 1, 2, 555, 555, (0, 0), 1),
    (128, 1, 1, 4, 800, 800, (0, 0), 0), (128, 0, 1, 66, 1025, 1025, (0, 0), 1)])
def test_same_bits_as_the_launches(D, variant, B, Hh, Sq, Skv, mask, pre, polls):
    rng = np.random.default_rng(Skv + D)
    q = f32_to_bf16_bits(rng.standard_normal((B, Sq, Hh, D), dtype=np.float32))
    k = f32_to_bf16_bits(rng.standard_normal((B, Skv, Hh, D), dtype=np.float32) + 3 * rng.standard_normal((B, 1, Hh, D)).astype(np.float32))
    v = f32_to_bf16_bits(rng.standard_normal((B, Skv, Hh, D), dtype=np.float32))
    blkq = 128 if variant == 0 else 32
    scale = D ** -0.5
    if pre is None:
        want = H.quant_qkv(q, k, v, scale, variant, blkq, 64, mask=mask)
        p = None
    else:
        gq, gk = _gains(rng, D)
        cos, sin = _tables(rng, Skv * Hh, D)
        p = (gq, gk, cos, sin, pre)
        want = _gpu_quant(q, k, scale, blkq, 64, True, gq, gk, 1e-6, cos, sin, 0, halfsplit=pre == 1)
        want.update({n: x for n, x in H.quant_v(v, variant).items() if n != "dev"})
    got = _once(q, k, v, scale, variant, blkq, mask, p, polls)
    for name in ("kmean", "kmul", "qmul", "kscale", "k8", "qscale", "q8") + (("vscale",) if variant == 1 else ()):
        np.testing.assert_array_equal(got[name].view(np.uint8), want[name].view(np.uint8), err_msg=name)
    np.testing.assert_array_equal(got["vq"].view(np.uint8), np.ascontiguousarray(want["vq"]).view(np.uint8), err_msg="vq")


def test_one_shot_calls_that_share_a_workspace():
    """Calls of several shapes in turn on one stream, whose flags lie over each other's workspace, eager and under capture."""
    import torch
    from mojodiffusion_amd import attention_sage as A
    torch.manual_seed(3)
    qkv = [[torch.randn(1, s, h, d, device="cuda").to(torch.bfloat16) for _ in range(3)] for s, h, d in ((1153, 24, 128), (1500, 12, 64), (2400, 30, 128), (600, 9, 128))]
    first = [A.sdpa_nomask(*x, x[0].shape[3] ** -0.5).clone() for x in qkv]
    torch.cuda.synchronize()
    for _ in range(20):
        outs = [A.sdpa_nomask(*x, x[0].shape[3] ** -0.5) for x in qkv]
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(first, outs))
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        captured = [A.sdpa_nomask(*x, x[0].shape[3] ** -0.5) for x in qkv]
    for _ in range(3):
        g.replay()
        A.sdpa_nomask(*qkv[0], 128 ** -0.5)
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(first, captured))


@pytest.mark.parametrize("D,variant,Hh,S", [(128, 0, 2, 700), (64, 0, 70, 700), (64, 1, 3, 600), (128, 0, 29, 2305)])
def test_non_finite_values_as_the_launches_take_them(D, variant, Hh, S):
    """Infinities and NaNs in single tokens, NaNs alone in a leaf's channel, and values whose distance to the mean is the largest there is."""
    rng = np.random.default_rng(S)
    q, k, v = (f32_to_bf16_bits(rng.standard_normal((1, S, Hh, D), dtype=np.float32)) for _ in range(3))
    k[0, 5, 0, 3] = 0x7F80
    k[0, 300, 1, 7] = 0xFF80
    k[0, 270, 0, 9] = 0x7FC0
    k[0, 272:288, 1, 11] = 0x7FC0
    k[0, 40, 1, 13], k[0, 41, 1, 13] = 0x7F7F, 0xFF7F
    v[0, 17, 0, 2], v[0, 18, 1, 2] = 0x7F80, 0x7FC0
    blkq = 128 if variant == 0 else 32
    want = H.quant_qkv(q, k, v, D ** -0.5, variant, blkq, 64)
    got = _once(q, k, v, D ** -0.5, variant, blkq, (0, 0), None, 1024)
    for name in ("kscale", "k8", "qscale", "q8", "vq"):
        np.testing.assert_array_equal(np.ascontiguousarray(got[name]).view(np.uint8), np.ascontiguousarray(want[name]).view(np.uint8), err_msg=name)
    for name in ("kmean", "kmul", "qmul"):
        np.testing.assert_array_equal(got[name], want[name], err_msg=name)          # (NaNs where there are NaNs)
