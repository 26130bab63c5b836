"""The waits of the one-launch quantize stage: each run by itself leaves the bits of the launches, in buffers that hold something else
before — handed over with no group computed twice, with a single look before a workgroup computes what is missing, and where no flag is
ever raised — and calls of all kinds on two streams at once, and under capture, give the bits they give alone."""
import numpy as np
import pytest

import gpu_harness as H
from mojodiffusion_amd import _lib
from mojodiffusion_amd.workloads import f32_to_bf16_bits
from test_gpu_norm_rope import _gains, _gpu_quant, _tables

pytestmark = pytest.mark.gpu


class Stage:
    """mi355_sage_quant_once on buffers that are kept from run to run."""

    def __init__(self, q, k, v, variant, blkq, mask, pre):
        import torch
        L = self.L = _lib.lib()
        self.B, self.S, self.Hh, self.D = B, S, Hh, D = q.shape
        self.Skv, self.variant, self.blkq, self.mask = k.shape[1], variant, blkq, mask
        self.groups, self.words = (self.Skv + 255) // 256, (self.Skv + 255) // 256 * (2 if variant else 1)
        self.x = [H.dev_bf16(t) for t in (q, k, v)]
        nqp, self.nkp = L.mi355_sage_pad_q(S), L.mi355_sage_pad_kv(self.Skv)
        self.nq_blk = nqp // blkq
        shapes = dict(q8=((B, Hh, nqp, D), torch.int8), qscale=((B, Hh, self.nq_blk), torch.float32), k8=((B, Hh, self.nkp, D), torch.int8),
                      kscale=((B, Hh, self.nkp // 64), torch.float32), kmean=((B, Hh, D), torch.float32), qmul=((B, Hh, D), torch.float32),
                      kmul=((B, Hh, D), torch.float32), vq=((B, Hh, self.nkp // 64, D, 64), torch.uint8 if variant else torch.int16),
                      vscale=((B, Hh, D), torch.float32))
        self.out = {n: torch.empty(s, dtype=t, device="cuda") for n, (s, t) in shapes.items()}
        self.data_bytes = L.mi355_sage_quant_scratch_bytes(B, Hh, self.Skv, D)
        self.scr = torch.full((self.data_bytes + 16 * B * Hh * self.groups,), 0xAB, dtype=torch.uint8, device="cuda")
        self.pre, self.held = [None, None, 0.0, None, None, 0], []
        if pre is not None:
            gq, gk, cos, sin, layout = pre
            self.held = [H.dev_bf16(gq), H.dev_bf16(gk), torch.from_numpy(cos).cuda(), torch.from_numpy(sin).cuda()]
            self.pre = [self.held[0].data_ptr(), self.held[1].data_ptr(), 1e-6, self.held[2].data_ptr(), self.held[3].data_ptr(), layout]
        self.k_apart = pre is None and variant == 0 and self.groups * B * Hh * D <= 100 * 128

    def run(self, polls, fill):
        """One launch on outputs and group results that hold `fill`; the flags stay as the last run left them."""
        import torch
        L, D = self.L, self.D
        for t in self.out.values():
            t.view(torch.uint8).fill_(fill)
        self.scr[:self.data_bytes].fill_(fill)
        torch.cuda.synchronize()
        L.mi355_sage_quant_once_helps(1)
        st, sk = _lib.strides_bhnd(self.S, self.Hh, D), _lib.strides_bhnd(self.Skv, self.Hh, D)
        rc = L.mi355_sage_quant_once(*(t.data_ptr() for t in self.x), self.B, self.Hh, self.S, self.Skv, D, D ** -0.5, st, sk, sk, self.variant, self.blkq,
                                     *self.mask, *self.pre, *(t.data_ptr() for t in self.out.values()), self.scr.data_ptr(), self.scr.numel(), polls, H.stream())
        assert rc == 0, rc
        torch.cuda.synchronize()
        return {n: t.cpu().numpy() for n, t in self.out.items()}, L.mi355_sage_quant_once_helps(1)

    def flags(self):
        n = self.B * self.Hh * self.words
        return self.scr[self.data_bytes:self.data_bytes + 8 * n].cpu().numpy().view(np.uint64)

    def helps_without_flags(self):
        """Every workgroup that waits computes all groups of its head."""
        waiting = (self.nkp // 64 if self.k_apart else self.groups) + self.nq_blk + (self.groups if self.variant else 0)
        return self.B * self.Hh * waiting * self.groups


def _inputs(B, Hh, Sq, Skv, D):
    rng = np.random.default_rng(Skv + D)
    q = f32_to_bf16_bits(rng.standard_normal((B, Sq, Hh, D), dtype=np.float32))
    k = f32_to_bf16_bits(rng.standard_normal((B, Skv, Hh, D), dtype=np.float32) + 3 * rng.standard_normal((B, 1, Hh, D)).astype(np.float32))
    v = f32_to_bf16_bits(rng.standard_normal((B, Skv, Hh, D), dtype=np.float32))
    return rng, q, k, v


def _by_launches(rng, q, k, v, variant, blkq, mask, pre):
    """The launches' results, and the pre-ops' operands."""
    D = q.shape[3]
    if pre is None:
        return H.quant_qkv(q, k, v, D ** -0.5, variant, blkq, 64, mask=mask), None
    gq, gk = _gains(rng, D)
    cos, sin = _tables(rng, k.shape[1] * k.shape[2], D)
    want = _gpu_quant(q, k, D ** -0.5, blkq, 64, True, gq, gk, 1e-6, cos, sin, 0, halfsplit=pre == 1)
    want.update({n: x for n, x in H.quant_v(v, variant).items() if n != "dev"})
    return want, (gq, gk, cos, sin, pre)


def _same(got, want, variant, bits=True):
    for name in ("k8", "kscale", "q8", "qscale", "vq") + (("vscale",) if variant else ()):
        np.testing.assert_array_equal(np.ascontiguousarray(got[name]).view(np.uint8), np.ascontiguousarray(want[name]).view(np.uint8), err_msg=name)
    for name in ("kmean", "kmul", "qmul"):
        if bits:
            np.testing.assert_array_equal(got[name].view(np.uint32), want[name].view(np.uint32), err_msg=name)
        else:
            np.testing.assert_array_equal(got[name], want[name], err_msg=name)          # (NaNs where there are NaNs)


SHAPES = [
    (128, 0, 2, 5, 700, 1153, (100, 400), None), (64, 0, 1, 3, 257, 257, (0, 0), None),                     # K's blocks apart
    (64, 1, 1, 3, 100, 8192, (0, 0), None), (128, 1, 2, 7, 300, 1300, (5, 900), None),                      # e4m3
    (128, 0, 1, 35, 130, 641, (0, 0), None), (64, 0, 1, 90, 65, 600, (0, 0), None),                         # with the groups, V with them too
    (64, 0, 1, 60, 64, 2310, (0, 0), None),                                                                 # heads in chunks
    (128, 0, 1, 3, 513, 513, (0, 0), 0), (64, 1, 1, 2, 555, 555, (0, 0), 1), (128, 1, 1, 4, 800, 800, (0, 0), 0), (128, 0, 1, 66, 1025, 1025, (0, 0), 1)]


@pytest.mark.parametrize("D,variant,B,Hh,Sq,Skv,mask,pre", SHAPES)
def test_each_run_by_itself(D, variant, B, Hh, Sq, Skv, mask, pre):
    rng, q, k, v = _inputs(B, Hh, Sq, Skv, D)
    blkq = 128 if variant == 0 else 32
    want, p = _by_launches(rng, q, k, v, variant, blkq, mask, pre)
    s = Stage(q, k, v, variant, blkq, mask, p)
    before = s.flags().copy()
    got, helps = s.run(-2, 0x55)
    _same(got, want, variant)
    assert helps == s.helps_without_flags()
    np.testing.assert_array_equal(s.flags(), before)
    tags = {int(before[0])}
    for polls, fill in ((1024, 0x5A), (1024, 0xC3), (1, 0x3C), (1, 0xA5)):        # (each finds the flags of the one in front)
        got, helps = s.run(polls, fill)
        _same(got, want, variant)
        flags = s.flags()
        assert (flags == flags[0]).all() and int(flags[0]) not in tags
        tags.add(int(flags[0]))
        assert helps == 0 if polls > 1 else helps < s.helps_without_flags()


@pytest.mark.parametrize("D,variant,Hh,S,pre", [(128, 0, 3, 700, 0), (64, 0, 3, 1100, 1), (64, 1, 3, 600, 0), (128, 1, 3, 600, 1)])
def test_non_finite_values_behind_the_pre_ops(D, variant, Hh, S, pre):
    rng, q, k, v = _inputs(1, Hh, S, S, D)
    k[0, 5, 0, 3], k[0, 300, 1, 7], k[0, 270, 0, 9], k[0, 17, 2, 1] = 0x7F80, 0xFF80, 0x7FC0, 0x7F81
    k[0, 40, 1, 13], k[0, 41, 1, 13] = 0x7F7F, 0xFF7F
    q[0, 9, 0, 4], q[0, 130, 1, 4], q[0, 131, 2, 4] = 0x7F80, 0x7FC0, 0xFF81
    v[0, 17, 0, 2], v[0, 18, 1, 2], v[0, 19, 2, 2] = 0x7F80, 0x7FC0, 0x7F81
    blkq = 128 if variant == 0 else 32
    want, p = _by_launches(rng, q, k, v, variant, blkq, (0, 0), pre)
    s = Stage(q, k, v, variant, blkq, (0, 0), p)
    for polls in (1024, -1):
        _same(s.run(polls, 0x5A)[0], want, variant, bits=False)


def _calls():
    """One-shot calls of the forms the stage has, as functions of no arguments that return their output."""
    import torch
    from mojodiffusion_amd import attention_sage as A
    g = torch.Generator(device="cuda")
    g.manual_seed(11)
    rand = lambda *s: torch.randn(s, generator=g, device="cuda").to(torch.bfloat16)
    calls = []
    for S, Hh, D, variant in ((1153, 24, 128, A.PV_FP16), (1500, 12, 64, A.PV_FP16), (2400, 30, 128, A.PV_FP8), (4608, 24, 128, A.PV_FP16), (1000, 16, 64, A.PV_FP8)):
        x = [rand(1, S, Hh, D) for _ in range(3)]
        calls.append(lambda x=x, D=D, variant=variant: A.sdpa_nomask(*x, D ** -0.5, variant))
    for S, Hh, D, variant in ((1100, 24, 128, A.PV_FP16), (1300, 30, 64, A.PV_FP8), (2050, 30, 128, A.PV_FP8)):
        x = [rand(1, S, Hh, D) for _ in range(3)]
        gains = [rand(D) for _ in range(2)]
        tables = [torch.rand((S * Hh, D // 2), generator=g, device="cuda") for _ in range(2)]
        calls.append(lambda x=x, gains=gains, tables=tables, D=D, variant=variant: A.qk_norm_rope_sdpa_nomask(*x, *gains, 1e-6, *tables, D ** -0.5, variant))
    return calls


def test_one_workspace_for_calls_of_all_kinds():
    """In turn on one stream, whose flags and group results lie over each other's workspace, eager and in a graph's replays."""
    import torch
    calls = _calls()
    g = torch.cuda.CUDAGraph()
    first = [f().clone() for f in calls]
    with torch.cuda.graph(g):
        captured = [f() for f in calls]
    for turn in range(6):
        outs = [f() for f in (calls if turn % 2 else calls[::-1])]
        for o, want in zip(outs if turn % 2 else outs[::-1], first):
            assert torch.equal(o, want)
        g.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(o, want) for o, want in zip(captured, first))


def test_calls_on_two_streams_at_once():
    """One stream holds the chip with calls of many workgroups while the other's wait for each other."""
    import torch
    from mojodiffusion_amd import attention_sage as A
    calls = _calls()
    large = [torch.randn(1, 8192, 24, 128, device="cuda").to(torch.bfloat16) for _ in range(3)]
    alone = [f().clone() for f in calls]
    large_alone = A.sdpa_nomask(*large, 128 ** -0.5)
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    outs, larges = [], []
    for _ in range(4):
        with torch.cuda.stream(streams[0]):
            larges += [A.sdpa_nomask(*large, 128 ** -0.5) for _ in range(2)]
            outs.append([f() for f in calls])
        with torch.cuda.stream(streams[1]):
            outs.append([f() for f in calls])
    torch.cuda.synchronize()
    assert all(torch.equal(o, large_alone) for o in larges)
    for got in outs:
        assert all(torch.equal(a, b) for a, b in zip(got, alone))
