"""GPU tests of one-shot calls whose output lies over an input: O written over Q, K or V has the bits of O in memory of its own,
in the form that quantizes K and V itself, in those that encode Q themselves and in those that do neither."""
import pytest

from mojodiffusion_amd import _lib

pytestmark = pytest.mark.gpu


# (one launch with eight and four runs; the short form, two runs, the main kernel, four waves; 256 channels)
@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("D,H,S", [(128, 30, 256), (128, 60, 190), (64, 8, 512), (64, 3, 33), (128, 8, 700), (64, 24, 1000), (128, 40, 1100), (128, 30, 2304),
                                   (64, 40, 1600), (256, 4, 300), (256, 30, 1200)])
@pytest.mark.parametrize("over", ["q", "k", "v", "shifted"])
def test_output_over_an_input(variant, D, H, S, over):
    import torch
    import gpu_harness as G
    L = _lib.lib()
    g = torch.Generator(device="cuda").manual_seed(S + D)
    mem = torch.randn((3 * S + 16, H, D), generator=g, device="cuda").bfloat16()
    st, row = _lib.strides_bhnd(S, H, D), H * D
    at = {"q": 0, "k": S, "v": 2 * S}
    want_o = {"shifted": S // 2}.get(over, at.get(over)) * row          # (shifted: over parts of Q and of K)
    own = torch.zeros((S, H, D), dtype=torch.bfloat16, device="cuda")

    def call(base, out, out_off, stats):
        p = base.data_ptr()
        a = (p, p, p, out.data_ptr())
        b = (1, H, S, S, D, float(D ** -0.5), st, st, st, st, 0, S * row, 2 * S * row, out_off)
        if stats is None:
            return L.mi355_sage_sdpa_bf16(*a, *b, 0, G.stream(), variant, None, 0)
        return L.mi355_sage_sdpa_bf16_train_fwd(*a, stats.data_ptr(), *b, 0, 0, 0, 0, G.stream(), variant, None, 0)

    for with_stats in (False, True):
        stats = [torch.zeros((1, H, S, 1), device="cuda") if with_stats else None for _ in range(2)]
        assert call(mem, own, 0, stats[0]) == 0
        there = mem.clone()
        assert call(there, there, want_o, stats[1]) == 0
        torch.cuda.synchronize()
        got = there.view(-1)[want_o:want_o + S * row].view(S, H, D)
        assert torch.isfinite(own.float()).all() and torch.equal(got, own), with_stats
        assert not with_stats or torch.equal(stats[0], stats[1])
        rest = torch.cat([there.view(-1)[:want_o], there.view(-1)[want_o + S * row:]])
        assert torch.equal(rest, torch.cat([mem.view(-1)[:want_o], mem.view(-1)[want_o + S * row:]]))
