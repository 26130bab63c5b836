"""The backward's three-slot ring of tiles and its row-wise loads and stores, where they can go wrong: one to
five tiles on the walked side, lengths on and next to the tile edges, workgroups whose owner rows are all padding."""
import pytest

from test_gpu_bwd import _check, _run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Sq,Skv,rq,rk", [
    (1, 1, 0, 0), (63, 65, 0, 0), (64, 129, 0, 0), (65, 192, 0, 0), (129, 64, 0, 0), (193, 257, 0, 0), (257, 320, 0, 0),
    (300, 300, 1, 1),              # the second workgroup of either kind owns padding only
    (520, 400, 256, 128),          # ... and the valid lengths end on a workgroup's edge
    (130, 700, 129, 513),
])
def test_ring_and_padding_owners(oracle, D, Sq, Skv, rq, rk):
    outs, want = _run_case(oracle, 2, Sq, Skv, 3, D, float(D ** -0.5), seed=7 * Sq + Skv, real_q=rq, real_kv=rk)
    for name, got, ref in zip(("dQ", "dK", "dV"), outs, want):
        _check("%s %s" % (name, (Sq, Skv, D, rq, rk)), got, ref)
    if rq:
        assert not outs[0][:, rq:].float().abs().max().item()
    if rk:
        assert not outs[1][:, rk:].float().abs().max().item() and not outs[2][:, rk:].float().abs().max().item()
