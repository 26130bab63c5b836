"""GPU test of the backward at 64 channels around the edges of its blocks: a workgroup owns 128 query rows or 128 keys,
32 to a wave, and walks the other side in tiles of 64.  Bars of the other backward tests."""
import pytest

from test_gpu_bwd import _check, _run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Sq,Skv", [(1, 127), (31, 128), (128, 129), (129, 64), (160, 255), (257, 65), (384, 1)])
def test_block_edges(oracle, Sq, Skv):
    for valid in ({}, {"real_q": (Sq + 1) // 2, "real_kv": (Skv + 2) // 3}):
        outs, want = _run_case(oracle, 1, Sq, Skv, 3, 64, 0.125, 40 + Sq, **valid)
        for name, got, ref in zip(("dQ", "dK", "dV"), outs, want):
            _check("%s %d %d %s" % (name, Sq, Skv, valid), got, ref)
