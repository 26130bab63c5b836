"""The encoders that add up the group results themselves against the form with a launch for it, at the lengths where
one gives way to the other (8 groups of 256 keys with e4m3 V, 10 otherwise), and both against the CPU checker."""
import numpy as np
import pytest

import gpu_harness as H
from mojodiffusion_amd.workloads import WORKLOADS, make_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,variant,S,mask", [
    (64, 1, 1025, (0, 0)), (128, 1, 2048, (0, 0)), (128, 1, 2049, (100, 900)), (64, 1, 2560, (0, 0)), (64, 0, 2560, (0, 0)),
    (64, 0, 2561, (0, 0)), (128, 0, 1281, (5, 1000)), (256, 0, 2049, (0, 0)), (256, 1, 2049, (0, 0))])
def test_both_forms_have_the_checker_s_bits(oracle, D, variant, S, mask):
    w = WORKLOADS[1 if D == 64 else 2].scaled(B=1, H=2, S=S, D=D)
    q, k, v = make_inputs(w)
    blkq = 128 if variant == 0 else 32
    got = H.quant_qkv(q, k, v, w.scale, variant, blkq, 64, mask=mask)
    alone, vv = H.quant_qk(q, k, w.scale, blkq, 64, True, mask=mask), H.quant_v(v, variant, mask=mask)      # (between 8 and 10 groups: the other form)
    for name in ("q8", "qscale", "k8", "kscale", "kmean", "qmul", "kmul"):
        np.testing.assert_array_equal(got[name], alone[name], err_msg=name)
    np.testing.assert_array_equal(got["vq"], vv["vq"])
    if variant == 1:
        np.testing.assert_array_equal(got["vscale"], vv["vscale"])
    if mask == (0, 0):
        want = H.oracle_quant_qk(oracle, q, k, w.scale, blkq, 64, True, True)
        for name in ("kmean", "qmul", "kmul"):
            np.testing.assert_array_equal(got[name].view(np.uint32), want[name].view(np.uint32), err_msg=name)
        for name in ("q8", "k8"):
            np.testing.assert_array_equal(got[name], want[name], err_msg=name)
