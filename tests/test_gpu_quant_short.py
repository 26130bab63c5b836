"""GPU test of the one-launch quantizer (short key sequences): every code, scale and statistic has the bits of
the stage entry points that take three launches whatever the length (mi355_sage_quant_qk_bf16, _quant_v_f16,
_quant_v_fp8), which are bit-exact against the CPU checker.  Lengths on and next to the leaf (16), tile (64),
padding (128) and group (256) sizes and at the longest sequence that takes one launch; a masked key range."""
import numpy as np
import pytest

from mojodiffusion_amd.workloads import WORKLOADS, make_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,variant,Sq,Skv,blkq,blkk,mask,encode_q", [
    (64, 0, 1, 1, 128, 64, (0, 0), True), (64, 1, 65, 1024, 32, 64, (0, 0), True), (64, 0, 300, 769, 64, 32, (10, 700), True),
    (128, 0, 130, 17, 128, 128, (0, 0), True), (128, 1, 77, 255, 32, 64, (3, 40), True), (128, 0, 256, 512, 128, 64, (256, 512), False),
    (128, 1, 33, 257, 128, 128, (0, 0), False), (256, 0, 100, 256, 128, 64, (0, 0), True), (256, 1, 40, 129, 32, 128, (1, 100), True)])
def test_one_launch_quantizer_has_the_bits_of_the_stage_calls(D, variant, Sq, Skv, blkq, blkk, mask, encode_q):
    import gpu_harness as H
    w = WORKLOADS[1 if D == 64 else 2].scaled(B=2, H=3, S=max(Sq, Skv), D=D)
    q, k, v = make_inputs(w)
    q, k, v = (np.ascontiguousarray(x[:, :n]) for x, n in ((q, Sq), (k, Skv), (v, Skv)))
    got = H.quant_qkv(q, k, v, w.scale, variant, blkq, blkk, mask=mask, encode_q=encode_q)
    qk, vv = H.quant_qk(q, k, w.scale, blkq, blkk, True, mask=mask), H.quant_v(v, variant, mask=mask)
    for name in ("k8", "kscale", "kmean", "qmul", "kmul") + (("q8", "qscale") if encode_q else ()):
        np.testing.assert_array_equal(got[name], qk[name], err_msg=name)
    np.testing.assert_array_equal(got["vq"], vv["vq"])
    if variant == 1:
        np.testing.assert_array_equal(got["vscale"], vv["vscale"])
