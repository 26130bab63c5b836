"""Encoders with interleaved rotation tables of 16 MiB and more (32 for one batch in Q blocks below 128 rows) deal their blocks in sets that read the same table rows: the same bits as
fewer heads at a time, whose tables are smaller and whose blocks go in the order of the heads."""
import numpy as np
import pytest

from mojodiffusion_amd.workloads import f32_to_bf16_bits
from test_gpu_norm_rope import _gains, _gpu_quant, _tables

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,S,blkq,blkk,per_batch,bf16", [(1, 1801, 128, 64, False, False), (2, 1801, 128, 64, False, False), (2, 897, 128, 64, True, False),
                                                          (3, 1700, 32, 64, False, False), (1, 6700, 64, 128, False, True)])
def test_blocks_in_sets_give_the_same_bits(B, S, blkq, blkk, per_batch, bf16):
    D, Hh, part = 128, 20, 4
    rng = np.random.default_rng(S)
    q, k = (f32_to_bf16_bits(rng.standard_normal((B, S, Hh, D), dtype=np.float32)) for _ in range(2))
    gq, gk = _gains(rng, D)
    batches = B if per_batch else 1
    cos, sin = _tables(rng, batches * S * Hh, D)
    if bf16:
        cos, sin = f32_to_bf16_bits(cos), f32_to_bf16_bits(sin)
    assert cos.nbytes + sin.nbytes >= (32 if B == 1 and blkq < 128 else 16) << 20
    run = lambda x, y, c, s, h: _gpu_quant(x, y, D ** -0.5, blkq, blkk, True, gq, gk, 1e-6, c, s, S * h if per_batch else 0)
    got = run(q, k, cos, sin, Hh)
    by_head = [t.reshape(batches, S, Hh, D // 2) for t in (cos, sin)]
    for h in range(0, Hh, part):
        c, s = (np.ascontiguousarray(t[:, :, h:h + part]).reshape(-1, D // 2) for t in by_head)
        assert c.nbytes + s.nbytes < 16 << 20
        want = run(np.ascontiguousarray(q[:, :, h:h + part]), np.ascontiguousarray(k[:, :, h:h + part]), c, s, part)
        for name in ("kmean", "qmul", "kmul", "qscale", "kscale", "q8", "k8"):
            np.testing.assert_array_equal(got[name][:, h:h + part], want[name], err_msg="%s, heads from %d" % (name, h))
