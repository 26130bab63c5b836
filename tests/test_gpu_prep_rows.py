"""K statistics behind the fused pre-ops: with more groups of 256 keys than compute units a wave takes sixteen rows in turn, with
fewer four times as many threads share them.  The same bits."""
import numpy as np
import pytest

from mojodiffusion_amd.workloads import f32_to_bf16_bits
from test_gpu_norm_rope import _gains, _gpu_quant, _tables

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,S,halfsplit,per_batch,full_row", [(1, 1793, False, False, False), (2, 1040, True, True, False), (3, 513, False, False, True)])
def test_statistics_of_many_and_of_few_groups(D, B, S, halfsplit, per_batch, full_row):
    rng = np.random.default_rng(S + D)
    Hh, rows = 48, -(-S // 256)
    assert B * Hh * rows > 256 >= Hh * rows // 2
    q, k = (f32_to_bf16_bits(rng.standard_normal((B, S, Hh, D), dtype=np.float32)) for _ in range(2))
    gq, gk = _gains(rng, D * Hh if full_row else D)
    tables = B if per_batch else 1
    cos, sin = _tables(rng, tables * S * Hh, D)
    many = _gpu_quant(q, k, D ** -0.5, 128, 64, True, gq, gk, 1e-6, cos, sin, S * Hh if per_batch else 0, halfsplit=halfsplit, full_row=full_row)
    # (few groups: one batch at a time, and half of its heads where the norm is a head's own)
    for b in range(B):
        for h in (slice(None),) if full_row else (slice(0, 24), slice(24, 48)):
            c, s = (np.ascontiguousarray(t.reshape(tables, S, Hh, D // 2)[b if per_batch else 0][:, h]).reshape(-1, D // 2) for t in (cos, sin))
            qb, kb = (np.ascontiguousarray(x[b:b + 1, :, h]) for x in (q, k))
            few = _gpu_quant(qb, kb, D ** -0.5, 128, 64, True, gq, gk, 1e-6, c, s, 0, halfsplit=halfsplit, full_row=full_row)
            for name in ("kmean", "kmul", "kscale", "k8"):
                np.testing.assert_array_equal(many[name][b:b + 1, h], few[name], err_msg=name)
