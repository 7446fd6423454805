"""The attention kernel's workgroup sizes and schedules at the edges of their ranges, against the oracle's exact softmax with
the bounds of test_gpu_kernels.test_attention_vs_oracle (fp16 P and output rounding, about 3x the measured errors)."""
import numpy as np
import pytest

from oracle import hxo
from tests._helpers import f16, rel
from tests.test_gpu_kernels import _attn, _hip, say

pytestmark = pytest.mark.gpu


# 192 queries, three-phase (one round of them where 128-query workgroups would take two): 5 tiles, the last with 1 key, in 190
# ragged queries; 6 tiles, half 1 as long as half 0, 321 of 328 keys; whole tiles; 7 tiles over 385 queries (a third
# workgroup of one query); batch 2
# 128 queries, ping-pong over 3 and 5 tiles a half
# 64 queries, ping-pong: one query past a workgroup, an odd number of tiles a half
@pytest.mark.parametrize("T,NKV,nvalid,H,batch", [(190, 264, 257, 200, 1), (384, 328, 321, 100, 1), (384, 384, 384, 100, 1),
                                                  (385, 448, 430, 70, 1), (192, 320, 300, 100, 2), (1536, 384, 384, 16, 1),
                                                  (1100, 640, 640, 20, 1), (65, 640, 640, 3, 1), (192, 384, 384, 4, 2)])
def test_attention_forms(T, NKV, nvalid, H, batch):
    hip = _hip()
    say(f"attention form T={T} NKV={NKV} nvalid={nvalid} H={H} batch={batch}")
    rng = np.random.default_rng(T + NKV + H)
    D = 128 * H
    q = f16(rng.standard_normal((batch * T, D)) / np.sqrt(128) * 2.0)
    k = f16(rng.standard_normal((batch * NKV, D)))
    v = f16(rng.standard_normal((batch * NKV, D)))
    for b in range(batch):  # the scores of masked keys never count, whatever they are
        k[b * NKV + nvalid:(b + 1) * NKV] = np.float16(np.nan)
    got = _attn(hip, q, k, v, nvalid, batch)
    again = _attn(hip, q, k, v, nvalid, batch)
    assert np.array_equal(got.view(np.uint16), again.view(np.uint16))
    rows = np.unique(np.r_[np.arange(0, T, 13), T - 1])
    for b in range(batch):
        kb, vb = np.nan_to_num(k[b * NKV:(b + 1) * NKV]), v[b * NKV:(b + 1) * NKV]
        g = got[b * T:(b + 1) * T][rows].astype(np.float64)
        exact = hxo.attention(np.ascontiguousarray(q[b * T:(b + 1) * T][rows]), kb, vb, nvalid, mode=1)
        exact = exact.view(np.float16).astype(np.float64)
        assert np.max(np.abs(g - exact)) < 4e-3
        assert rel(g, exact) < 1e-3
