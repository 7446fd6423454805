"""The attention kernel's workgroup sizes and schedules at the edges of their ranges, against the oracle's exact softmax with
the bounds of test_gpu_kernels.test_attention_vs_oracle (fp16 P and output rounding, about 3x the measured errors)."""
import ctypes as C

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


@pytest.mark.parametrize("T", [2304, 2176])
def test_three_phase_attention_with_the_weight_touch(T):
    """An fp16 Anima block (below 4096 rows its self attention touches the weights that follow) of as many tokens as take one
    round of 192-query workgroups: after the attention stage, o equals, bit for bit, hxa_attention without the touch on the
    block's own q, k and v, and a sample of its rows the oracle's exact softmax. The weights it touches stay as they are."""
    from tests.test_gpu_block import make_anima_pack
    hip = _hip()
    say(f"three-phase attention with touch T={T}")
    L = hip.lib()
    rng = np.random.default_rng(T)
    D, F, DC, C_ = 2048, 256, 128, 64
    img, _, H = make_anima_pack(hip, rng, D, F, DC, 0)
    x = rng.standard_normal((T, D)).astype(np.float32)
    mod = (rng.standard_normal((9, D)) * 0.2).astype(np.float32)
    ang = np.arange(T)[:, None] * 10000.0 ** (-np.arange(64) / 64.0)[None, :]
    bufs = [hip.DeviceArray.from_numpy(a) for a in (img, f16(rng.standard_normal((C_, DC))), mod, np.cos(ang).astype(np.float32),
                                                    np.sin(ang).astype(np.float32))]
    d = hip.BlockDims(0, D, H, F, C_, DC, T, 1, T, 0, 0, 1)
    ws, dx = hip.block_ws(d), hip.DeviceArray.from_numpy(x)
    rec = hip.DeviceArray((1024, 4), np.uint64, zero=True)
    hip.check(L.hxa_clock_record(1, rec.ptr, 1024), "clock_record")
    try:
        hip.check(L.hxa_block_run(C.byref(d), bufs[0].ptr, dx.ptr, bufs[1].ptr, bufs[2].ptr, bufs[3].ptr, bufs[4].ptr, ws.ptr, 4,
                                  None, 0, None), "block_run")
        hip.sync()
    finally:
        L.hxa_clock_record(1, None, 0)
    assert np.count_nonzero(rec.numpy()[:, 0]) == -(-T // 192) * H  # the 192-query form
    (q, ldq), (k, ldk), (vt, ldvt), (o, ldo) = (hip.ws_buffer(d, ws, w) for w in (hip.WS_Q, hip.WS_K, hip.WS_VT, hip.WS_O))
    alone = hip.DeviceArray((T, D), np.float16)
    hip.check(L.hxa_attention(q, ldq, k, ldk, vt, ldvt, alone.ptr, D, T, T, T, H, 1, 0, 0, 0, 0, None), "attention")
    hip.sync()
    got = hip.read_ws(d, ws, hip.WS_O, T, D)
    assert np.array_equal(got.view(np.uint16), alone.numpy().view(np.uint16))
    qh, kh, vh = (hip.read_ws(d, ws, w, r, c) for w, r, c in ((hip.WS_Q, T, D), (hip.WS_K, T, D), (hip.WS_VT, D, T)))
    rows = np.unique(np.r_[np.arange(0, T, 97), T - 1])
    exact = hxo.attention(np.ascontiguousarray(qh[rows]), kh, np.ascontiguousarray(vh.T), T, mode=1).view(np.float16)
    assert rel(got[rows].astype(np.float64), exact.astype(np.float64)) < 1e-3
    assert np.array_equal(bufs[0].numpy(), img)


@pytest.mark.parametrize("lat_hw,wgs,alone", [((64, 32), 64, 128), ((64, 48), 96, 192)])
def test_attention_that_hosts_the_modulation_keeps_128_queries(lat_hw, wgs, alone, monkeypatch):
    """2B-class DiT at 512 and 768 tokens, batch 1: the self-attention launch that streams the next block's modulation runs in
    128-query workgroups (8 waves each, the CUs it leaves idle host the rows); with the modulation in its own launches
    (HXA_DIT_SIDE=0) in 64-query ones. Counted from the clock record each attention workgroup writes; the latents are the same
    bits either way."""
    hip = _hip()
    L = hip.lib()
    say(f"hosting attention lat {lat_hw}")
    rng = np.random.default_rng(12)
    lat = rng.standard_normal((1, 16) + lat_hw).astype(np.float32)
    ctx = rng.standard_normal((1, 256, 1024)).astype(np.float32)
    outs = []
    for side, want in (("1", wgs), ("0", alone)):
        monkeypatch.setenv("HXA_DIT_SIDE", side)
        rec = hip.DeviceArray((1024, 4), np.uint64, zero=True)
        bd = hip.BlockDims(0, 2048, 16, 8192, 256, 1024, 0, 1, 0, 0, 0, 1)
        cfg = hip.DitCfg(bd, 2, 16, lat_hw[0], lat_hw[1], 256, 0)
        p = C.c_void_p()
        hip.check(L.hxa_dit_create(C.byref(cfg), 77, C.byref(p)), "dit_create")
        try:
            hip.check(L.hxa_clock_record(1, rec.ptr, 1024), "clock_record")
            hip.check(L.hxa_dit_set_inputs(p, lat.ctypes.data, ctx.ctypes.data), "set_inputs")
            hip.check(L.hxa_dit_step(p, 1.0, 0.5, 1), "step")
            cur = np.zeros_like(lat)
            hip.check(L.hxa_dit_get_latent(p, cur.ctypes.data), "get")
        finally:
            L.hxa_clock_record(1, None, 0)
            L.hxa_dit_destroy(p)
        assert np.count_nonzero(rec.numpy()[:, 0]) == want
        outs.append(cur)
    assert np.abs(outs[0] - lat).max() > 0.1
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
