"""The GEMM kernels at the sizes where their pipelines can go wrong: odd numbers of 32-k groups, fewer stages than the ring
holds, ragged rows and columns; the launches that must not depend on timing. Tolerance: assert_gemm_close (one fp16 ulp plus
the fp32 accumulation-order error, tests/_helpers.py)."""
import ctypes as C

import numpy as np
import pytest

from oracle import hxo
from tests._helpers import assert_gemm_close, f16, ulp_diff
from tests.test_gpu_kernels import _hip, _q4a_weights, _run_gemm, say

pytestmark = pytest.mark.gpu


def _weights(rng, fmt, asym, N, K):
    wf = (rng.standard_normal((N, K)) * 0.05).astype(np.float32)
    if fmt == 0:
        return f16(wf), None, None, f16(wf).view(np.uint16)
    if asym:
        q, s, z = _q4a_weights(rng, N, K)
        return q, s, z, hxo.q4_dequant(q, s, z)
    q, s = hxo.q8_quantize(wf) if fmt == 1 else hxo.q4_quantize(wf)
    return q, s, None, hxo.q8_dequant(q, s) if fmt == 1 else hxo.q4_dequant(q, s)


FORMATS = [(0, False), (1, False), (2, False), (2, True)]


@pytest.mark.parametrize("fmt,asym", FORMATS)
@pytest.mark.parametrize("K", [32, 64, 96, 160, 288, 352])
def test_every_tile_at_odd_and_short_k(K, fmt, asym):
    """One and few 32-k groups, odd and even (stage 0 of an odd count pairs its group with zeros), ragged in M and N: the
    128x128 tile against the oracle, every other tile equal to it bit for bit (one k order)."""
    hip = _hip()
    say(f"tiles fmt={fmt} asym={asym} K={K}")
    rng = np.random.default_rng(500 + K + 7 * fmt + asym)
    M, N = 272, 392
    A = f16(rng.standard_normal((M, K)))
    q, s, z, wdq = _weights(rng, fmt, asym, N, K)
    tiles = [(128, 128, 4), (256, 256, 9), (192, 256, 9), (256, 192, 9), (192, 192, 4), (128, 256, 9), (256, 128, 4),
             (192, 128, 8), (64, 128, 4), (64, 64, 4)] + ([(128, 64, 4)] if fmt != 2 else [])
    base = _run_gemm(hip, A, fmt, q, s, N, K, tile=tiles[0], z=z)
    assert_gemm_close(base, hxo.gemm(A, wdq), A, np.asarray(wdq).view(np.float16))
    for t in tiles[1:]:
        got = _run_gemm(hip, A, fmt, q, s, N, K, tile=t, z=z)
        assert np.array_equal(got.view(np.uint16), base.view(np.uint16)), t


@pytest.mark.parametrize("fmt,asym", FORMATS)
@pytest.mark.parametrize("tile", [(256, 192, 9), (192, 192, 4), (64, 128, 4), (64, 64, 4)])
def test_split_k_of_odd_slices(tile, fmt, asym):
    """Split-K partials whose slices hold 3 groups each (odd) and 2 (even): each against the oracle over its own slice."""
    hip = _hip()
    rng = np.random.default_rng(600 + fmt + asym)
    M, N = 200, 264
    for K, S in ((192, 2), (384, 4), (256, 4)):
        say(f"split-K fmt={fmt} asym={asym} tile={tile} K={K} S={S}")
        A = f16(rng.standard_normal((M, K)))
        q, s, z, wdq = _weights(rng, fmt, asym, N, K)
        w16 = np.asarray(wdq).view(np.float16)
        got = _run_gemm(hip, A, fmt, q, s, N, K, epi=hip.EPI_PARTIAL, ksplit=S, tile=tile, z=z)
        for k in range(S):
            sl = slice(k * K // S, (k + 1) * K // S)
            Az, Wz = np.ascontiguousarray(A[:, sl]), np.ascontiguousarray(w16[:, sl])
            assert_gemm_close(got[k], hxo.gemm(Az, Wz.view(np.uint16)), Az, Wz)


@pytest.mark.parametrize("fmt,M,N,K", [(1, 1536, 2560, 2560), (0, 512, 2048, 2048), (2, 300, 2048, 2048), (1, 64, 512, 8192)])
def test_launches_repeat_bit_for_bit(fmt, M, N, K):
    """40 launches on the same operands, one after another, at most a workgroup a CU, give the same bits."""
    hip = _hip()
    say(f"repeat fmt={fmt} {M}x{N}x{K}")
    L = hip.lib()
    rng = np.random.default_rng(700 + fmt)
    A = f16(rng.standard_normal((M, K)))
    q, s, _, _ = _weights(rng, fmt, False, N, K)
    dA, dW = hip.DeviceArray.from_numpy(A), hip.DeviceArray.from_numpy(q)
    dS = hip.DeviceArray.from_numpy(s) if s is not None else None
    for ks in (1, 4):
        outs = [hip.DeviceArray((ks, M, N), np.float16) for _ in range(8)]
        first = None
        for rep in range(5):
            for o in outs:
                hip.check(L.hxa_gemm(dA.ptr, K, M, fmt, dW.ptr, dS.ptr if dS else None, None, N, K, ks,
                                     hip.EPI_PARTIAL if ks > 1 else hip.EPI_STORE, o.ptr, N, M * N, None, 0, None, None, 0, 0,
                                     None), "gemm")
            hip.sync()
            for o in outs:
                b = o.numpy().view(np.uint16)
                first = b if first is None else first
                assert np.array_equal(b, first), (ks, rep)


@pytest.mark.parametrize("tile,fmt,asym", [(t, f, a) for t in ((64, 64, 4), (64, 128, 4), (128, 64, 4)) for f, a in FORMATS
                                           if not (f == 2 and t == (128, 64, 4))])  # (no such int4 kernel)
def test_two_workgroups_a_cu_repeat_bit_for_bit(tile, fmt, asym):
    """The tiles whose LDS ring lets two workgroups share a CU, on grids of two and more a CU: there the neighbour's loads put
    lines into L1 that this workgroup's loads then find, and a stage lands soonest after its barrier. A fragment read that it
    could overtake shows as a difference between launches."""
    hip = _hip()
    say(f"two workgroups a CU fmt={fmt} asym={asym} tile={tile}")
    L = hip.lib()
    rng = np.random.default_rng(720 + fmt + asym)
    M, N, K = 2048, 2048, 2048
    A = f16(rng.standard_normal((M, K)))
    q, s, z, _ = _weights(rng, fmt, asym, N, K)
    dA, dW = hip.DeviceArray.from_numpy(A), hip.DeviceArray.from_numpy(q)
    dS = hip.DeviceArray.from_numpy(s) if s is not None else None
    dZ = hip.DeviceArray.from_numpy(z) if z is not None else None
    outs = [hip.DeviceArray((M, N), np.float16) for _ in range(8)]
    first = None
    for rep in range(3):
        for o in outs:
            hip.check(L.hxa_gemm_tile(dA.ptr, K, M, fmt, dW.ptr, dS.ptr if dS else None, dZ.ptr if dZ else None, N, K, 1, 0,
                                      o.ptr, N, 0, None, 0, None, *tile, None), "gemm_tile")
        hip.sync()
        for o in outs:
            b = o.numpy().view(np.uint16)
            first = b if first is None else first
            assert np.array_equal(b, first), rep


@pytest.mark.parametrize("fmt,D,T,C_", [(1, 2560, 1536, 256), (0, 2560, 1792, 512), (2, 2560, 1536, 256)])
def test_block_with_the_paired_launch_repeats_bit_for_bit(fmt, D, T, C_):
    """The block whose cross q and text k / v run as one launch of more workgroups than CUs (2.9B class: 240 tiles and 80), 12
    times on the same input: the same bits. There a stage's loads once overtook fragment reads of the GEMM loop."""
    from tests.test_gpu_block import make_anima_pack
    hip = _hip()
    say(f"block repeat fmt={fmt} D={D} T={T}")
    L = hip.lib()
    rng = np.random.default_rng(740 + fmt)
    F, DC = 1024, 1024
    img, _, H = make_anima_pack(hip, rng, D, F, DC, fmt)
    x = rng.standard_normal((T, D)).astype(np.float32)
    mod = (rng.standard_normal((9, D)) * 0.2).astype(np.float32)
    ang = np.arange(T)[:, None] * 10000.0 ** (-np.arange(64) / 64.0)[None, :]
    bufs = [hip.DeviceArray.from_numpy(a) for a in (img, f16(rng.standard_normal((C_, DC))), mod, np.cos(ang).astype(np.float32),
                                                    np.sin(ang).astype(np.float32))]
    d = hip.BlockDims(0, D, H, F, C_, DC, T, 1, T, fmt, fmt, 1)
    ws = hip.block_ws(d)
    first = None
    for rep in range(12):
        dx = hip.DeviceArray.from_numpy(x)
        hip.check(L.hxa_block_run(C.byref(d), bufs[0].ptr, dx.ptr, bufs[1].ptr, bufs[2].ptr, bufs[3].ptr, bufs[4].ptr, ws.ptr, 0,
                                  None, 0, None), "block_run")
        hip.sync()
        b = dx.numpy().view(np.uint32)
        assert np.isfinite(b.view(np.float32)).all()
        first = b if first is None else first
        assert np.array_equal(b, first), rep


@pytest.mark.parametrize("fmt,asym", FORMATS)
@pytest.mark.parametrize("M,N,K", [(1, 136, 64), (31, 40, 192), (33, 200, 256), (65, 32, 832), (130, 72, 1280), (200, 520, 2048)])
def test_skinny_tiles(M, N, K, fmt, asym):
    """The 64x32 and 32x32 tiles with K split over the waves: fewer stages than waves (K = 64, 192), rings that do not fill,
    ragged rows and columns, a padded output whose padding stays, row-major and k-tiled weights: against the oracle, and the
    two tiles and layouts bit for bit alike (one wave split, one k order)."""
    hip = _hip()
    say(f"skinny fmt={fmt} asym={asym} {M}x{N}x{K}")
    L = hip.lib()
    rng = np.random.default_rng(800 + M + K + 7 * fmt + asym)
    A = f16(rng.standard_normal((M, K)))
    q, s, z, wdq = _weights(rng, fmt, asym, N, K)
    kt = hip.ktile(np.ascontiguousarray(q).view(np.uint8).reshape(-1), N, K)
    dA = hip.DeviceArray.from_numpy(A)
    dS = hip.DeviceArray.from_numpy(s) if s is not None else None
    dZ = hip.DeviceArray.from_numpy(z) if z is not None else None
    ldo, base = N + 8, None
    for fl, w in ((fmt, q), (fmt | hip.W_KTILED, kt)):
        dW = hip.DeviceArray.from_numpy(w)
        for bm in (64, 32):
            out = hip.DeviceArray.from_numpy(np.full((M, ldo), np.float16(3.0)))
            hip.check(L.hxa_gemm_tile(dA.ptr, K, M, fl, dW.ptr, dS.ptr if dS else None, dZ.ptr if dZ else None, N, K, 1, 0,
                                      out.ptr, ldo, 0, None, 0, None, bm, 32, 4, None), "gemm_tile")
            hip.sync()
            got = out.numpy()
            assert np.all(got[:, N:] == np.float16(3.0))
            got = np.ascontiguousarray(got[:, :N])
            if base is None:
                base = got
                assert_gemm_close(got, hxo.gemm(A, wdq), A, np.asarray(wdq).view(np.float16))
            assert np.array_equal(got.view(np.uint16), base.view(np.uint16)), (fl, bm)
    for bad in (dict(K=K - 32), dict(epi=hip.EPI_GELU_TANH), dict(ks=2)):  # whole stages, plain stores, one slice
        assert L.hxa_gemm_tile(dA.ptr, K, M, fmt, dW.ptr, dS.ptr if dS else None, dZ.ptr if dZ else None, N, bad.get("K", K),
                               bad.get("ks", 1), bad.get("epi", 0), out.ptr, ldo, 0, None, 0, None, 64, 32, 4, None) != 0


@pytest.mark.parametrize("fmt", [0, 1, 2])
def test_linear_takes_the_skinny_tile_for_few_output_tiles(fmt):
    """hxa_linear at 256 x 2048 x 2048 needs no workspace and gives the 64x32 tile's bits; with K % 64 = 32 it gives the
    one-launch GEMM's."""
    hip = _hip()
    L = hip.lib()
    rng = np.random.default_rng(900 + fmt)
    for M, N, K in ((256, 2048, 2048), (64, 256, 544)):
        say(f"linear fmt={fmt} {M}x{N}x{K}")
        A = f16(rng.standard_normal((M, K)))
        q, s, _, _ = _weights(rng, fmt, False, N, K)
        dA, dW = hip.DeviceArray.from_numpy(A), hip.DeviceArray.from_numpy(q)
        dS = hip.DeviceArray.from_numpy(s) if s is not None else None
        sp = dS.ptr if dS else None
        assert L.hxa_linear_split_k(M, N, K, fmt) == 1 and L.hxa_linear_ws_bytes(M, N, K, fmt) == 0
        o, t = hip.DeviceArray((M, N), np.float16), hip.DeviceArray((M, N), np.float16)
        hip.check(L.hxa_linear(dA.ptr, K, M, fmt, dW.ptr, sp, None, N, K, o.ptr, N, None, 0, None), "linear")
        tile = (64, 32, 4) if K % 64 == 0 else (128, 128, 4)
        hip.check(L.hxa_gemm_tile(dA.ptr, K, M, fmt, dW.ptr, sp, None, N, K, 1, 0, t.ptr, N, 0, None, 0, None, *tile, None),
                  "gemm_tile")
        hip.sync()
        assert np.array_equal(o.numpy().view(np.uint16), t.numpy().view(np.uint16))


@pytest.mark.parametrize("tile", [(256, 256, 9), (192, 256, 9), (128, 128, 4), (64, 64, 4)])
def test_gelu_erf_over_every_fp16_value(tile):
    """GELU-erf of every finite fp16 value, which the LDS part of the lookup table (2^-11 <= |t| < 6) and the global one share:
    within 2 ulps of the oracle (the fp16 rounding of T2 and of the result); rows with a NaN or inf operand are NaN (inf * 0 in
    the product). Infinities reach the epilogue in test_gelu_erf_of_overflowed_sums."""
    hip = _hip()
    say(f"gelu erf tile={tile}")
    M, N, K = 256, 256, 32
    vals = np.arange(65536, dtype=np.uint16).view(np.float16).reshape(M, N)
    # one launch per 32 columns: A[m][k] = vals[m][32 j + k], W[n] = e_(n % 32)
    W = f16(np.tile(np.eye(32), (N // 32, 1)))
    for j in range(0, N // 32):
        A = vals[:, 32 * j:32 * j + 32].copy()
        bad = ~np.isfinite(A).all(axis=1)  # inf * 0: the whole row is NaN
        got = _run_gemm(hip, A, 0, W, None, N, K, epi=hip.EPI_GELU_ERF, tile=tile)[:, :32]
        t = np.where(np.isfinite(A), A, np.float16(0))
        ref = hxo.gelu(t, 0).view(np.float16)
        assert ulp_diff(np.ascontiguousarray(got[~bad]), np.ascontiguousarray(ref[~bad])).max() <= 2
        assert np.isnan(got[bad]).all()


@pytest.mark.parametrize("fmt,N", [(0, 2**24 + 264), (1, 2**24 + 264), (2, 2**24 + 264), (0, 2**25 + 1032)])
def test_linear_of_many_columns(fmt, N):
    """k-tiled weights whose second k group lies 2^28 to 2^31 bytes and more behind the first, where the loaders' 32-bit offsets
    have to reach it: the first and last 264 columns against the oracle."""
    hip = _hip()
    say(f"linear fmt={fmt} N={N}")
    L = hip.lib()
    M, K, n = 8, 96, 264
    rng = np.random.default_rng(1000 + fmt)
    A = f16(rng.standard_normal((M, K)))
    dA, out = hip.DeviceArray.from_numpy(A), hip.DeviceArray((M, N), np.float16)
    unit = (64, 32, 16)[fmt]
    dW = hip.DeviceArray((K // 32 * N * unit,), np.uint8)
    cols = []  # the weights of both ends, the rest stays what a fill leaves
    hip.check(L.hxa_fill_normal(dW.ptr, 1, K // 32 * N * unit // 2, 5, 0.0, 0.05, None), "fill")
    dS = None
    if fmt:
        dS = hip.DeviceArray((K // 32, N), np.float16)
        hip.check(L.hxa_fill_const(dS.ptr, 1, K // 32 * N, 1e-3, None), "fill")
    hip.sync()
    for n0 in (0, N - n):
        q, s, _, wdq = _weights(rng, fmt, False, n, K)
        kt = hip.ktile(np.ascontiguousarray(q).view(np.uint8).reshape(-1), n, K).reshape(K // 32, n * unit)
        for g in range(K // 32):
            row = np.ascontiguousarray(kt[g])
            hip.check(L.hxa_h2d(dW.at((g * N + n0) * unit), row.ctypes.data, row.nbytes), "h2d")
            if fmt:
                sr = np.ascontiguousarray(np.asarray(s).reshape(K // 32, n)[g])
                hip.check(L.hxa_h2d(dS.at((g * N + n0) * 2), sr.ctypes.data, sr.nbytes), "h2d")
        cols.append((n0, np.asarray(wdq).view(np.float16)))
    hip.check(L.hxa_linear(dA.ptr, K, M, fmt | hip.W_KTILED, dW.ptr, dS.ptr if dS else None, None, N, K, out.ptr, N, None, 0,
                           None), "linear")
    hip.sync()
    for n0, w in cols:
        got = np.zeros((M, n), np.float16)
        for m in range(M):
            hip.check(L.hxa_d2h(got[m:].ctypes.data, out.at((m * N + n0) * 2), 2 * n), "d2h")
        assert_gemm_close(got, hxo.gemm(A, w.view(np.uint16)), A, w)


@pytest.mark.parametrize("asym", [False, True])
def test_int4_values_under_every_scale(asym):
    """Every nibble in every position of a word under each of the 65536 fp16 scale patterns (subnormals, infinities and NaN too;
    with offsets, one of as many): the oracle's bits."""
    hip = _hip()
    rng = np.random.default_rng(77)
    N, K = 65536, 32
    q = rng.integers(0, 256, (N, K // 2), dtype=np.uint8)
    q[:, 0] = np.arange(N) & 255
    s = np.arange(N, dtype=np.uint16).reshape(1, N)
    z = rng.permutation(np.arange(N, dtype=np.uint16)).reshape(1, N) if asym else None
    dq, ds = hip.DeviceArray.from_numpy(q), hip.DeviceArray.from_numpy(s)
    dz = hip.DeviceArray.from_numpy(z) if asym else None
    out = hip.DeviceArray((1, N, 32), np.float16)
    hip.check(hip.lib().hxa_dequant(2, dq.ptr, ds.ptr, dz.ptr if dz else None, N, K, out.ptr, None), "dequant")
    hip.sync()
    ref = np.asarray(hxo.q4_dequant(q, s, z) if asym else hxo.q4_dequant(q, s)).view(np.float16).reshape(N, 32)
    got = out.numpy()[0]
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got.view(np.uint16)[~nan], ref.view(np.uint16)[~nan])


@pytest.mark.parametrize("M,N,K,fmt,ks", [(1152, 8192, 2048, 1, 1), (1152, 2048, 8192, 1, 4), (1152, 9216, 3072, 2, 1)])
def test_pick_covers_no_idle_rows_at_equal_cost(M, N, K, fmt, ks):
    """256x192 and 192x256 tiles within 1% of each other in the model: the pick is the one whose tiles end with the rows."""
    hip = _hip()
    pk = hip.gemm_pick(M, N, K, fmt, ks, hip.EPI_PARTIAL if ks > 1 else 0)
    assert (pk["bm"], pk["bn"]) == (192, 256)


@pytest.mark.parametrize("tile", [(256, 256, 9), (128, 128, 4), (64, 64, 4)])
def test_gelu_erf_of_overflowed_sums(tile):
    """Products past the fp16 range reach the epilogue as infinities: GELU-erf of them is the oracle's inf and 0 (T2 is 0
    there), beside finite values and NaN."""
    hip = _hip()
    M, N, K = 64, 64, 32
    A = np.zeros((M, K), np.float16)
    A[:, 0] = np.float16(60000.0)
    A[1::4, 0] = np.float16(-60000.0)
    A[2::4, 0] = np.float16(1.5)
    A[3::4, 0] = np.float16(np.nan)
    W = np.zeros((N, K), np.float16)
    W[:, 0] = np.float16(2.0)
    got = _run_gemm(hip, A, 0, W, None, N, K, epi=hip.EPI_GELU_ERF, tile=tile)
    assert np.all(got[0::4] == np.inf) and np.all(got[1::4] == 0)
    ref = hxo.gelu(np.full((1, 1), 3.0, np.float16), 0).view(np.float16)
    assert ulp_diff(got[2::4], np.broadcast_to(ref, got[2::4].shape).copy()).max() <= 2
    assert np.isnan(got[3::4]).all()
