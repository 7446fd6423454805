// The GEMM kernels' device code: O[M][N] = A[M][K] . W[N][K]^T with fused epilogues, instantiated per weight format in
// gemm_f16.hip, gemm_q8.hip and gemm_q4.hip (one translation unit each); gemm.hip holds the host side.
//
// Replaces the reference's HMX GEMM engine (hexagon/mega/gemm2.c:96-137, gemm_run_geo) including its q8 tile
// dequantisation (gemm2.c:19-35 dq_tile), the MOSS q4a dequantisation (moss/hexagon/mega/gemm2.c:39-56) and the
// flush epilogues (gemm2.c:58-82: gated residual, GELU, split-K residual partial; moss mode 5 SiTU).
//
// Design (CDNA4, 64-wide waves):
//  * 256 or 512 threads = 4 or 8 waves in a 2 x 2 or 2 x 4 grid over a BM x BN tile, v_mfma_f32_16x16x32_f16 with the
//    weight fragment as the A operand (fp32 accumulate; each lane accumulates 4 consecutive output columns of a row).
//  * K is consumed in stages of 64. A and W go from global memory straight into an LDS ring of 2 - 5 stages
//    (global_load_lds_dwordx4, no VGPR staging); one s_barrier per stage, with explicit vmcnt waits so the prefetches
//    stay in flight. 16-byte LDS chunks are XOR-swizzled per row, which spreads one lane group's 16 rows over the banks; the
//    passes of a ds_read_b128 mix two lane groups, whose rows still meet in pairs (SQ_LDS_BANK_CONFLICT is half of
//    SQ_LDS_IDX_ACTIVE). A placement without these conflicts (bits 0 and 1 of the chunk exchanged before the XOR; counted: 0.04,
//    LDS active 57 -> 29% of the MLP-down's cycles) leaves the times as they are, blocks fp16 0.0%, int8 -0.4%, int4 -1.5%,
//    linears +0.1 / +0.1 / -0.6% (single ones +5%): LDS reads are not what the loops wait for.
//  * int8 / int4 weights stay raw in LDS and are dequantised into the W fragments in registers with the fp16
//    exponent-bias trick: a byte u placed under the exponent 0x64 is the fp16 value 1024+u, so (1024+u) - 1152 = q
//    exactly, then one fp16 multiply by the group scale gives f16(q*s) -- the reference's exact dequantised value
//    (gemm2.c:19-22).
//  * The fp16-rounded output tile is staged through LDS for a coalesced epilogue (16-byte loads / stores).
//  * The block index is remapped so each of the 8 XCDs (own L2) works on a rectangle of output tiles.
#pragma once
#include <type_traits>

#include "hxa_common.h"
#include "kernels.h"

namespace hxg {

struct GemmParams {
  const hxa_h *A;
  long lda;
  const void *W;
  const hxa_h *S, *Z;
  // W element (fp16 / int8; q4: byte) offset of row n, k group g: n * w_rs + g * w_gs. Row-major [N][K]: w_rs = K
  // (q4: K/2), w_gs = 32 (16); k-tiled [K/32][N][32] (q4: [K/32][N][16 bytes]): w_rs = 32 (16), w_gs = 32 N (16 N)
  long w_rs, w_gs;
  int M, N, Kslice, Ktot;
  int epi;
  hxa_h *out;
  long ldo, out_zstride;
  float *out32;  // PARTIAL_F32: slice z's fp32 sums at out32[z * out_zstride + m * ldo + n]
  float *x;
  long ldx;
  const float *gate;
  hxa_h *out_t;  // columns >= split_col go transposed to out_t[n - split_col][m]
  long ldo_t;
  int split_col;
  int tiles_m, tiles_n;
  // XCD placement: workgroup b runs on XCD b % 8. xcd_gm > 0: the tile grid is cut into 8 equal rectangles, xcd_gm
  // along M, and XCD x takes rectangle x (M-fastest inside); 0: XCD x takes the x-th eighth of the M-fastest order
  int xcd_gm;
  // head norm (STORE epilogue): columns [0, hn_cols), in whole heads of 128, get RMSNorm * gain and optional RoPE
  int hn_cols, hn_gsplit, hn_ttab;
  const float *hn_g0, *hn_g1, *hn_cos, *hn_sin;
  const uint8_t *pf;  // bytes to touch after the main loop (HxaGemm::pf)
  long pf_bytes;
  HxaClk clk;  // shader-clock record (hxa_clock_record), indexed by the launch's flat workgroup id
  const hxa_h *erf_t2;  // GELU-erf: T2 of every non-negative fp16 bit pattern (null: evaluated in the epilogue)
  int erf_lds;          // > 0: byte offset in LDS where the epilogue copies the table from ERF_T2_LDS_LO on
  // fused cross attention (gemm_xattn_kernel): the tile's queries attend to image (m0 / xa_T)'s keys
  // xa_k [NKV][xa_ldk] (+ image * xa_kb), V^T xa_vt [D][xa_ldvt] (+ image * xa_vb); O to xa_o [M][xa_ldo]
  const hxa_h *xa_k, *xa_vt;
  hxa_h *xa_o;
  long xa_ldk, xa_ldvt, xa_ldo, xa_kb, xa_vb;
  int xa_nkv, xa_nvalid, xa_T;
  // side_wgs > 0 (8-wave kernels, one K slice): workgroups past the tile grid run side's GEMV rows
  HxaSideGemv side;
  int side_wgs;
};

// Touch this workgroup's share of [p.pf, p.pf + p.pf_bytes), one 4-byte load per 128-byte line: the lines come into
// L2 / MALL for the next kernel while this one runs its epilogue. The loads go straight to LDS (no register is
// written behind the compiler's back) into `sink`, PF_LDS bytes past everything the kernel uses, whose contents are
// never read; the workgroup drains them (vmcnt 0) before it ends, as every LDS DMA must.
HXA_DEV void prefetch_share(const GemmParams &p, int wg, int nwg, int tid, int nt, const uint8_t *sink) {
  const long lines = (p.pf_bytes + 127) >> 7;
  const long per = (lines + nwg - 1) / nwg;
  const long l0 = (long)wg * per, l1 = min(lines, l0 + per);
  const uint32_t la = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_void_t *)sink);
  for (long l = l0 + tid; l < l1; l += nt) {
    const uint8_t *a = p.pf + min(l << 7, p.pf_bytes - 4);  // pf_bytes >= 4 (checked on the host)
    asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dword %0, off" ::"v"(a), "s"(la) : "memory", "m0");
  }
}

// a pointer the compiler is to hold in scalar registers (every lane has the same)
HXA_DEV const uint8_t *uniform_ptr(const uint8_t *p) {
  const uint64_t v = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return (const uint8_t *)(((uint64_t)hi << 32) | lo);
}

// tile (tm, tn) of workgroup bid
HXA_DEV void tile_coords(const GemmParams &p, int bid, int &tm, int &tn) {
  const int ntiles = p.tiles_m * p.tiles_n;
  if (p.xcd_gm > 0) {
    const int x = bid & 7, i = bid >> 3;
    const int xm = p.tiles_m / p.xcd_gm, xn = p.tiles_n * p.xcd_gm / 8;
    tm = (x % p.xcd_gm) * xm + i % xm;
    tn = (x / p.xcd_gm) * xn + i / xm;
    return;
  }
  const int tile = (ntiles % 8 == 0) ? (bid % 8) * (ntiles / 8) + bid / 8 : bid;
  tm = tile % p.tiles_m;
  tn = tile / p.tiles_m;
}

// the gains of head-normed columns n .. n+7 and a row's RoPE coefficients of dims (n & 63) .. +7
HXA_DEV void hn_gains(const GemmParams &p, int n, float (&g)[8]) {
  const float *gp = (n < p.hn_gsplit ? p.hn_g0 : p.hn_g1) + (n & 127);
  const float4_t a = *(const float4_t *)gp, b = *(const float4_t *)(gp + 4);
#pragma unroll
  for (int e = 0; e < 4; e++) {
    g[e] = a[e];
    g[e + 4] = b[e];
  }
}
HXA_DEV void hn_rope_t(const GemmParams &p, int tt, int n, float (&cs)[8], float (&sn)[8]) {
  const long o = (long)tt * 64 + (n & 63);
  const float4_t c0 = *(const float4_t *)(p.hn_cos + o), c1 = *(const float4_t *)(p.hn_cos + o + 4);
  const float4_t s0 = *(const float4_t *)(p.hn_sin + o), s1 = *(const float4_t *)(p.hn_sin + o + 4);
#pragma unroll
  for (int e = 0; e < 4; e++) {
    cs[e] = c0[e];
    cs[e + 4] = c1[e];
    sn[e] = s0[e];
    sn[e + 4] = s1[e];
  }
}

HXA_DEV half2_t as_h2(uint32_t u) { return __builtin_bit_cast(half2_t, u); }
HXA_DEV uint32_t as_u(half2_t h) { return __builtin_bit_cast(uint32_t, h); }

// 4 int8 (two's complement, k-consecutive) -> 2 x half2 of f16(q*s)
HXA_DEV void dq8_word(uint32_t d, half2_t s2, uint32_t &o0, uint32_t &o1) {
  const uint32_t x = d ^ 0x80808080u;                         // offset binary u = q + 128
  const uint32_t lo = __builtin_amdgcn_perm(0x64646464u, x, 0x04010400u);  // (0x64|u0, 0x64|u1) = 1024+u
  const uint32_t hi = __builtin_amdgcn_perm(0x64646464u, x, 0x04030402u);
  const half2_t c = {(hxa_h)1152.0f, (hxa_h)1152.0f};
  o0 = as_u((as_h2(lo) - c) * s2);
  o1 = as_u((as_h2(hi) - c) * s2);
}

// (d & mask) | magic in one operation: as C++ it becomes v_and + v_or, since a three-operand instruction takes no literal
HXA_DEV uint32_t and_or(uint32_t d, uint32_t mask, uint32_t magic) {
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(d), "s"(mask), "v"(magic));
  return r;
}
// 8 int4 of one 32-bit word -> 4 x half2. Even nibbles n land in the low mantissa bits, 1024 + n, odd ones four bits up, 1024 +
// 16 n, which an exact fma by 1/16 brings down: one shift for the word instead of three, 13 operations instead of 19. The int4
// tiles at and below 256x128 are bound by these (128x128: as many cycles of them as of MFMAs); int4 linears of 14 shapes x 1 -
// 6656 rows take 4.5% less time (512 x 2048 -> 6144 29.4 -> 25.9 us, 1536 x 2560 -> 2560 35.6 -> 31.6, 6656 x 10240 -> 2560
// 410 -> 402)
template <bool ASYM>
HXA_DEV void dq4_word(uint32_t d, half2_t s2, half2_t z2, uint32_t *o) {
  const half2_t c = ASYM ? (half2_t){(hxa_h)-1024.0f, (hxa_h)-1024.0f} : (half2_t){(hxa_h)-1032.0f, (hxa_h)-1032.0f};
  const half2_t c16 = ASYM ? (half2_t){(hxa_h)-64.0f, (hxa_h)-64.0f} : (half2_t){(hxa_h)-72.0f, (hxa_h)-72.0f};
  const half2_t r16 = {(hxa_h)0.0625f, (hxa_h)0.0625f};
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const uint32_t w = j < 2 ? d : d >> 8;
    const half2_t v = as_h2(and_or(w, j & 1 ? 0x00F000F0u : 0x000F000Fu, 0x64006400u));  // (n_{2j}, n_{2j+1})
    const half2_t q = j & 1 ? __builtin_elementwise_fma(v, r16, c16) : v + c;
    o[j] = as_u(ASYM ? __builtin_elementwise_fma(q, s2, z2) : q * s2);
  }
}

HXA_DEV float gelu_tanh_f(float t) {
  // 0.5 t (1 + tanh u) written as t / (1 + exp(-2u)) (kern.c:116-132): no cancellation for negative t. With
  // u = sqrt(2/pi) (t + 0.044715 t^3), exp(-2u) = 2^(t (K1 + K3 t^2)): the constants folded, three VALU operations
  // for the exponent instead of six (the MLP-up epilogue runs this on every output)
  constexpr float K1 = (float)(-2.0 * 1.4426950408889634 * 0.7978845608028654);
  constexpr float K3 = (float)(-2.0 * 1.4426950408889634 * 0.7978845608028654 * 0.044715);
  const float e = __builtin_amdgcn_exp2f(t * fmaf(K3, t * t, K1));
  return t * __builtin_amdgcn_rcpf(1.0f + e);  // v_rcp_f32 (1 ulp): far below the fp16 rounding
}
// T2(a) = f16(a * 0.5 * erfc(a / sqrt 2)) for a >= 0, 0 at infinity (where the product is inf * 0)
HXA_DEV hxa_h gelu_t2(float a) { return a == INFINITY ? (hxa_h)0.0f : (hxa_h)(a * 0.5f * erfcf(a * 0.7071067811865476f)); }
HXA_DEV float gelu_erf_f(float t) {  // kern.c:248-260: f16(max(t,0) - T2(|t|))
  return fmaxf(t, 0.0f) - (float)gelu_t2(fabsf(t));
}
// T2 of every non-negative fp16 bit pattern b (a = |t|; NaN and inf patterns included): the GELU-erf epilogue looks its values
// up instead of evaluating erfcf per output. Filled once per device by erf_t2_kernel with gelu_t2, so a lookup returns the same
// bits.
constexpr int ERF_T2_N = 0x8000;
// the part of the table a GELU-erf epilogue copies into LDS past its tile: 2^-11 <= |t| < 6 (bit patterns 0x1000 to
// 0x4600), 27648 bytes = 27 wave-wide 16-byte copies, what 256x256 leaves of 160 KB; other |t| (rare) are looked up in the
// global table. (With the 35 KB of all |t| < 6 the 256x256 tiles had no room and made every lookup from memory: int8 1536 x
// 2560 x 10240 took 15.2 us longer than with a plain store, now 5.5.)
constexpr int ERF_T2_LDS_LO = 0x1000, ERF_T2_LDS_N = 0x4600 - ERF_T2_LDS_LO, ERF_T2_LDS_BYTES = ERF_T2_LDS_N * 2;
HXA_DEV float gelu_erf_tab(float t, const hxa_h *__restrict__ t2tab) {
  const uint32_t b = __builtin_bit_cast(uint16_t, (hxa_h)t) & 0x7fffu;
  return fmaxf(t, 0.0f) - (float)t2tab[b];
}
HXA_DEV float situ_f(float u, float g) {
  // moss kern.c:376-405: f16(f16(25 tanh(u/25)) * f16(4 tanh(g/4) sigmoid(g)))
  const float tu = (float)(hxa_h)(25.0f * tanhf(u * 0.04f));
  const float gs = (float)(hxa_h)(4.0f * tanhf(g * 0.25f) / (1.0f + __expf(-g)));
  return tu * gs;
}

// ---- geometry of a tile's LDS ring ----
// A stage holds 64 k of the tile (two quantisation groups): BM rows of 128 B of A, BN rows of W (fp16 128 B, int8 64 B,
// int4 32 B) and the two groups' scale (and offset) vectors. 64 deep, because a row's 128 B is one cache line: 32-deep
// stages read each line of A in two halves a k step apart, and the tiles whose step does not fit L1 (32 KB) fetched
// every line of A from L2 twice.
template <int BM, int BN, int FMT>
struct GemmGeo {
  static constexpr int RBW = FMT == HXA_W_F16 ? 128 : FMT == HXA_W_Q8 ? 64 : 32;  // W bytes per row per stage
  static constexpr int A_BYTES = BM * 128;
  static constexpr int W_BYTES = BN * RBW;
  static constexpr int S_BYTES = FMT == HXA_W_F16 ? 0 : BN * 4;      // one vector: 2 groups x BN fp16
  static constexpr int STAGE = A_BYTES + W_BYTES + 2 * S_BYTES;      // scale + optional offset vectors
  static constexpr int CROW = BN + 8;
  static constexpr int C_BYTES = BM * CROW * 2;
  static constexpr int PF_LDS = 256;                                 // prefetch_share's sink (64 lanes x 4 B)
  // Tiles below 128x128 have too few MFMAs per slice to cover an LDS read: they keep a whole stage of fragments ahead in
  // registers (gemm_body; 64x64 at K 8192: 32.6 -> 27.3 us)
  static constexpr bool DEEP = BM * BN < 128 * 128;
  // ring stages: as many as fit in 160 KB, 4 at most; below 128x128 what lets two workgroups share a CU, 3, for 64x64 5 (64x128
  // with 6 stages, one workgroup a CU: 9.6 -> 10.2 us at 512 x 2048 x 2048 in two K slices)
  static constexpr int NSMAX = BM * BN <= 64 * 64 ? 5 : BM * BN < 128 * 128 ? 3 : 4;
  static constexpr int NS = NSMAX * STAGE <= 160 * 1024 ? NSMAX : 3 * STAGE <= 160 * 1024 ? 3 : 2;
  static constexpr int lds(int ns) { return ns * STAGE > C_BYTES + PF_LDS ? ns * STAGE : C_BYTES + PF_LDS; }
  // past the staged tile (the ring is dead by then): the touch's sink, then a GELU-erf launch's copy of the T2 table
  static constexpr int PF_OFF = C_BYTES, ERF_OFF = C_BYTES + PF_LDS;
  static constexpr int lds_erf(int ns) {
    return lds(ns) > ERF_OFF + ERF_T2_LDS_BYTES ? lds(ns) : ERF_OFF + ERF_T2_LDS_BYTES;
  }
  static constexpr int NA = A_BYTES / 1024, NWI = W_BYTES / 1024, NLI = NA + NWI;  // 1 KB load instructions per stage
};

// PARTIAL_F32: the K slice's fp32 sums straight from the accumulators (no fp16 rounding, no LDS staging). For block
// (j, i) the lane holds row mrow + 16 i and columns ncol + 16 j + 0..3: one 16-byte store each, so a wave's store
// fills 16 rows x 64 contiguous bytes. N % 8 == 0, so a chunk of 4 is inside N or past it.
template <int MI, int NI>
HXA_DEV void store_partial_f32(const GemmParams &p, const float4_t (&acc)[NI][MI], int mrow, int ncol, int z) {
  float *base = p.out32 + (long)z * p.out_zstride;
#pragma unroll
  for (int i = 0; i < MI; i++) {
    const int m = mrow + i * 16;
    if (m >= p.M) continue;
#pragma unroll
    for (int j = 0; j < NI; j++) {
      const int n = ncol + j * 16;
      if (n < p.N) *(float4_t *)(base + (long)m * p.ldo + n) = acc[j][i];
    }
  }
}
// f16(acc) as the row-major [BM][CROW] tile in LDS: for block (j, i) the lane holds row ml + 16 i and columns
// nl + 16 j + 0..3
template <int MI, int NI, int CROW>
HXA_DEV void stage_tile(hxa_h *Cs, const float4_t (&acc)[NI][MI], int ml, int nl) {
#pragma unroll
  for (int j = 0; j < NI; j++)
#pragma unroll
    for (int i = 0; i < MI; i++)
      *(half4_t *)(Cs + (ml + i * 16) * CROW + nl + j * 16) =
          (half4_t){(hxa_h)acc[j][i][0], (hxa_h)acc[j][i][1], (hxa_h)acc[j][i][2], (hxa_h)acc[j][i][3]};
}

template <int BM, int BN, int NT, bool SPLIT2>
HXA_DEV void gemm_epilogue(const GemmParams &p, const hxa_h *Cs, int m0, int n0, int tid, int z) {
  constexpr int CROW = BN + 8;
  constexpr int C8 = BN / 8;
  if (p.epi == HXA_EPI_SITU) {
    // columns interleaved per 32 (up_j, gate_j): output column (n0/2) + p*32 + c
    for (int c = tid; c < BM * (C8 / 2); c += NT) {
      const int ml = c / (C8 / 2), oc = (c % (C8 / 2)) * 8;
      const int m = m0 + ml, on = n0 / 2 + oc;
      if (m >= p.M || on * 2 >= p.N) continue;
      const int pr = oc / 32, cc = oc % 32;
      const half8_t u = *(const half8_t *)(Cs + ml * CROW + pr * 64 + cc);
      const half8_t g = *(const half8_t *)(Cs + ml * CROW + pr * 64 + 32 + cc);
      half8_t o;
#pragma unroll
      for (int e = 0; e < 8; e++) o[e] = (hxa_h)situ_f((float)u[e], (float)g[e]);
      *(half8_t *)(p.out + (long)m * p.ldo + on) = o;
    }
    return;
  }
  // local columns [0, nsplit) row-major, [nsplit, BN) transposed into out_t. Without out_t the chunk count per row
  // is the compile-time BN / 8 (no runtime division in the loop).
  const int nsplit = p.out_t == nullptr ? BN : min(max(p.split_col - n0, 0), BN);
  if (p.epi == HXA_EPI_RESADD) {
    // x += gate * t: the x / gate loads of RB chunks are issued together before any of them is used, so a thread
    // waits one memory latency per batch instead of one per chunk (x stores may alias later x loads otherwise)
    constexpr int NC8 = BN / 8, ITERS = BM * NC8 / NT, RB = ITERS % 4 == 0 ? 4 : ITERS % 3 == 0 ? 3 : ITERS % 2 == 0 ? 2 : 1;
    static_assert(BM * NC8 % NT == 0 && ITERS % RB == 0, "whole chunk passes");
#pragma unroll
    for (int b0 = 0; b0 < ITERS; b0 += RB) {
      float4_t xv[RB][2], gv[RB][2];
      float t[RB][8];
      bool ok[RB];
#pragma unroll
      for (int u = 0; u < RB; u++) {
        const int c = tid + (b0 + u) * NT, ml = c / NC8, nl = (c % NC8) * 8, m = m0 + ml, n = n0 + nl;
        ok[u] = m < p.M && n < p.N;
        if (ok[u]) {
          const float4_t *xp = (const float4_t *)(p.x + (long)m * p.ldx + n);
          xv[u][0] = xp[0];
          xv[u][1] = xp[1];
          gv[u][0] = *(const float4_t *)(p.gate + n);
          gv[u][1] = *(const float4_t *)(p.gate + n + 4);
          const half8_t v = *(const half8_t *)(Cs + ml * CROW + nl);
#pragma unroll
          for (int e = 0; e < 8; e++) t[u][e] = (float)v[e];
          if constexpr (SPLIT2) {
            const half8_t v1 = *(const half8_t *)(Cs + BM * CROW + ml * CROW + nl);
#pragma unroll
            for (int e = 0; e < 8; e++) t[u][e] = (float)v1[e] + t[u][e];
          }
        }
      }
#pragma unroll
      for (int u = 0; u < RB; u++) {
        if (!ok[u]) continue;
        const int c = tid + (b0 + u) * NT, ml = c / NC8, nl = (c % NC8) * 8;
        float4_t *xp = (float4_t *)(p.x + (long)(m0 + ml) * p.ldx + n0 + nl);
#pragma unroll
        for (int e = 0; e < 4; e++) {
          xv[u][0][e] = fmaf(gv[u][0][e], t[u][e], xv[u][0][e]);
          xv[u][1][e] = fmaf(gv[u][1][e], t[u][e + 4], xv[u][1][e]);
        }
        xp[0] = xv[u][0];
        xp[1] = xv[u][1];
      }
    }
    return;
  }
  if constexpr (BN % 128 == 0) {
  if (p.hn_cols > 0 && (n0 + BN <= p.hn_cols || p.hn_cols >= p.N)) {
    // every (valid) column of this tile is head-normed. Thread (row group r0, jj) owns dims [8jj, 8jj+8) and
    // [64+8jj, 64+8jj+8) of every head of the tile on its rows: the gains are loaded once, the RoPE coefficients once
    // per row for all heads (fetched one pass ahead), and the rotation partners sit in the same thread.
    constexpr int HT = BN / 128, RP = NT / 8;  // heads per tile, rows per pass
    static_assert(BM % RP == 0, "whole passes");
    const int jj = tid & 7, r0 = tid >> 3;
    const bool rope = p.hn_cos != nullptr;
    float glo[HT][8], ghi[HT][8], cs[8] = {}, sn[8] = {}, csn[8] = {}, snn[8] = {};
#pragma unroll
    for (int hh = 0; hh < HT; hh++) {
      hn_gains(p, n0 + hh * 128 + 8 * jj, glo[hh]);
      hn_gains(p, n0 + hh * 128 + 64 + 8 * jj, ghi[hh]);
    }
    // RoPE table row of the next pass's row, stepped by RP rows without a division (rows past M are not stored)
    int tt = rope ? min(m0 + r0, p.M - 1) % p.hn_ttab : 0;
    if (rope) hn_rope_t(p, tt, 8 * jj, cs, sn);
    for (int it = 0; it < BM / RP; it++) {
      const int ml = r0 + it * RP, m = m0 + ml;
      if (rope && it + 1 < BM / RP) {
        if (m + RP < p.M) {
          tt += RP;
          while (tt >= p.hn_ttab) tt -= p.hn_ttab;
        }
        hn_rope_t(p, tt, 8 * jj, csn, snn);
      }
      if (m < p.M) {  // whole 8-lane groups share m
#pragma unroll
        for (int hh = 0; hh < HT; hh++) {
          const int nl = hh * 128 + 8 * jj;
          if (n0 + nl >= p.N) break;
          half8_t lo = *(const half8_t *)(Cs + ml * CROW + nl), hi = *(const half8_t *)(Cs + ml * CROW + nl + 64);
          head_norm2(lo, hi, glo[hh], ghi[hh], rope, cs, sn);
          *(half8_t *)(p.out + (long)m * p.ldo + n0 + nl) = lo;
          *(half8_t *)(p.out + (long)m * p.ldo + n0 + nl + 64) = hi;
        }
      }
      if (rope) {
#pragma unroll
        for (int e = 0; e < 8; e++) {
          cs[e] = csn[e];
          sn[e] = snn[e];
        }
      }
    }
    return;
  }
  }
  if (p.epi == HXA_EPI_GELU_ERF && p.erf_lds > 0 && nsplit == BN) {
    // GELU-erf through the T2 table: the LDS reads and table lookups of RB chunks are issued together before any
    // of them is used, so a thread waits one lookup latency per batch instead of one per chunk. The
    // table's frequent part is first copied into LDS past the staged tile (LDS gathers, where global ones issue at
    // a few lanes per clock)
    constexpr int ITERS = BM * C8 / NT, RB = ITERS % 4 == 0 ? 4 : ITERS % 3 == 0 ? 3 : ITERS % 2 == 0 ? 2 : 1;
    static_assert(BM * C8 % NT == 0 && ITERS % RB == 0, "whole chunk passes");
    static_assert(ERF_T2_LDS_BYTES % 1024 == 0, "whole wave-wide copies");
    const hxa_h *tl;
    {
      uint8_t *dst = (uint8_t *)Cs + p.erf_lds;
      const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
      for (int c0 = wave * 64; c0 < ERF_T2_LDS_BYTES / 16; c0 += NT) {
        const uint32_t la = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_void_t *)(dst + c0 * 16));
        asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(p.erf_t2 + ERF_T2_LDS_LO + (c0 + lane) * 8), "s"(la)
                     : "memory", "m0");
      }
      wait_vm<0>();
      __syncthreads();
      tl = (const hxa_h *)dst;
    }
#pragma unroll
    for (int b0 = 0; b0 < ITERS; b0 += RB) {
      half8_t v[RB];
      hxa_h t2[RB][8];
      bool ok[RB];
#pragma unroll
      for (int u = 0; u < RB; u++) {
        const int c = tid + (b0 + u) * NT, ml = c / C8, nl = (c % C8) * 8;
        ok[u] = m0 + ml < p.M && n0 + nl < p.N;
        v[u] = *(const half8_t *)(Cs + ml * CROW + nl);
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const hxa_h x = v[u][e];  // (a scalar copy: bit_cast of a vector element itself read element 0 only)
          const uint32_t b = __builtin_bit_cast(uint16_t, x) & 0x7fffu;
          t2[u][e] = b - ERF_T2_LDS_LO < (uint32_t)ERF_T2_LDS_N ? tl[b - ERF_T2_LDS_LO] : p.erf_t2[b];
        }
      }
#pragma unroll
      for (int u = 0; u < RB; u++) {
        if (!ok[u]) continue;
        const int c = tid + (b0 + u) * NT, ml = c / C8, nl = (c % C8) * 8;
        half8_t o;
#pragma unroll
        for (int e = 0; e < 8; e++) o[e] = (hxa_h)(fmaxf((float)v[u][e], 0.0f) - (float)t2[u][e]);
        *(half8_t *)(p.out + (long)(m0 + ml) * p.ldo + n0 + nl) = o;
      }
    }
    return;
  }
  auto rows_pass = [&](auto ncols_c) {
  const int nc8 = ncols_c / 8;
  for (int c = tid; c < BM * nc8; c += NT) {
    const int ml = c / nc8, nl = (c % nc8) * 8;
    const int m = m0 + ml, n = n0 + nl;
    if (m >= p.M || n >= p.N) continue;
    half8_t v = *(const half8_t *)(Cs + ml * CROW + nl);
    const long o = (long)m * p.ldo + n;
    if (p.epi == HXA_EPI_PARTIAL) {
      *(half8_t *)(p.out + (long)z * p.out_zstride + o) = v;
    } else {
      if (p.epi == HXA_EPI_GELU_TANH) {  // (head-normed tiles never get here: whole tiles take the path above)
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = (hxa_h)gelu_tanh_f((float)v[e]);
      } else if (p.epi == HXA_EPI_GELU_ERF) {  // (without the T2 table, or with transposed columns)
        if (p.erf_t2) {
#pragma unroll
          for (int e = 0; e < 8; e++) v[e] = (hxa_h)gelu_erf_tab((float)v[e], p.erf_t2);
        } else {
#pragma unroll
          for (int e = 0; e < 8; e++) v[e] = (hxa_h)gelu_erf_f((float)v[e]);
        }
      }
      *(half8_t *)(p.out + o) = v;
    }
  }
  };
  if (p.out_t == nullptr)
    rows_pass(std::integral_constant<int, BN>{});
  else
    rows_pass(nsplit);
  if (nsplit < BN) {
    // transposed columns (a multiple of 32: split_col % 32 == 0): a thread takes 4 adjacent columns x 8 rows, read as
    // 8-byte LDS words, and writes four 16-byte runs of 8 rows, one per output row n of out_t. Four consecutive
    // threads take consecutive 8-row chunks of the same columns, so each store instruction writes 64-byte runs
    // (16 rows of out_t per wave) rather than 64 scattered 16-byte pieces; the LDS reads of those four threads are 8
    // rows apart (two-way bank conflicts).
    static_assert(BM % 32 == 0, "8-row chunks in fours");
    const int ngrp = (BN - nsplit) / 4;
    for (int c = tid; c < ngrp * (BM / 8); c += NT) {
      const int rest = c >> 2;
      const int nl = nsplit + (rest % ngrp) * 4, ml = ((rest / ngrp) * 4 + (c & 3)) * 8;
      const int m = m0 + ml;
      if (m >= p.M) continue;
      uint2_t w[8];
#pragma unroll
      for (int e = 0; e < 8; e++) w[e] = *(const uint2_t *)(Cs + (ml + e) * CROW + nl);
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int n = n0 + nl + q;
        if (n >= p.N) break;
        uint32_t o[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {  // rows 2k, 2k+1 of column q: halves (q & 1) of word (q >> 1)
          const uint32_t a = (q >> 1) ? w[2 * k].y : w[2 * k].x, b = (q >> 1) ? w[2 * k + 1].y : w[2 * k + 1].x;
          o[k] = __builtin_amdgcn_perm(b, a, (q & 1) ? 0x07060302u : 0x05040100u);
        }
        hxa_h *dst = p.out_t + (long)(n - p.split_col) * p.ldo_t + m;
        if (m + 7 < p.M) {
          *(uint4_t *)dst = (uint4_t){o[0], o[1], o[2], o[3]};
        } else {
          const half8_t v = __builtin_bit_cast(half8_t, (uint4_t){o[0], o[1], o[2], o[3]});
          for (int e = 0; e < 8 && m + e < p.M; e++) dst[e] = v[e];
        }
      }
    }
  }
}

// ---- fused cross attention (blk.c:163-169 in one kernel) ----
// After the main loop of a 128 x 128 fp16 tile of the cross-q projection (one head: the tile's 128 columns), the
// tile becomes that head's 128 queries: f16(acc) is staged in LDS and RMSNorm * gain is applied in place (kern.c:163-197,
// the head-norm epilogue's arithmetic), each of the 4 waves takes 32 queries as MFMA fragments, and the head's text
// keys are swept in 64-key tiles of K and V^T, double-buffered in LDS behind the query tile (the attention kernel's
// layouts: K rows in krow_key order, chunks XOR-swizzled), with the exact online softmax in fp32; O = f16(P V / l).
// LDS: the 128x128 fp16 ring of four stages [0, 128 KB). Its buffers 2 and 3 take key tiles 0 and 1 (K, then V^T, 16 KB
// each) as the ring's stages nst and nst + 1; buffers 0 and 1 become the query tile [128][136] fp16 and then the two-pass
// form's V^T tiles 2 and 3; that form's K tiles 2 and 3 are at XA_K23_OFF, loaded when the workgroup starts: 160 KB.
// (With a ring of two stages behind the key tiles the projection waits out the latency of every stage: 36.6 us at 512
// tokens x 2048, 256 keys, cold weights.)
constexpr int XA_KV_OFF = 2 * GemmGeo<128, 128, HXA_W_F16>::STAGE;
constexpr int XA_K23_OFF = XA_KV_OFF + 4 * 16384;
constexpr int XA_LDS = XA_K23_OFF + 2 * 16384;
static_assert(GemmGeo<128, 128, HXA_W_F16>::STAGE == 32768 && XA_KV_OFF >= GemmGeo<128, 128, HXA_W_F16>::C_BYTES &&
                  XA_LDS <= 160 * 1024,
              "fused cross-attention LDS layout");
// load l of key tile i of the workgroup's head and image, 1 KB per wave: l < 4 the K tile into kb (rows in krow_key order,
// 256 B each, chunk c at c ^ (row & 15)), else the V^T tile into vb + 16 KB (128 rows of 64 keys, chunk c at
// c ^ ((d >> 1) & 7)): the attention kernel's layouts. Keys past NKV read a valid row (probability 0).
HXA_DEV void xattn_load1(const GemmParams &p, int m0, int n0, int i, int l, int wave, int lane, uint8_t *kb, uint8_t *vb) {
  const int img = m0 / p.xa_T, h = n0 >> 7, key0 = i * 64, NKV = p.xa_nkv;
  const int blk = (l & 3) * 4 + wave;
  if (l < 4) {
    const hxa_h *kh = p.xa_k + (long)img * p.xa_kb + h * 128;
    const int row = 4 * blk + (lane >> 4), c = (lane & 15) ^ (row & 15);
    const int key = min(key0 + krow_key(row), NKV - 1);
    g2l16_opaque(kh + (long)key * p.xa_ldk + c * 8, kb + blk * 1024);
  } else {
    const hxa_h *vh = p.xa_vt + (long)img * p.xa_vb + (long)h * 128 * p.xa_ldvt;
    const int d = 8 * blk + (lane >> 3), c = (lane & 7) ^ ((d >> 1) & 7);
    int key = key0 + c * 8;
    if (key >= NKV) key = 0;
    g2l16_opaque(vh + (long)d * p.xa_ldvt + key, vb + 16384 + blk * 1024);
  }
}
HXA_DEV void xattn_load_k(const GemmParams &p, int m0, int n0, int i, int wave, int lane, uint8_t *kb) {
#pragma unroll
  for (int l = 0; l < 4; l++) xattn_load1(p, m0, n0, i, l, wave, lane, kb, kb);
}
HXA_DEV void xattn_load_v(const GemmParams &p, int m0, int n0, int i, int wave, int lane, uint8_t *vb) {
#pragma unroll
  for (int l = 4; l < 8; l++) xattn_load1(p, m0, n0, i, l, wave, lane, vb, vb - 16384);
}
// key tile i at its K / V^T buffer in the ring (the online form's tiles past the first two)
HXA_DEV void xattn_load_kv(const GemmParams &p, int m0, int n0, int i, int wave, int lane, uint8_t *lds8) {
  uint8_t *const b = lds8 + XA_KV_OFF + (i & 1) * 32768;
  xattn_load_k(p, m0, n0, i, wave, lane, b);
  xattn_load_v(p, m0, n0, i, wave, lane, b + 16384);
}
template <int MI, int NI>
HXA_DEV void xattn_tail(const GemmParams &p, const float4_t (&acc)[NI][MI], int m0, int n0, int tid, int lane, int wave,
                        int ml, int nl, uint8_t *lds8) {
  constexpr float L2E = 1.4426950408889634f, RESCALE_TH = 5.5f;
  constexpr int CROW = 136;
  const int g = lane >> 5, ql = lane & 31;
  const int h = n0 >> 7, ntiles = (p.xa_nvalid + 63) / 64;
  auto kbuf = [&](int i) { return lds8 + XA_KV_OFF + (i & 1) * 32768; };
  auto vbuf = [&](int i) { return kbuf(i) + 16384; };
  // the head's gains
  const int jj = tid & 7, r0 = tid >> 3;
  float glo[8], ghi[8];
  hn_gains(p, n0 + 8 * jj, glo);
  hn_gains(p, n0 + 64 + 8 * jj, ghi);
  wait_vm<0>();  // (and the main loop's trailing loads must land before its LDS ring is reused)
  __syncthreads();
  // stage f16(acc) as the row-major query tile
  hxa_h *Cs = (hxa_h *)lds8;
  stage_tile<MI, NI, CROW>(Cs, acc, ml, nl);
  __syncthreads();
  // RMSNorm * gain per query row, in place: 8 lanes per row (lane jj owns dims [8jj, 8jj+8) and [64+8jj, 64+8jj+8))
  {
    const float z8[8] = {};
#pragma unroll
    for (int it = 0; it < 4; it++) {
      hxa_h *row = Cs + (r0 + it * 32) * CROW;
      half8_t lo = *(const half8_t *)(row + 8 * jj), hi = *(const half8_t *)(row + 64 + 8 * jj);
      head_norm2(lo, hi, glo, ghi, false, z8, z8);
      *(half8_t *)(row + 8 * jj) = lo;
      *(half8_t *)(row + 64 + 8 * jj) = hi;
    }
  }
  __syncthreads();
  half8_t qf[8];
#pragma unroll
  for (int sd = 0; sd < 8; sd++) qf[sd] = *(const half8_t *)(Cs + (wave * 32 + ql) * CROW + sd * 16 + 8 * g);
  float16_t o[4];
#pragma unroll
  for (int d = 0; d < 4; d++) o[d] = (float16_t){};
  float mrun = -INFINITY, lsum = 0.0f;
  if (ntiles <= 4) {
    // Up to 256 keys: every tile stays in LDS (tiles 2 and 3 in the staging region, free once every wave holds its
    // q fragments), so the scores of all tiles are formed first and the row max is exact: no running rescale, and
    // the exponentials of tile t + 1 run between the P V MFMAs of tile t.
    // (K of tiles 2 and 3 was loaded with tiles 0 and 1 and has landed; their V^T goes to the staging region)
    __syncthreads();
    auto kt = [&](int t) -> const uint8_t * {
      return t < 2 ? kbuf(t) : lds8 + XA_K23_OFF + (t - 2) * 16384;
    };
    auto vt = [&](int t) -> const uint8_t * {
      return t < 2 ? vbuf(t) : lds8 + (t - 2) * 16384;
    };
    if (ntiles > 2) xattn_load_v(p, m0, n0, 2, wave, lane, lds8);
    if (ntiles > 3) xattn_load_v(p, m0, n0, 3, wave, lane, lds8 + 16384);
    const uint8_t *const kts[4] = {kt(0), kt(1), kt(2), kt(3)}, *const vts[4] = {vt(0), vt(1), vt(2), vt(3)};
    attn_two_pass(qf, kts, vts, ntiles, p.xa_nvalid, true, lane, o, lsum);
  } else {
  for (int i = 0; i < ntiles; i++) {
    if (i + 1 < ntiles) wait_vm<8>();  // tile i landed (tile i + 1 may still fly)
    else wait_vm<0>();
    reads_done_barrier();  // (tile i + 1's loads stay in flight)
    const uint8_t *kb = kbuf(i), *vb = vbuf(i);
    // every K fragment of the tile, then the V^T fragments, read ahead of the MFMAs that use them (the V^T reads
    // land during the QK MFMAs and the softmax)
    half8_t kf[8][2], vf[16];
#pragma unroll
    for (int ds = 0; ds < 8; ds++)
#pragma unroll
      for (int kb2 = 0; kb2 < 2; kb2++) {
        const int row = kb2 * 32 + ql, c = 2 * ds + g;
        kf[ds][kb2] = *(const half8_t *)(kb + row * 256 + ((c ^ (row & 15)) << 4));
      }
#pragma unroll
    for (int j = 0; j < 16; j++) {  // j = (kb2 * 2 + ks) * 4 + dblk
      const int dblk = j & 3, kk = j >> 2, d = dblk * 32 + ql, c = 2 * kk + g;
      vf[j] = *(const half8_t *)(vb + d * 128 + ((c ^ ((d >> 1) & 7)) << 4));
    }
    float16_t S[2];
    S[0] = (float16_t){};
    S[1] = (float16_t){};
#pragma unroll
    for (int ds = 0; ds < 8; ds++)
#pragma unroll
      for (int kb2 = 0; kb2 < 2; kb2++) S[kb2] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[ds][kb2], qf[ds], S[kb2], 0, 0, 0);
    const int key0 = i * 64;
    if (key0 + 64 > p.xa_nvalid) {
#pragma unroll
      for (int kb2 = 0; kb2 < 2; kb2++)
#pragma unroll
        for (int r = 0; r < 16; r++)
          if (key0 + kb2 * 32 + 16 * (r >> 3) + 8 * g + (r & 7) >= p.xa_nvalid) S[kb2][r] = -INFINITY;
    }
    float mt = -INFINITY;
#pragma unroll
    for (int kb2 = 0; kb2 < 2; kb2++)
#pragma unroll
      for (int r = 0; r < 16; r++) mt = fmaxf(mt, S[kb2][r]);
    {
      float lo, hi;
      halves(mt, lo, hi);
      mt = fmaxf(lo, hi);
    }
    const bool need = mt > mrun + RESCALE_TH;  // also while mrun is -inf
    if (__any(need)) {
      const float alpha = need ? __builtin_amdgcn_exp2f((mrun - mt) * L2E) : 1.0f;
      if (need) mrun = mt;
      lsum *= alpha;
#pragma unroll
      for (int d = 0; d < 4; d++) o[d] *= alpha;
    }
    const float mb = (mrun == -INFINITY ? 0.0f : mrun) * L2E;
    half8_t pf[2][2];
    float ls[2] = {0.0f, 0.0f};
#pragma unroll
    for (int kb2 = 0; kb2 < 2; kb2++)
#pragma unroll
      for (int r = 0; r < 16; r += 2) {  // fp16 pairs, summed by v_dot2 (the row sum of the fp16 P)
        const float p0 = __builtin_amdgcn_exp2f(fmaf(S[kb2][r], L2E, -mb));
        const float p1 = __builtin_amdgcn_exp2f(fmaf(S[kb2][r + 1], L2E, -mb));
        const half2_t h2 = {(hxa_h)p0, (hxa_h)p1};
        pf[kb2][r >> 3][r & 7] = h2[0];
        pf[kb2][r >> 3][(r & 7) + 1] = h2[1];
        ls[(r >> 1) & 1] = __builtin_amdgcn_fdot2(h2, (half2_t){(hxa_h)1.0f, (hxa_h)1.0f}, ls[(r >> 1) & 1], false);
      }
    lsum += ls[0] + ls[1];
#pragma unroll
    for (int j = 0; j < 16; j++)
      o[j & 3] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[j], pf[j >> 3][(j >> 2) & 1], o[j & 3], 0, 0, 0);
    if (i + 2 < ntiles) {
      reads_done_barrier();  // buffer i & 1 has been read by every wave
      xattn_load_kv(p, m0, n0, i + 2, wave, lane, lds8);
    }
  }
  }
  float llo, lhi;
  halves(lsum, llo, lhi);
  const float ltot = llo + lhi;
  const float inv = ltot > 0.0f ? 1.0f / ltot : 0.0f;
  half4_t v[4][4];
#pragma unroll
  for (int d = 0; d < 4; d++)
#pragma unroll
    for (int r4 = 0; r4 < 4; r4++)
#pragma unroll
      for (int e = 0; e < 4; e++) v[d][r4][e] = (hxa_h)(o[d][4 * r4 + e] * inv);
  // whole output rows, staged in the K-tile 2 / 3 region: unused with at most two key tiles, and with more every
  // wave has passed the barrier before tile 2's P V, so every QK pass is done (the online form never uses it)
  store_rows32(lds8 + XA_K23_OFF + wave * 8192, v, lane, p.xa_o + (long)(m0 + wave * 32) * p.xa_ldo + h * 128, p.xa_ldo,
               32);
}

// One output tile (and K slice z). NW = 4 (2 x 2 waves) or 8 (2 x 4, two per SIMD); each wave owns a (BM/2) x
// (BN / (NW/2)) sub-tile of v_mfma_f32_16x16x32_f16 blocks.
// What bounds it: at full occupancy of the chip the board's power limit, so the loop is built for few bytes and few
// register-file accesses per MAC. v_mfma_f32_16x16x32_f16 reads and writes half the accumulators per MAC of
// v_mfma_f32_32x32x16_f16 and the chip clocks 10% higher on it (4096 x 4096 x 2048 on 256x256 tiles: 61.9 us with
// 32x32x16, 55.3 us with this; both loops 1200 cycles per 32 k).
// Pipeline over slices of 32 k (two per stage): the MFMAs of a slice carry, a few per MFMA and pinned there by
// sched_barrier, the LDS reads of the next slice's fragments, the global -> LDS loads NS stages ahead and the
// dequantisation of the next W fragment. One barrier per stage, between its two slices: past it stage t + 1 has
// landed for every wave, and stage t has been read by every wave (lgkmcnt(0) before it), so its buffer takes the loads
// of stage t + NS. The loop this replaced (32-deep stages: half a 128-byte line per row, a step's LDS reads behind its
// loads) took, best tile to best tile, back to back: fp16 4096 x 2048 x 6144 115.6 -> 89.4 us, 1536 x 6144 x 2048 43.9 ->
// 38.6, 256 x 2048 x 2048 15.5 -> 9.7; int8 1024 x 2048 x 8192 42.2 -> 36.7, 1536 x 10240 x 2560 81.1 -> 72.4.
// k order: lane group h4 = lane / 16 takes the stage's k 16 h4 + 8 s .. + 7 in slice s, for A and W alike, so a lane's
// int8 (int4) values of both slices are one 16-byte (8-byte) LDS read and belong to one quantisation group. Every tile
// of this file uses this order, so its fp32 sums are the same whatever the tile; the skinny tiles (gemm_skinny.hip) use it within
// each of the four K quarters that they add at the end.
// An odd number of 32-k groups: stage 0 pairs group 0 with zeros, later stages start one group earlier.
// SPLIT2: the first and second halves of K are rounded to fp16 separately and combined in the residual epilogue,
// x += gate * (f16(first half) + f16(second half)) (blk.c:172-174 + kern.c:330-339 in one kernel): the first half's
// f16 accumulators are kept in registers while the second half accumulates.
template <int BM, int BN, int FMT, bool ASYM, bool SPLIT2, int NW, bool XATTN = false>
HXA_DEV void gemm_body(const GemmParams &p, const int bid, const int z) {
  using G = GemmGeo<BM, BN, FMT>;
  constexpr bool QW = FMT != HXA_W_F16;
  constexpr int NT = 64 * NW, WNW = NW / 2;
  constexpr int WTM = BM / 2, WTN = BN / WNW, MI = WTM / 16, NI = WTN / 16, NMF = MI * NI;
  constexpr bool DEEP = G::DEEP && !XATTN;
  constexpr int NS = G::NS, NA = G::NA, NLI = G::NLI, NL = (NLI + NW - 1) / NW;
  constexpr int NVEC = QW ? (ASYM ? 2 : 1) : 0;
  constexpr int LMIN = NLI / NW + NVEC;  // loads per stage that every wave issues
  static_assert(BM % 32 == 0 && BN % (16 * WNW) == 0 && (NW == 4 || NW == 8) && NA % NW == 0 && (BN / 4) % NW == 0 &&
                    G::W_BYTES % 1024 == 0 && (NS - 2) * LMIN < 64,
                "tile shape");
  extern __shared__ __attribute__((aligned(16))) uint8_t lds8[];

  int tm, tn;
  tile_coords(p, bid, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int ng = p.Kslice / 32, odd = ng & 1, nst = (ng + 1) >> 1, g0 = z * ng;
  const bool one = ng == 1;  // a single group: every stage loads it twice, the first copy zeroed
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1, h4 = lane >> 4, r16 = lane & 15;
  const HxaClkMark clk0 = clk_mark(p.clk);
  if constexpr (XATTN) {  // the two-pass form's K of key tiles 2 and 3, past the ring
    if (p.xa_nvalid > 128 && p.xa_nvalid <= 256) {
      xattn_load_k(p, m0, n0, 2, wave, lane, lds8 + XA_K23_OFF);
      if (p.xa_nvalid > 192) xattn_load_k(p, m0, n0, 3, wave, lane, lds8 + XA_K23_OFF + 16384);
    }
  }
  // ring buffer of stage 0. XATTN: such that the last stage sits in buffer 1 and buffers 2 and 3 are free at the end
  const int rot = XATTN ? (2 - nst) & 3 : 0;

  // ---- loader. 1 KB instruction t of a stage: 8 rows of A (t < NA) or 8 / 16 / 32 rows of fp16 / int8 / int4 W, 16
  // bytes per lane, XOR-swizzled so that 16 rows' equal chunks fall in distinct banks. The per-lane
  // offsets from the tile corner are fixed; a stage moves the wave-uniform bases. Rows past M / N clamp to the last.
  constexpr long ES = FMT == HXA_W_F16 ? 2 : 1;
  // group (0, 1) of the stage that this lane's chunk of instruction t belongs to
  auto chunk_of = [&](int t, int &row, int &c) {
    if (t < NA) {
      row = t * 8 + (lane >> 3);
      c = (lane & 7) ^ ((row >> 1) & 7);
      return c >> 2;
    }
    if constexpr (FMT == HXA_W_F16) {
      row = (t - NA) * 8 + (lane >> 3);
      c = (lane & 7) ^ ((row >> 1) & 7);
      return c >> 2;
    } else if constexpr (FMT == HXA_W_Q8) {
      row = (t - NA) * 16 + (lane >> 2);
      c = (lane & 3) ^ ((row >> 2) & 3);
      return c >> 1;
    } else {
      row = (t - NA) * 32 + (lane >> 1);
      c = (lane & 1) ^ ((row >> 3) & 1);
      return c;
    }
  };
  uint32_t off[NL], soff = 0;
#pragma unroll
  for (int l = 0; l < NL; l++) {
    const int t = min(l * NW + wave, NLI - 1);
    int row, c;
    const int g = one ? (chunk_of(t, row, c), 0) : chunk_of(t, row, c);
    if (t < NA) off[l] = ((uint32_t)(min(m0 + row, p.M - 1) - m0) * (uint32_t)p.lda + g * 32 + (c & 3) * 8) * 2u;
    else {
      const uint32_t r = (uint32_t)(min(n0 + row, p.N - 1) - n0) * (uint32_t)p.w_rs + g * (uint32_t)p.w_gs;
      off[l] = FMT == HXA_W_F16 ? (r + (c & 3) * 8) * 2u : FMT == HXA_W_Q8 ? r + (c & 1) * 16 : r;
    }
  }
  constexpr int CPW = QW ? BN / 4 / NW : 1;  // 16-byte chunks of the scale vectors per wave
  const int sg = one ? 0 : (wave * CPW + lane) / (BN / 8);  // their group
  if constexpr (QW) soff = ((uint32_t)sg * p.N + min(n0 + (wave * CPW + lane) % (BN / 8) * 8, p.N - 8)) * 2u;
  const uint8_t *const abase = (const uint8_t *)(p.A + (long)m0 * p.lda + (long)g0 * 32);
  const uint8_t *const wbase = (const uint8_t *)p.W + ((long)n0 * p.w_rs + (long)g0 * p.w_gs) * ES;
  const long wstep = p.w_gs * ES, sstep = 2L * p.N;
  [[maybe_unused]] const uint8_t *const sbase = (const uint8_t *)p.S + g0 * sstep, *const zbase = (const uint8_t *)p.Z + g0 * sstep;
  // load instruction l of this wave for stage t into ring buffer s; FIRST: stage 0 of an odd count, both groups group 0
  auto load1 = [&](int l, int t, int s, auto first_c) {
    constexpr bool FIRST = decltype(first_c)::value;
    const int g = FIRST || one ? 0 : 2 * min(t, nst - 1) - odd;  // stages past the end reload the last one (never used)
    const int ti = l * NW + wave;
    if (NLI % NW != 0 && ti >= NLI) return;
    const bool isa = l * NW < NA;  // NA % NW == 0: the same for every wave
    uint32_t o = off[l];
    if constexpr (FIRST) {
      int row, c;
      const int gi = chunk_of(ti, row, c);
      if (odd && gi && !one) o -= isa ? 64u : (uint32_t)wstep;
    }
    g2l16_sbase(isa ? abase + (long)g * 64 : wbase + g * wstep, o, lds8 + s * G::STAGE + ti * 1024);
  };
  auto load_vec = [&](int t, int s, auto first_c) {
    if constexpr (QW) {
      constexpr bool FIRST = decltype(first_c)::value;
      const int g = FIRST || one ? 0 : 2 * min(t, nst - 1) - odd;
      const uint8_t *sb = uniform_ptr(sbase + g * sstep), *zb = uniform_ptr(zbase + g * sstep);
      uint8_t *ws = lds8 + s * G::STAGE + G::A_BYTES + G::W_BYTES + 16 * wave * CPW;
      uint32_t o = soff;
      if constexpr (FIRST) {
        if (odd && sg) o -= (uint32_t)p.N * 2u;
      }
      if (lane < CPW) {
        g2l16_sbase(sb, o, ws);
        if constexpr (ASYM) g2l16_sbase(zb, o, ws + G::S_BYTES);
      }
    }
  };

  // XATTN: past the last stage come the first two key tiles (buffers 2 and 3, the attention's K / V^T buffers: as many
  // loads as a stage), so they arrive under the last stages' MFMAs
  auto load_x = [&](int l, int t, int s, auto kv_c) {
    if constexpr (decltype(kv_c)::value) {
      if (t == nst || t == nst + 1) {
        static_assert(NLI == 32 && NL == 8 && NW == 4 && NS == 4, "a key tile of K and V^T is one stage");
        xattn_load1(p, m0, n0, t - nst, l, wave, lane, lds8 + s * G::STAGE, lds8 + s * G::STAGE);
        return;
      }
    }
    load1(l, t, s, std::false_type{});
  };
  typedef std::integral_constant<bool, XATTN> xattn_c;

  // ---- fragments of a slice: A rows fa[set][i]; fp16 W rows fb[set][j]. Quantised W is read raw once per stage
  // (rw[j]: both slices) with its scale, and fragment j + 1 is dequantised under block row j's MFMAs (fb ring of two).
  typedef typename std::conditional<FMT == HXA_W_Q8, uint4_t, uint2_t>::type raw_t;
  // DEEP: the set of a stage is both slices, fa[set][2][MI] and fb[set][2][NI] (rw[set][NI]) flattened.
  constexpr int FS = DEEP ? 2 : 1;
  half8_t fa[2][FS * MI], fb[2][QW ? (DEEP ? 2 : 1) : FS * NI];
  [[maybe_unused]] raw_t rw[DEEP ? 2 : 1][NI];
  [[maybe_unused]] hxa_h sc[DEEP ? 2 : 1][NI], zc[DEEP ? 2 : 1][NI];
  auto rd_a = [&](int s, int ks, int i) {
    const int row = wm * WTM + i * 16 + r16;
    return *(const half8_t *)(lds8 + s * G::STAGE + row * 128 + (((2 * h4 + ks) ^ ((row >> 1) & 7)) << 4));
  };
  auto rd_w16 = [&](int s, int ks, int j) {
    const int row = wn * WTN + j * 16 + r16;
    return *(const half8_t *)(lds8 + s * G::STAGE + G::A_BYTES + row * 128 + (((2 * h4 + ks) ^ ((row >> 1) & 7)) << 4));
  };
  auto rd_raw = [&](int s, int set, int j) {
    if constexpr (QW) {
      const int row = wn * WTN + j * 16 + r16;
      const uint8_t *ws = lds8 + s * G::STAGE + G::A_BYTES;
      if constexpr (FMT == HXA_W_Q8) rw[set][j] = *(const uint4_t *)(ws + row * 64 + ((h4 ^ ((row >> 2) & 3)) << 4));
      else rw[set][j] = *(const uint2_t *)(ws + row * 32 + (((h4 >> 1) ^ ((row >> 3) & 1)) << 4) + ((h4 & 1) << 3));
      const hxa_h *sv = (const hxa_h *)(ws + G::W_BYTES) + (h4 >> 1) * BN + row;
      sc[set][j] = *sv;
      zc[set][j] = ASYM ? sv[G::S_BYTES / 2] : (hxa_h)0.0f;
    }
  };
  auto dequant = [&](int set, int ks, int j, half8_t &o8) {
    if constexpr (QW) {
      const half2_t s2 = {sc[set][j], sc[set][j]};
      uint32_t o[4];
      if constexpr (FMT == HXA_W_Q8) {
        dq8_word(rw[set][j][2 * ks], s2, o[0], o[1]);
        dq8_word(rw[set][j][2 * ks + 1], s2, o[2], o[3]);
      } else {
        const half2_t z2 = {zc[set][j], zc[set][j]};
        dq4_word<ASYM>(rw[set][j][ks], s2, z2, o);
      }
      o8 = __builtin_bit_cast(half8_t, (uint4_t){o[0], o[1], o[2], o[3]});
    }
  };

  float4_t acc[NI][MI];
#pragma unroll
  for (int j = 0; j < NI; j++)
#pragma unroll
    for (int i = 0; i < MI; i++) acc[j][i] = (float4_t){0.0f, 0.0f, 0.0f, 0.0f};

  // ---- prologue: NS stages in flight (the last one's second half goes out with slice 0 when NS > 2), stage 0 landed
  constexpr int H1 = NS > 2 && !DEEP ? NL / 2 : NL;  // loads of a stage issued right after the barrier; the rest a slice later
#pragma unroll
  for (int l = 0; l < NL; l++) load1(l, 0, rot, std::true_type{});
  load_vec(0, 0, std::true_type{});
#pragma unroll
  for (int s = 1; s < NS; s++) {
    load_vec(s, s, std::false_type{});
#pragma unroll
    for (int l = 0; l < (s == NS - 1 ? H1 : NL); l++) load_x(l, s, XATTN ? (rot + s) & 3 : s, xattn_c{});
  }
  wait_vm<(NS - 2) * LMIN>();
  __syncthreads();
  if (odd) {  // group "-1" of stage 0: zeros
    uint8_t *const l0 = lds8 + rot * G::STAGE;
    for (int i = tid; i < BM * 4; i += NT) {
      const int row = i >> 2, c = i & 3;
      *(uint4_t *)(l0 + row * 128 + ((c ^ ((row >> 1) & 7)) << 4)) = (uint4_t){0, 0, 0, 0};
    }
    if constexpr (!QW) {
      for (int i = tid; i < BN * 4; i += NT) {
        const int row = i >> 2, c = i & 3;
        *(uint4_t *)(l0 + G::A_BYTES + row * 128 + ((c ^ ((row >> 1) & 7)) << 4)) = (uint4_t){0, 0, 0, 0};
      }
    } else {
      for (int i = tid; i < BN; i += NT) {
        hxa_h *sv = (hxa_h *)(l0 + G::A_BYTES + G::W_BYTES) + i;
        sv[0] = (hxa_h)0.0f;
        if (ASYM) sv[G::S_BYTES / 2] = (hxa_h)0.0f;
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < NI; j++) {
    if constexpr (QW) rd_raw(0, 0, j);
    else {
      fb[0][j] = rd_w16(rot, 0, j);
      if constexpr (DEEP) fb[0][NI + j] = rd_w16(0, 1, j);
    }
  }
#pragma unroll
  for (int i = 0; i < MI; i++) {
    fa[0][i] = rd_a(rot, 0, i);
    if constexpr (DEEP) fa[0][MI + i] = rd_a(0, 1, i);
  }
  if constexpr (QW && !DEEP) dequant(0, 0, 0, fb[0][0]);

  // One slice: the MFMAs of fragment set ks; with them, in slot order, the reads of the next slice (slice nks of ring
  // buffer rs), the loads of stage lt into buffer ls, and (quantised W) the dequantisation of the next fragment. W
  // fragment ring: fragment j of either slice sits in fb[(ks * NI + j) & 1].
  auto slice = [&](auto ks_c, int rs, int lt, int ls, auto kv_c) {
    if constexpr (!DEEP) {
    constexpr int KS = decltype(ks_c)::value, NK = KS ^ 1;
    constexpr int RD = MI + (QW ? 0 : NI), RPS = (RD + NMF - 1) / NMF;
    constexpr int L0 = KS == 1 ? 0 : H1, L1 = KS == 1 ? H1 : NL, LN = L1 - L0;
#pragma unroll
    for (int q = 0; q < NMF; q++) {
      const int j = q / MI, i = q % MI;
      const half8_t w = fb[QW ? (KS * NI + j) & 1 : KS][QW ? 0 : j];
      acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w, fa[KS][i], acc[j][i], 0, 0, 0);
      if constexpr (QW) {
        // raw fragment j of the next stage, once this stage's second slice of it is dequantised
        if (KS == 1 && i == 0) rd_raw(rs, 0, j);
        if (i == MI / 2) {
          if (j + 1 < NI) dequant(0, KS, j + 1, fb[(KS * NI + j + 1) & 1][0]);
          else dequant(0, NK, 0, fb[(NK * NI) & 1][0]);
        }
      }
#pragma unroll
      for (int u = 0; u < RPS; u++) {
        const int x = q * RPS + u;
        if (x < RD) {
          if constexpr (QW) fa[NK][x] = rd_a(rs, NK, x);
          else if (x == 0) fb[NK][0] = rd_w16(rs, NK, 0);
          else if (x <= MI) fa[NK][x - 1] = rd_a(rs, NK, x - 1);
          else fb[NK][x - MI] = rd_w16(rs, NK, x - MI);
        }
      }
      if constexpr (LN > 0) {
#pragma unroll
        for (int l = 0; l < LN; l++)
          if (l * NMF / LN == q) load_x(L0 + l, lt, ls, kv_c);
      }
      if (KS == 1 && q == 0) load_vec(lt, ls, std::false_type{});
      if (q % 2 == 1 || q + 1 == NMF) __builtin_amdgcn_sched_barrier(0);
    }    }
  };
  // DEEP: one stage, both slices of it already in registers (set c): the reads of the next stage's fragments (set n)
  // first, so that they land during the MFMAs, then the loads of stage t + NS. Quantised W: fragment j + 1 of both
  // slices is dequantised under fragment j's MFMAs (fb[ring][slice]).
  auto stage = [&](int c, int n, int rs, int lt, int ls) {
    if constexpr (DEEP) {
      constexpr int RD = QW ? 2 * MI + NI : 2 * (MI + NI), RPS = (RD + NMF - 1) / NMF;
      if constexpr (QW) {
        dequant(c, 0, 0, fb[0][0]);
        dequant(c, 1, 0, fb[0][1]);
      }
#pragma unroll
      for (int q = 0; q < 2 * NMF; q++) {
        // fp16: slice 0's blocks, then slice 1's; quantised: both slices of one W fragment after another
        const int j = QW ? q / (2 * MI) : q % NMF / MI, ks = QW ? q % (2 * MI) / MI : q / NMF, i = q % MI;
        const half8_t w = QW ? fb[j & 1][ks] : fb[c][ks * NI + j];
        acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w, fa[c][ks * MI + i], acc[j][i], 0, 0, 0);
#pragma unroll
        for (int u = 0; u < RPS; u++) {
          const int x = q * RPS + u;
          if (x < RD) {
            if constexpr (QW) {
              if (x < NI) rd_raw(rs, n, x);
              else fa[n][x - NI] = rd_a(rs, (x - NI) / MI, (x - NI) % MI);
            } else {
              const int k2 = x / (MI + NI), y = x % (MI + NI);
              if (y < NI) fb[n][k2 * NI + y] = rd_w16(rs, k2, y);
              else fa[n][k2 * MI + y - NI] = rd_a(rs, k2, y - NI);
            }
          }
        }
        if constexpr (QW) {
          if (i == MI / 2 && j + 1 < NI) dequant(c, ks, j + 1, fb[(j + 1) & 1][ks]);
        }
        if (q == 0) load_vec(lt, ls, std::false_type{});
#pragma unroll
        for (int l = 0; l < NL; l++)
          if (l * 2 * NMF / NL == q) load1(l, lt, ls, std::false_type{});
        if (q % 2 == 1 || q + 1 == 2 * NMF) __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  // stage t + 1 landed for every wave, and this wave's LDS reads are in registers
  auto stage_barrier = [&]() {
    wait_vm<(NS - 2) * LMIN>();
    reads_done_barrier();
  };
  [[maybe_unused]] half4_t first[SPLIT2 ? NI : 1][SPLIT2 ? MI : 1];
  auto half_done = [&](int t) {
    if constexpr (SPLIT2) {
      if (t + 1 == nst / 2) {  // first half of K done: keep its fp16 rounding, restart the accumulators
#pragma unroll
        for (int j = 0; j < NI; j++)
#pragma unroll
          for (int i = 0; i < MI; i++) {
            first[j][i] = (half4_t){(hxa_h)acc[j][i][0], (hxa_h)acc[j][i][1], (hxa_h)acc[j][i][2], (hxa_h)acc[j][i][3]};
            acc[j][i] = (float4_t){0.0f, 0.0f, 0.0f, 0.0f};
          }
      }
    }
  };
  int cur = rot;
  if constexpr (DEEP) {
    auto step = [&](int t, int c) {
      const int nxt = cur + 1 == NS ? 0 : cur + 1;
      stage_barrier();
      stage(c, c ^ 1, nxt, t + NS, cur);
      cur = nxt;
      half_done(t);
    };
    for (int t = 0; t < nst; t += 2) {
      step(t, 0);
      if (t + 1 < nst) step(t + 1, 1);
    }
  } else {
    auto step = [&](int t, auto kv_c) {
      const int nxt = cur + 1 == NS ? 0 : cur + 1, prv = cur == 0 ? NS - 1 : cur - 1;
      slice(std::integral_constant<int, 0>{}, cur, t + NS - 1, prv, kv_c);
      stage_barrier();
      slice(std::integral_constant<int, 1>{}, nxt, t + NS, cur, kv_c);
      cur = nxt;
      half_done(t);
    };
    int t = 0;
    for (; t < (XATTN ? nst - NS : nst); t++) step(t, std::false_type{});
    if constexpr (XATTN) {
      for (; t < nst; t++) step(t, std::true_type{});
    }
  }
  clk_store(p.clk, (int)(blockIdx.x + blockIdx.z * gridDim.x), tid, clk0);
  const int ml = wm * WTM + r16, nl = wn * WTN + 4 * h4;
  if constexpr (XATTN) {
    xattn_tail<MI, NI>(p, acc, m0, n0, tid, lane, wave, ml, nl, lds8);
    return;
  }
  wait_vm<0>();  // the trailing (dummy) stage loads must land before the epilogue reuses the LDS ring
  if constexpr (!SPLIT2) {
    if (p.epi == HXA_EPI_PARTIAL_F32) {  // no LDS staging and no prefetch (gemm_prepare rejects pf with it)
      store_partial_f32<MI, NI>(p, acc, m0 + ml, n0 + nl, z);
      return;
    }
  }
  __syncthreads();
  if (p.pf_bytes > 0)
    prefetch_share(p, bid + z * p.tiles_m * p.tiles_n, p.tiles_m * p.tiles_n * (int)gridDim.z, tid, NT, lds8 + G::PF_OFF);
  hxa_h *Cs = (hxa_h *)lds8;
  stage_tile<MI, NI, G::CROW>(Cs, acc, ml, nl);
  if constexpr (SPLIT2) {
#pragma unroll
    for (int j = 0; j < NI; j++)
#pragma unroll
      for (int i = 0; i < MI; i++) *(half4_t *)(Cs + (BM + ml + i * 16) * G::CROW + nl + j * 16) = first[j][i];
  }
  __syncthreads();
  gemm_epilogue<BM, BN, NT, SPLIT2>(p, Cs, m0, n0, tid, z);
  if (p.pf_bytes > 0) wait_vm<0>();
}

// At least two waves per SIMD also for 4-wave kernels, so that the accumulators stay in the 256 directly addressable
// registers (with 512 the compiler kept them in AGPRs and copied them in and out around the MFMAs: 64x128 at 512 x 2048 x
// 2048 17.2 -> 13.8 us)
template <int BM, int BN, int FMT, bool ASYM, bool SPLIT2, int NW>
__global__ __launch_bounds__(64 * NW, 2) void gemm_kernel(GemmParams p) {
  if constexpr (NW == 8 && !SPLIT2) {
    if ((int)blockIdx.x >= p.tiles_m * p.tiles_n) {  // an appended workgroup: side GEMV rows, no LDS and no barrier
      side_gemv<2>(p.side, (blockIdx.x - p.tiles_m * p.tiles_n) * 8 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6),
                   p.side_wgs * 8, threadIdx.x & 63);
      return;
    }
  }
  gemm_body<BM, BN, FMT, ASYM, SPLIT2, NW>(p, blockIdx.x, blockIdx.z);
}
// two independent GEMMs of the same tile shape and weight format in one launch: workgroups [0, nwg0) run p0,
// the rest p1 (nwg0 a multiple of 8 keeps each GEMM's XCD placement)
template <int BM, int BN, int FMT, bool ASYM, int NW>
__global__ __launch_bounds__(64 * NW, 2) void gemm_pair_kernel(GemmParams p0, GemmParams p1, int nwg0) {
  if ((int)blockIdx.x < nwg0) gemm_body<BM, BN, FMT, ASYM, false, NW>(p0, blockIdx.x, 0);
  else gemm_body<BM, BN, FMT, ASYM, false, NW>(p1, blockIdx.x - nwg0, 0);
}
// G independent GEMMs of one tile shape and weight format, each with its own parameters (a device array): workgroup
// (x, y) runs tile x of GEMM y
template <int BM, int BN, int FMT, bool ASYM, int NW>
__global__ __launch_bounds__(64 * NW) void gemm_group_kernel(const GemmParams *__restrict__ ps) {
  gemm_body<BM, BN, FMT, ASYM, false, NW>(ps[blockIdx.y], blockIdx.x, 0);
}

// ---- launches of one weight format (explicitly instantiated in that format's translation unit) ----
template <int BM, int BN, int FMT, bool ASYM, bool SPLIT2, int NW>
hipError_t launch_t(const GemmParams &p, int ksplit, hipStream_t st) {
  auto kern = gemm_kernel<BM, BN, FMT, ASYM, SPLIT2, NW>;
  using G = GemmGeo<BM, BN, FMT>;
  constexpr int base = G::lds(G::NS), lds = SPLIT2 && 2 * G::C_BYTES > base ? 2 * G::C_BYTES : base;
  constexpr int most = !SPLIT2 && G::lds_erf(G::NS) > lds ? G::lds_erf(G::NS) : lds;
  static_assert(most <= 160 * 1024, "LDS");
  static bool attr = false;
  if (!attr) {
    hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, most);
    if (e != hipSuccess) return e;
    attr = true;
  }
  const dim3 grid(p.tiles_m * p.tiles_n + (NW == 8 && !SPLIT2 && ksplit == 1 ? p.side_wgs : 0), 1, ksplit);
  if (!SPLIT2 && p.epi == HXA_EPI_GELU_ERF && p.erf_t2 != nullptr) {  // the T2 table past the staged tile
    GemmParams pe = p;
    pe.erf_lds = G::ERF_OFF;
    hxa_launch(kern, grid, dim3(64 * NW), most, st, pe);
  } else {
    hxa_launch(kern, grid, dim3(64 * NW), lds, st, p);
  }
  return hipGetLastError();
}
template <int BM, int BN, int FMT, bool ASYM, int NW>
hipError_t launch_pair_t(const GemmParams &p0, const GemmParams &p1, hipStream_t st) {
  auto kern = gemm_pair_kernel<BM, BN, FMT, ASYM, NW>;
  constexpr int lds = GemmGeo<BM, BN, FMT>::lds(GemmGeo<BM, BN, FMT>::NS);
  static bool attr = false;
  if (!attr) {
    hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
    attr = true;
  }
  const int n0 = p0.tiles_m * p0.tiles_n;
  hxa_launch(kern, dim3(n0 + p1.tiles_m * p1.tiles_n), dim3(64 * NW), lds, st, p0, p1, n0);
  return hipGetLastError();
}

// The waves a tile runs on, as measured: 8 (two per SIMD) for the tiles above 128x128; 4 for 64x64 and 128x64 (half the
// LDS reads per MFMA of 8 narrower waves); 128x128 4 with fp16 weights (1024 x 2048 x 2048 in two K slices 13.6 against
// 14.6 us), 8 with quantised ones (the other wave's MFMAs cover the dequantisation: int8 16.8 against 15.7 us), and so
// 64x128 (int8 512 x 2048 x 2048 in four slices 12.5 against 15.3 us).
constexpr int tile_nw(int bm, int bn, int fmt) {
  if (bm * bn > 128 * 128) return 8;
  if (bm * bn < 128 * 128 && bn == 64) return 4;
  return fmt == HXA_W_F16 ? 4 : 8;
}
// a single GEMM on tile bm x bn (tile_built says which exist)
template <int FMT, bool ASYM>
hipError_t launch_fmt(int bm, int bn, const GemmParams &p, int ksplit, hipStream_t st) {
#define HXG_TILE(BM, BN) \
  if (bm == BM && bn == BN) return launch_t<BM, BN, FMT, ASYM, false, tile_nw(BM, BN, FMT)>(p, ksplit, st);
  HXG_TILE(256, 256)
  HXG_TILE(256, 192)
  HXG_TILE(192, 256)
  HXG_TILE(192, 192)
  HXG_TILE(256, 128)
  HXG_TILE(128, 256)
  HXG_TILE(192, 128)
  HXG_TILE(128, 128)
  HXG_TILE(64, 128)
  HXG_TILE(64, 64)
  if constexpr (FMT != HXA_W_Q4) {
    HXG_TILE(128, 64)
  }
#undef HXG_TILE
  return hipErrorInvalidValue;
}
template <int FMT, bool ASYM>
hipError_t launch_split2(int bm, int bn, const GemmParams &p, hipStream_t st) {
  if (bm == 128 && bn == 128) return launch_t<128, 128, FMT, ASYM, true, 4>(p, 1, st);
  if (bm == 64 && bn == 128) return launch_t<64, 128, FMT, ASYM, true, 4>(p, 1, st);
  return hipErrorInvalidValue;
}
template <int FMT, bool ASYM>
hipError_t launch_pair_fmt(int bm, int bn, const GemmParams &p0, const GemmParams &p1, hipStream_t st) {
  if (bm == 128 && bn == 128) return launch_pair_t<128, 128, FMT, ASYM, tile_nw(128, 128, FMT)>(p0, p1, st);
  if (bm == 192 && bn == 256) return launch_pair_t<192, 256, FMT, ASYM, 8>(p0, p1, st);
  return hipErrorInvalidValue;
}
// the grouped launch's tile is 192x256, 8 waves
template <int FMT, bool ASYM>
hipError_t launch_group_fmt(const GemmParams *ps, int G, int tiles, hipStream_t st) {
  auto kern = gemm_group_kernel<192, 256, FMT, ASYM, 8>;
  constexpr int lds = GemmGeo<192, 256, FMT>::lds(GemmGeo<192, 256, FMT>::NS);
  static bool attr = false;
  if (!attr) {
    hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
    attr = true;
  }
  hxa_launch(kern, dim3(tiles, G), dim3(512), lds, st, ps);
  return hipGetLastError();
}
hipError_t launch_xattn(const GemmParams &p, hipStream_t st);  // gemm_f16.hip
hipError_t launch_skinny(int bm, int fmt, bool asym, const GemmParams &p, hipStream_t st);  // gemm_skinny.hip: bm 32, 64

#define HXG_LAUNCHES(X, FMT, ASYM)                                                                                   \
  X template hipError_t launch_fmt<FMT, ASYM>(int, int, const GemmParams &, int, hipStream_t);                       \
  X template hipError_t launch_split2<FMT, ASYM>(int, int, const GemmParams &, hipStream_t);                         \
  X template hipError_t launch_pair_fmt<FMT, ASYM>(int, int, const GemmParams &, const GemmParams &, hipStream_t); \
  X template hipError_t launch_group_fmt<FMT, ASYM>(const GemmParams *, int, int, hipStream_t);
#ifndef HXG_INSTANTIATE
HXG_LAUNCHES(extern, HXA_W_F16, false)
HXG_LAUNCHES(extern, HXA_W_Q8, false)
HXG_LAUNCHES(extern, HXA_W_Q4, false)
HXG_LAUNCHES(extern, HXA_W_Q4, true)
#endif
}  // namespace hxg
