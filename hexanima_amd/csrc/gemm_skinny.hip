// The plain linear of few output tiles: O[M][N] = f16(A[M][K] . W[N][K]^T) on 64x32 or 32x32 tiles, K split over the 4 waves
// of a workgroup.
#include "gemm_kernel.h"

namespace hxg {

// Stage (64 k) of one wave: A rows of 128 B, W rows (fp16 128 B, int8 64 B, int4 32 B), the two groups' scale (and offset)
// vectors; swizzled like gemm_body's stages.
template <int BM, int FMT>
struct SkinnyGeo {
  static constexpr int BN = 32, NW = 4;
  static constexpr int A_BYTES = BM * 128, W_BYTES = BN * (FMT == HXA_W_F16 ? 128 : FMT == HXA_W_Q8 ? 64 : 32);
  static constexpr int S_BYTES = FMT == HXA_W_F16 ? 0 : BN * 4;
  static constexpr int STAGE = A_BYTES + W_BYTES + 2 * S_BYTES;
  static constexpr int NS = 160 * 1024 / (NW * STAGE) < 6 ? 160 * 1024 / (NW * STAGE) : 6;
  static constexpr int SROW = BN + 4;  // fp32 row stride of a wave's staged sums (spreads 16 rows' chunks over the banks)
  static constexpr int LDS = NW * NS * STAGE > NW * BM * SROW * 4 ? NW * NS * STAGE : NW * BM * SROW * 4;
};

// One BM x 32 output tile per workgroup; wave w takes the w-th quarter of K, in stages of 64. Where the tiles of
// gemm_kernel.h leave most CUs idle, a launch's time is a chain of K / 64 stages, each behind a barrier; here a wave has a
// ring of its own in LDS and waits for nothing but its own loads, the chain is a quarter as long, and the waves' fp32
// sums meet in LDS once (added in wave order: the result does not depend on timing). Bound by latency (a chain of K / 256
// stages) and by the CU's global -> LDS rate (BM + 32 rows read for 32 columns). The loads go through LDS because a
// fragment's consecutive lanes are different rows: loaded straight into registers they fetch 16 bytes per address and ran
// at 16 - 18 B / clk a CU.
// Measured (cold weights, back to back; before: the fastest of one launch and split-K with a sum): int8 256 x 2048 x 2048
// 13.3 -> 7.7 us, 64 x 2048 x 2048 9.8 -> 6.9, 1562 x 3072 x 128 (M x K x N) 20.9 (one launch) -> 10.1, 1562 x 8192 x 128
// 48.7 (one launch) -> 18.4; fp16 256 x 2048 x 2048 11.9 -> 9.4.
template <int BM, int FMT, bool ASYM>
__global__ __launch_bounds__(256, 2) void gemm_skinny_kernel(GemmParams p) {
  using G = SkinnyGeo<BM, FMT>;
  constexpr int BN = G::BN, NW = G::NW, NS = G::NS, MI = BM / 16, NI = BN / 16;
  constexpr bool QW = FMT != HXA_W_F16;
  constexpr int NA = G::A_BYTES / 1024, NL = NA + G::W_BYTES / 1024, L = NL + (QW ? ASYM ? 2 : 1 : 0);
  static_assert(NS >= 3 && NS * L < 64, "ring");
  extern __shared__ __attribute__((aligned(16))) uint8_t lds8[];
  // workgroup b runs on XCD b % 8: XCD x takes the x-th eighth of the tiles in the order that repeats the larger operand's
  // rows, so that each is read through one XCD's L2
  const int nt = p.tiles_m * p.tiles_n, x = blockIdx.x & 7, q = nt >> 3, r = nt & 7;
  const int tile = x * q + min(x, r) + (blockIdx.x >> 3);
  int tm, tn;
  if ((long)p.M * 2 > (long)p.N * (FMT == HXA_W_F16 ? 2 : 1)) {
    tm = tile / p.tiles_n;
    tn = tile - tm * p.tiles_n;
  } else {
    tn = tile / p.tiles_m;
    tm = tile - tn * p.tiles_m;
  }
  const int m0 = tm * BM, n0 = tn * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h4 = lane >> 4, r16 = lane & 15;
  const HxaClkMark clk0 = clk_mark(p.clk);
  const int ns = p.Ktot / 64, s0 = wave * ns / NW, n = (wave + 1) * ns / NW - s0;  // stages [s0, s0 + n)
  uint8_t *const ring = lds8 + wave * NS * G::STAGE;

  // loader: 1 KB instruction l of a stage, 8 rows of A (l < NA) or 8 / 16 / 32 rows of fp16 / int8 / int4 W; rows past M /
  // N clamp to the last
  constexpr long ES = FMT == HXA_W_F16 ? 2 : 1;
  uint32_t off[NL], soff = 0;
#pragma unroll
  for (int l = 0; l < NL; l++) {
    if (l < NA) {
      const int row = l * 8 + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
      off[l] = ((uint32_t)(min(m0 + row, p.M - 1) - m0) * (uint32_t)p.lda + c * 8) * 2u;
    } else {
      int row, g, c;  // row, k group of the stage, 16-byte chunk of the group
      if constexpr (FMT == HXA_W_F16) {
        row = (l - NA) * 8 + (lane >> 3);
        c = (lane & 7) ^ ((row >> 1) & 7);
        g = c >> 2, c &= 3;
      } else if constexpr (FMT == HXA_W_Q8) {
        row = (l - NA) * 16 + (lane >> 2);
        c = (lane & 3) ^ ((row >> 2) & 3);
        g = c >> 1, c &= 1;
      } else {
        row = (l - NA) * 32 + (lane >> 1);
        g = (lane & 1) ^ ((row >> 3) & 1), c = 0;
      }
      off[l] = ((uint32_t)(min(n0 + row, p.N - 1) - n0) * (uint32_t)p.w_rs + g * (uint32_t)p.w_gs) * (uint32_t)ES + c * 16;
    }
  }
  // (lanes 0 .. BN / 4 - 1: 8 scales each, N % 8 == 0)
  if constexpr (QW) soff = ((uint32_t)(lane / (BN / 8)) * p.N + min(n0 + lane % (BN / 8) * 8, p.N - 8)) * 2u;
  const uint8_t *const abase = (const uint8_t *)(p.A + (long)m0 * p.lda);
  const uint8_t *const wbase = (const uint8_t *)p.W + (long)n0 * p.w_rs * ES;
  const long wstep = 2 * p.w_gs * ES, sstep = 4L * p.N;
  auto load = [&](int t, int s) {  // stage t of this wave into ring buffer s
    const long g = s0 + t;
    uint8_t *const b = ring + s * G::STAGE;
#pragma unroll
    for (int l = 0; l < NL; l++) g2l16_sbase(l < NA ? abase + g * 128 : wbase + g * wstep, off[l], b + l * 1024);
    if constexpr (QW) {
      const uint8_t *sb = uniform_ptr((const uint8_t *)p.S + g * sstep), *zb = uniform_ptr((const uint8_t *)p.Z + g * sstep);
      if (lane < BN / 4) {
        g2l16_sbase(sb, soff, b + G::A_BYTES + G::W_BYTES);
        if constexpr (ASYM) g2l16_sbase(zb, soff, b + G::A_BYTES + G::W_BYTES + G::S_BYTES);
      }
    }
  };

  // fragments of a stage (two sets): lane (h4, r16) holds k 16 h4 .. + 15 of row r16, two MFMAs of 8 each
  typedef typename std::conditional<FMT == HXA_W_F16, half8_t,
                                    typename std::conditional<FMT == HXA_W_Q8, uint4_t, uint2_t>::type>::type raw_t;
  half8_t fa[2][MI][2];
  raw_t fw[2][NI][QW ? 1 : 2];
  [[maybe_unused]] hxa_h sc[2][NI], zc[2][NI];
  auto read = [&](int u, int s) {
    const uint8_t *const b = ring + s * G::STAGE, *const ws = b + G::A_BYTES;
#pragma unroll
    for (int j = 0; j < NI; j++) {
      const int row = j * 16 + r16;
      if constexpr (FMT == HXA_W_F16) {
#pragma unroll
        for (int k = 0; k < 2; k++)
          fw[u][j][k] = *(const half8_t *)(ws + row * 128 + (((2 * h4 + k) ^ ((row >> 1) & 7)) << 4));
      } else {
        if constexpr (FMT == HXA_W_Q8) fw[u][j][0] = *(const uint4_t *)(ws + row * 64 + ((h4 ^ ((row >> 2) & 3)) << 4));
        else fw[u][j][0] = *(const uint2_t *)(ws + row * 32 + (((h4 >> 1) ^ ((row >> 3) & 1)) << 4) + ((h4 & 1) << 3));
        const hxa_h *sv = (const hxa_h *)(ws + G::W_BYTES) + (h4 >> 1) * BN + row;
        sc[u][j] = *sv;
        if constexpr (ASYM) zc[u][j] = sv[G::S_BYTES / 2];
      }
    }
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
      for (int k = 0; k < 2; k++) {
        const int row = i * 16 + r16;
        fa[u][i][k] = *(const half8_t *)(b + row * 128 + (((2 * h4 + k) ^ ((row >> 1) & 7)) << 4));
      }
  };
  float4_t acc[NI][MI];
#pragma unroll
  for (int j = 0; j < NI; j++)
#pragma unroll
    for (int i = 0; i < MI; i++) acc[j][i] = (float4_t){0.0f, 0.0f, 0.0f, 0.0f};
  auto mac = [&](int u) {
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
      for (int j = 0; j < NI; j++) {
        half8_t w;
        if constexpr (FMT == HXA_W_F16) {
          w = fw[u][j][k];
        } else {
          const half2_t s2 = {sc[u][j], sc[u][j]};
          uint32_t o[4];
          if constexpr (FMT == HXA_W_Q8) {
            dq8_word(fw[u][j][0][2 * k], s2, o[0], o[1]);
            dq8_word(fw[u][j][0][2 * k + 1], s2, o[2], o[3]);
          } else {
            const hxa_h zz = ASYM ? zc[u][j] : (hxa_h)0.0f;
            dq4_word<ASYM>(fw[u][j][0][k], s2, (half2_t){zz, zz}, o);
          }
          w = __builtin_bit_cast(half8_t, (uint4_t){o[0], o[1], o[2], o[3]});
        }
#pragma unroll
        for (int i = 0; i < MI; i++) acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w, fa[u][i][k], acc[j][i], 0, 0, 0);
      }
  };
  // stage t has landed: the loads of the `newer` stages issued after it may still fly
  auto landed = [&](int newer) {
    if (newer >= NS - 1) wait_vm<(NS - 1) * L>();
    else if (newer == 2) wait_vm<2 * L>();
    else if (newer == 1) wait_vm<L>();
    else if (newer <= 0) wait_vm<0>();
    else wait_vm<3 * L>();
    asm volatile("" ::: "memory");
  };
  // stage t's fragments are in registers: its buffer takes stage t + NS
  auto refill = [&](int t, int s) {
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    asm volatile("" ::: "memory");
    if (t + NS < n) load(t + NS, s);
  };
#pragma unroll
  for (int s = 0; s < NS; s++)
    if (s < n) load(s, s);
  if (n > 0) {
    landed(min(n, NS) - 1);
    read(0, 0);
    refill(0, 0);
  }
  int cur = 0;
  auto step = [&](int t, int u) {  // stage t is in set u
    if (t + 1 < n) {
      const int nxt = cur + 1 == NS ? 0 : cur + 1;
      landed(min(n - 1, t + NS) - (t + 1));
      read(u ^ 1, nxt);
      mac(u);
      refill(t + 1, nxt);
      cur = nxt;
    } else {
      mac(u);
    }
  };
  for (int t = 0; t < n; t += 2) {
    step(t, 0);
    if (t + 1 < n) step(t + 1, 1);
  }
  clk_store(p.clk, (int)blockIdx.x, tid, clk0);

  // block (j, i): row 16 i + r16, columns 16 j + 4 h4 .. + 3
  __syncthreads();  // every wave's ring is dead
  float *const part = (float *)lds8, *const mine = part + wave * BM * G::SROW;
#pragma unroll
  for (int j = 0; j < NI; j++)
#pragma unroll
    for (int i = 0; i < MI; i++) *(float4_t *)(mine + (i * 16 + r16) * G::SROW + j * 16 + 4 * h4) = acc[j][i];
  __syncthreads();
#pragma unroll
  for (int i = tid; i < BM * BN / 4; i += 64 * NW) {
    const int row = i >> 3, c = (i & 7) * 4;
    if (m0 + row >= p.M || n0 + c >= p.N) continue;  // N % 8 == 0: four columns are inside N or past it
    float4_t s = *(const float4_t *)(part + row * G::SROW + c);
#pragma unroll
    for (int w = 1; w < NW; w++) s += *(const float4_t *)(part + (w * BM + row) * G::SROW + c);
    *(half4_t *)(p.out + (long)(m0 + row) * p.ldo + n0 + c) = (half4_t){(hxa_h)s[0], (hxa_h)s[1], (hxa_h)s[2], (hxa_h)s[3]};
  }
}

template <int BM, int FMT, bool ASYM>
static hipError_t launch_skinny_t(const GemmParams &p, hipStream_t st) {
  auto kern = gemm_skinny_kernel<BM, FMT, ASYM>;
  constexpr int lds = SkinnyGeo<BM, FMT>::LDS;
  static bool attr = false;
  if (!attr) {
    const hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
    attr = true;
  }
  hxa_launch(kern, dim3(p.tiles_m * p.tiles_n), dim3(256), lds, st, p);
  return hipGetLastError();
}
template <int FMT, bool ASYM>
static hipError_t launch_skinny_fmt(int bm, const GemmParams &p, hipStream_t st) {
  return bm == 32 ? launch_skinny_t<32, FMT, ASYM>(p, st) : launch_skinny_t<64, FMT, ASYM>(p, st);
}
hipError_t launch_skinny(int bm, int fmt, bool asym, const GemmParams &p, hipStream_t st) {
  if (fmt == HXA_W_F16) return launch_skinny_fmt<HXA_W_F16, false>(bm, p, st);
  if (fmt == HXA_W_Q8) return launch_skinny_fmt<HXA_W_Q8, false>(bm, p, st);
  return asym ? launch_skinny_fmt<HXA_W_Q4, true>(bm, p, st) : launch_skinny_fmt<HXA_W_Q4, false>(bm, p, st);
}
}  // namespace hxg
