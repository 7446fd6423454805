// Weight-only-quantised / fp16 GEMM for gfx950: O[M][N] = A[M][K] . W[N][K]^T with fused epilogues -- the host side
// (validation, tile choice, launches), the dequantisation pass and the split-K sum. Device code: gemm_kernel.h.
#include <mutex>

#include "gemm_kernel.h"

using namespace hxg;

namespace {

__device__ __align__(16) hxa_h g_erf_t2[ERF_T2_N];
__global__ __launch_bounds__(256) void erf_t2_kernel(hxa_h *t) {
  const int b = blockIdx.x * 256 + threadIdx.x;
  if (b >= ERF_T2_N) return;
  t[b] = gelu_t2((float)__builtin_bit_cast(hxa_h, (uint16_t)b));
}
// Tile cost model, per weight format (fp16, int8, int4): a launch of `rounds` rounds of workgroups over the CUs takes
// about rounds * (a * BM * BN * Kslice / 1e6 + b) + c microseconds. a, b, c >= 0 were fitted by least squares on the
// relative error to every tile timed on 289 (M, N, K, slices) of 32 - 6656 rows on a 256-CU MI355X, weights k-tiled, each
// launch repeated until the chip is at its power limit (where the block runner's chains keep it; a few launches after a
// pause clock higher and rank the tiles differently); the int4 column (but 64x64) anew, the tiles near the fastest weighing
// most, on 22 row counts x 15 shapes since its dequantisation takes 13 operations. With weights that come cold from HBM, as a
// block's do, fp16 and int8 launches take 10 - 40% longer than modelled, but the ranking holds: over those 330 shapes in one,
// two and four slices, cold weights, the picks are 1.0% (fp16), 0.3% (int8) and 0.4% (int4) above the fastest tile. a = 0
// marks a tile that format does not use. nw is the wave count under which hxa_gemm_tile takes the tile (tile_nw says what it
// runs on).
struct TileCost {
  int bm, bn, nw;
  float a[3], b[3], c[3];
};
constexpr TileCost kTiles[] = {
    {256, 256, 9, {0.2831f, 0.3081f, 0.3194f}, {7.81f, 8.13f, 12.77f}, {0.00f, 0.00f, 0.00f}},
    {256, 192, 9, {0.3031f, 0.3574f, 0.3756f}, {6.67f, 7.38f, 10.18f}, {0.00f, 0.00f, 0.00f}},
    {192, 256, 9, {0.3003f, 0.3604f, 0.3646f}, {6.89f, 7.32f, 10.46f}, {0.00f, 0.00f, 0.00f}},
    {192, 192, 4, {0.3291f, 0.4331f, 0.4576f}, {6.27f, 6.77f, 8.13f}, {0.00f, 0.00f, 0.17f}},
    {256, 128, 4, {0.3210f, 0.3878f, 0.4312f}, {5.91f, 6.09f, 8.46f}, {0.00f, 0.00f, 0.00f}},
    {128, 256, 9, {0.3341f, 0.4520f, 0.4403f}, {6.10f, 6.37f, 8.09f}, {0.00f, 0.00f, 0.00f}},
    {192, 128, 8, {0.3586f, 0.4163f, 0.4906f}, {5.60f, 5.81f, 6.87f}, {0.00f, 0.00f, 0.33f}},
    {128, 128, 4, {0.4027f, 0.5403f, 0.6007f}, {4.98f, 4.81f, 5.00f}, {0.00f, 0.00f, 1.08f}},
    {64, 128, 4, {0.5433f, 0.7834f, 0.8009f}, {1.64f, 0.78f, 0.59f}, {2.30f, 3.99f, 4.89f}},
    {128, 64, 4, {0.5638f, 0.6793f, 0.0000f}, {1.67f, 0.76f, 0.00f}, {2.00f, 4.33f, 0.00f}},
    {64, 64, 4, {0.7294f, 0.9569f, 0.9919f}, {1.14f, 0.62f, 0.00f}, {2.40f, 4.51f, 6.74f}},
};

// CUs of the device current at the first call (read once, thread-safe; 256 when the query fails)
int num_cu() {
  static const int n = [] {
    int dev = 0, c = 0;
    if (hipGetDevice(&dev) != hipSuccess) dev = 0;
    return hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && c > 0 ? c : 256;
  }();
  return n;
}

}  // namespace

// Choose the tile of least modelled time (kTiles). The model sees the rounds, not how much of them lies past the edges of M and
// N; so of two tiles above 128x128 within 1% of each other the one that covers at least 8% less is taken (1152 rows x 8192
// columns: 256x192 covers 1280 rows in 215 workgroups, 192x256 1152 in 192; int8, K 2048: 51.1 and 48.0 us, K 3072 x 9216 78.9
// and 69.7. By any smaller difference there is nothing to gain: over 100 such pairs as many lose as win). HXA_EPI_RESADD_SPLIT2
// keeps both K halves' accumulators in registers and runs on the 4-wave 128x128 / 64x128 tiles only (ranked with the fp16 costs).
static void pick_tile(int M, int N, int K, int ksplit, int fmt, int epi, int hn_cols, int *bm, int *bn, int *nw) {
  const bool headnorm = hn_cols > 0;
  const bool split2 = epi == HXA_EPI_RESADD_SPLIT2;
  const int ncu = num_cu();
  const int f = split2 ? 0 : fmt;
  auto grid = [&](const TileCost &c) { return (long)((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn); };
  auto time = [&](const TileCost &c) {  // < 0: not for this GEMM
    if (c.a[f] == 0.0f) return -1.0;
    if (split2 && !(c.bn == 128 && (c.bm == 128 || c.bm == 64) && c.nw == 4)) return -1.0;  // register budget
    if (epi == HXA_EPI_SITU && c.bn % 128 != 0) return -1.0;  // each wave needs whole (up, gate) block pairs
    if (headnorm && (c.bn % 128 != 0 || (hn_cols % c.bn != 0 && hn_cols < N))) return -1.0;  // whole head-normed tiles
    const long waves = (grid(c) * ksplit + ncu - 1) / ncu;
    return (double)waves * (c.a[f] * 1e-6 * c.bm * c.bn * (double)(K / ksplit) + c.b[f]) + c.c[f];
  };
  auto covers = [&](const TileCost &c) { return (double)grid(c) * c.bm * c.bn; };
  const TileCost *pick = nullptr;
  double best = 0.0;
  for (const TileCost &c : kTiles) {
    const double t = time(c);
    if (t >= 0.0 && (pick == nullptr || t < best - 1e-9)) {
      best = t;
      pick = &c;
    }
  }
  if (pick == nullptr) return;
  double least = 0.92 * covers(*pick);
  for (const TileCost &c : kTiles) {
    if (pick->bm * pick->bn <= 128 * 128 || c.bm * c.bn <= 128 * 128 || covers(c) >= least) continue;
    const double t = time(c);
    if (t < 0.0 || t > 1.01 * best) continue;
    least = covers(c);
    pick = &c;
  }
  *bm = pick->bm;
  *bn = pick->bn;
  *nw = pick->nw;
}

// the modelled time (us) of the tile pick_tile chooses for a plain-store GEMM with ksplit slices
static double tile_time(int M, int N, int K, int ksplit, int fmt) {
  int bm = 128, bn = 128, nw = 4;
  pick_tile(M, N, K, ksplit, fmt, HXA_EPI_STORE, 0, &bm, &bn, &nw);
  const int ncu = num_cu();
  for (const TileCost &c : kTiles) {
    if (c.bm != bm || c.bn != bn || c.nw != nw) continue;
    const long tiles = (long)((M + bm - 1) / bm) * ((N + bn - 1) / bn) * ksplit;
    return (double)((tiles + ncu - 1) / ncu) * (c.a[fmt] * 1e-6 * bm * bn * (double)(K / ksplit) + c.b[fmt]) + c.c[fmt];
  }
  return 1e30;
}
double hxa_gemm_model_us(int M, int N, int K, int fmt, int ksplit) {
  return tile_time(M, N, K, ksplit, fmt & ~HXA_W_KTILED);
}
// split-K linear cost terms: the sum kernel's launch (us) and the bytes per us of the slices' round trip through L2 /
// MALL, fitted with the gain below to one launch, two and four slices timed on 258 (M, N, K, format) of 16 - 4096 rows
// (geometric mean of choice / fastest form 1.008; the worst 1.42, fp16 544 x 12288 -> 3072); kSplitGain: the
// factor by which a split form must beat the form before it. Four int8 / int4 slices only need to tie with two.
constexpr double kSumLaunchUs = 2.0, kSumBytesPerUs = 12.0e6, kSplitGain = 0.95;

// the tiles launch_fmt has kernels for (split2: launch_split2's), under the wave counts hxa_gemm_tile takes for them: a
// tile has one kernel per weight format, whichever of its nw names it
static bool tile_built(int bm, int bn, int nw, int fmt, bool split2) {
  if (split2) return nw == 4 && bn == 128 && (bm == 128 || bm == 64);
  if (bn == 32) return nw == 4 && (bm == 64 || bm == 32);  // gemm_skinny.hip: plain stores only (gemm_prepare)
  const bool q4 = fmt == HXA_W_Q4;
  if (nw == 9) return (bn == 256 && (bm == 256 || bm == 192 || bm == 128)) || (bm == 256 && bn == 192) ||
                      ((bm == 128 || bm == 192 || bm == 256) && bn == 128 && !q4);
  if (nw == 8) return (bm == 192 || bm == 128) && (bn == 256 || bn == 128);
  if (nw != 4) return false;
  if (bm == 128 && bn == 64) return !q4;
  return (bm == 192 && (bn == 256 || bn == 192 || bn == 128)) || (bm == 256 && bn == 128) ||
         (bm == 128 && (bn == 256 || bn == 128)) || (bm == 64 && (bn == 128 || bn == 64));
}

// The device address of the GELU-erf T2 table on the current device, filled on first use there (a launch of
// erf_t2_kernel on `st`, waited for, so the table is complete for every later launch on any stream). Under stream
// capture an unfilled table is not filled (the epilogue then evaluates erfcf): null.
const hxa_h *erf_table(hipStream_t st) {
  static const hxa_h *tab[HXA_MAX_DEVICES];
  static std::mutex mu;
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= HXA_MAX_DEVICES) return nullptr;
  std::lock_guard<std::mutex> lk(mu);
  if (tab[dev]) return tab[dev];
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(st, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone) return nullptr;
  void *ptr = nullptr;
  if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(g_erf_t2)) != hipSuccess || ptr == nullptr) return nullptr;
  hxa_launch(erf_t2_kernel, dim3(ERF_T2_N / 256), dim3(256), 0, st, (hxa_h *)ptr);
  if (hipGetLastError() != hipSuccess || hipStreamSynchronize(st) != hipSuccess) return nullptr;
  tab[dev] = (const hxa_h *)ptr;
  return tab[dev];
}

// validate a GEMM description, fill its kernel parameters and choose (or take the forced) tile
static int gemm_prepare(const HxaGemm &g, GemmParams &p, int &bm, int &bn, int &nw, HxaWeight &w, bool &split2) {
  w = *g.w;
  const int wkt = (w.fmt & HXA_W_KTILED) ? 1 : 0;
  w.fmt &= ~HXA_W_KTILED;
  if (g.M <= 0 || w.N <= 0 || w.K <= 0 || g.ksplit < 1) return HXA_E_ARG;
  if (w.K % (32 * g.ksplit) != 0) return HXA_E_ARG;
  if (w.fmt != HXA_W_F16 && w.s == nullptr) return HXA_E_ARG;
  if (g.epi == HXA_EPI_SITU && (w.N % 64) != 0) return HXA_E_ARG;
  if ((g.lda % 8) != 0 || ((uintptr_t)g.A % 16) != 0 || ((uintptr_t)w.w % 16) != 0) return HXA_E_ARG;
  if (w.N % 8 != 0) return HXA_E_ARG;  // 16-byte epilogue chunks
  split2 = g.epi == HXA_EPI_RESADD_SPLIT2;
  if (split2 && (g.ksplit != 1 || w.K % 128 != 0)) return HXA_E_ARG;  // two halves of whole k-step pairs
  if (g.epi == HXA_EPI_RESADD || split2
          ? ((g.ldx % 8) != 0 || ((uintptr_t)g.x % 32) != 0 || ((uintptr_t)g.gate % 32) != 0)
          : ((g.ldo % (g.epi == HXA_EPI_PARTIAL_F32 ? 4 : 8)) != 0 || ((uintptr_t)g.out % 16) != 0))
    return HXA_E_ARG;
  const bool f32 = g.epi == HXA_EPI_PARTIAL_F32;
  if (f32 && (g.out_t != nullptr || g.hn_cols > 0 || g.pf_bytes > 0 || g.side != nullptr)) return HXA_E_ARG;
  p = GemmParams{};
  if (g.epi == HXA_EPI_STORE_T) {  // all columns transposed
    p.out_t = g.out;
    p.ldo_t = g.ldo;
    p.split_col = 0;
  } else if (g.epi == HXA_EPI_STORE && g.out_t != nullptr) {  // fused projections: the tail columns transposed
    if (g.split_col % 32 != 0 || g.split_col < 0 || g.split_col > w.N) return HXA_E_ARG;
    p.out_t = g.out_t;
    p.ldo_t = g.ldo_t;
    p.split_col = g.split_col;
  }
  if (p.out_t != nullptr && ((p.ldo_t % 8) != 0 || ((uintptr_t)p.out_t % 16) != 0)) return HXA_E_ARG;
  p.A = g.A;
  p.lda = g.lda;
  p.W = w.w;
  p.S = w.s;
  p.Z = w.z;
  {
    const long cb = w.fmt == HXA_W_Q4 ? 16 : 32;  // elements (q4: bytes) of one row's k group
    p.w_rs = wkt ? cb : (long)w.K / 32 * cb;
    p.w_gs = wkt ? cb * w.N : cb;
  }
  // the loaders' per-lane offsets within a stage (up to 256 rows, two k groups) are unsigned 32-bit
  {
    const long es = w.fmt == HXA_W_F16 ? 2 : 1;
    if (g.lda >= (1L << 22) || p.w_rs * es >= (1L << 23)) return HXA_E_ARG;
    if ((255 * p.w_rs + p.w_gs + 32) * es >= (1L << 32) || 4L * w.N >= (1L << 32)) return HXA_E_ARG;
  }
  p.M = g.M;
  p.N = w.N;
  p.Ktot = w.K;
  p.Kslice = w.K / g.ksplit;
  p.epi = split2 ? HXA_EPI_RESADD : g.epi;
  p.out = g.epi == HXA_EPI_STORE_T || f32 ? nullptr : g.out;
  p.out32 = f32 ? (float *)g.out : nullptr;
  p.ldo = g.ldo;
  p.out_zstride = g.out_zstride;
  p.x = g.x;
  p.ldx = g.ldx;
  p.gate = g.gate;
  const bool headnorm = g.hn_cols > 0;
  if (headnorm) {
    if (g.epi != HXA_EPI_STORE || g.ksplit != 1 || g.hn_cols % 128 || w.N % 128 || !g.hn_g0 || !g.hn_g1 ||
        (g.hn_cos && (!g.hn_sin || g.hn_ttab <= 0)) || ((uintptr_t)g.hn_g0 | (uintptr_t)g.hn_g1) % 16 ||
        (g.out_t && (g.split_col % 128 || g.split_col < g.hn_cols)))
      return HXA_E_ARG;
  }
  p.hn_cols = headnorm ? min(g.hn_cols, w.N) : 0;
  p.hn_gsplit = g.hn_gsplit;
  p.hn_ttab = g.hn_ttab;
  p.hn_g0 = g.hn_g0;
  p.hn_g1 = g.hn_g1;
  p.hn_cos = g.hn_cos;
  p.hn_sin = g.hn_sin;
  // the prefetch rides on epilogues that issue no loads of their own (their waits would wait for it too)
  if (g.pf_bytes > 0 && (g.pf == nullptr || g.pf_bytes < 4 || ((uintptr_t)g.pf & 3) || headnorm ||
                         g.epi == HXA_EPI_RESADD || split2))
    return HXA_E_ARG;
  p.pf = (const uint8_t *)g.pf;
  p.pf_bytes = g.pf_bytes > 0 ? g.pf_bytes : 0;
  p.clk = g_hxa_clk_gemm;
  bm = 128;
  bn = 128;
  nw = 4;
  pick_tile(g.M, w.N, w.K, g.ksplit, w.fmt, g.epi, headnorm ? min(g.hn_cols, w.N) : 0, &bm, &bn, &nw);
  if (g.force_bm) {
    bm = g.force_bm;
    bn = g.force_bn;
    nw = g.force_nw ? g.force_nw : 4;
    if (!tile_built(bm, bn, nw, w.fmt, split2)) return HXA_E_ARG;
    if (g.epi == HXA_EPI_SITU && bn % 128 != 0) return HXA_E_ARG;
    if (bn == 32 && (w.K % 64 != 0 || g.epi != HXA_EPI_STORE || g.ksplit != 1 || p.out_t != nullptr || p.pf_bytes > 0)) return HXA_E_ARG;
    if (headnorm && (bn % 128 != 0 || (p.hn_cols % bn != 0 && p.hn_cols < w.N))) return HXA_E_ARG;
  }
  p.tiles_m = (g.M + bm - 1) / bm;
  p.tiles_n = (w.N + bn - 1) / bn;
  // 8 XCD rectangles of the fewest A + W bytes per k step (each XCD's L2 then serves its CUs' shared rows)
  p.xcd_gm = 0;
  {
    const long wrow = w.fmt == HXA_W_F16 ? 64 : (w.fmt == HXA_W_Q8 ? 32 : 16);
    long best = -1;
    for (int gm = 1; gm <= 8; gm *= 2) {
      if (p.tiles_m % gm || p.tiles_n % (8 / gm)) continue;
      const long bytes = (long)(p.tiles_m / gm) * bm * 64 + (long)(p.tiles_n / (8 / gm)) * bn * wrow;
      if (best < 0 || bytes < best) {
        best = bytes;
        p.xcd_gm = gm;
      }
    }
  }
  return HXA_OK;
}

int hxa_gemm_launch(const HxaGemm &g, hipStream_t st) {
  GemmParams p;
  int bm, bn, nw;
  HxaWeight w;
  bool split2;
  const int r = gemm_prepare(g, p, bm, bn, nw, w, split2);
  if (r != HXA_OK) return r;
  if (g.epi == HXA_EPI_GELU_ERF) p.erf_t2 = erf_table(st);
  hipError_t e;
  if (split2) {
    if (w.fmt == HXA_W_F16) e = launch_split2<HXA_W_F16, false>(bm, bn, p, st);
    else if (w.fmt == HXA_W_Q8) e = launch_split2<HXA_W_Q8, false>(bm, bn, p, st);
    else if (w.z) e = launch_split2<HXA_W_Q4, true>(bm, bn, p, st);
    else e = launch_split2<HXA_W_Q4, false>(bm, bn, p, st);
    return e == hipSuccess ? HXA_OK : HXA_E_HIP;
  }
  // a side GEMV rides in the CUs an 8-wave grid leaves idle in its last round (at least 16 of them), else it
  // runs as its own launch after the GEMM
  bool side_after = false;
  if (g.side != nullptr) {
    const HxaSideGemv &sg = *g.side;
    if (!hxa_side_k_ok(sg.K) || sg.N <= 0 || sg.per <= 0 || !sg.x || !sg.W || !sg.y ||
        ((uintptr_t)sg.x | (uintptr_t)sg.W) % 16)
      return HXA_E_ARG;
    const int ncu = num_cu(), tiles = p.tiles_m * p.tiles_n, idle = (tiles + ncu - 1) / ncu * ncu - tiles;
    if (tile_nw(bm, bn, w.fmt) == 8 && bn > 32 && g.ksplit == 1 && idle >= 16) {
      p.side = sg;
      p.side_wgs = idle;
    } else {
      side_after = true;
    }
  }
  if (bn == 32) e = launch_skinny(bm, w.fmt, w.z != nullptr, p, st);
  else if (w.fmt == HXA_W_F16) e = launch_fmt<HXA_W_F16, false>(bm, bn, p, g.ksplit, st);
  else if (w.fmt == HXA_W_Q8) e = launch_fmt<HXA_W_Q8, false>(bm, bn, p, g.ksplit, st);
  else if (w.z) e = launch_fmt<HXA_W_Q4, true>(bm, bn, p, g.ksplit, st);
  else e = launch_fmt<HXA_W_Q4, false>(bm, bn, p, g.ksplit, st);
  if (e != hipSuccess) return HXA_E_HIP;
  if (side_after) {
    const HxaSideGemv &sg = *g.side;
    return hxa_modgemv_launch(sg.x, sg.K, sg.W, sg.N, sg.y, sg.per, sg.ostride, sg.split, sg.gap, sg.act, st);
  }
  return HXA_OK;
}

long hxa_gemm_group_param_bytes(int G) { return (long)G * (long)sizeof(GemmParams); }

int hxa_gemm_group_prepare(const HxaGemm *g, int G, void *params_host, int *tiles, int *fmt) {
  if (G < 1 || !g || !params_host || !tiles || !fmt) return HXA_E_ARG;
  GemmParams *ps = (GemmParams *)params_host;
  for (int i = 0; i < G; i++) {
    if (g[i].ksplit != 1 || g[i].pf_bytes > 0 || g[i].M != g[0].M || !g[i].w || !g[0].w || g[i].w->N != g[0].w->N ||
        g[i].w->K != g[0].w->K || (g[i].w->fmt & ~HXA_W_KTILED) != (g[0].w->fmt & ~HXA_W_KTILED) ||
        (g[i].w->z != nullptr) != (g[0].w->z != nullptr))
      return HXA_E_ARG;
    HxaGemm gf = g[i];
    gf.force_bm = 192;
    gf.force_bn = 256;
    gf.force_nw = 9;
    int bm, bn, nw;
    HxaWeight w;
    bool split2;
    const int r = gemm_prepare(gf, ps[i], bm, bn, nw, w, split2);
    if (r != HXA_OK) return r;
    if (split2 || bm != 192 || bn != 256 || nw != 9) return HXA_E_ARG;
    ps[i].clk = HxaClk{nullptr, 0};  // the parameters outlive any clock record
    *fmt = w.fmt | (w.z ? 0x100 : 0);
  }
  *tiles = ps[0].tiles_m * ps[0].tiles_n;
  return HXA_OK;
}


int hxa_gemm_group_launch(const void *params_dev, int G, int tiles, int fmt, hipStream_t st) {
  if (!params_dev || G < 1 || G > 65535 || tiles < 1) return HXA_E_ARG;
  const GemmParams *ps = (const GemmParams *)params_dev;
  hipError_t e;
  switch (fmt) {
    case HXA_W_F16: e = launch_group_fmt<HXA_W_F16, false>(ps, G, tiles, st); break;
    case HXA_W_Q8: e = launch_group_fmt<HXA_W_Q8, false>(ps, G, tiles, st); break;
    case HXA_W_Q4: e = launch_group_fmt<HXA_W_Q4, false>(ps, G, tiles, st); break;
    case HXA_W_Q4 | 0x100: e = launch_group_fmt<HXA_W_Q4, true>(ps, G, tiles, st); break;
    default: return HXA_E_ARG;
  }
  return e == hipSuccess ? HXA_OK : HXA_E_HIP;
}

// the tiles with a paired kernel
static bool pair_tile(int bm, int bn) { return (bm == 128 && bn == 128) || (bm == 192 && bn == 256); }

bool hxa_gemm_pair_fits(const HxaGemm &g0, const HxaGemm &g1) {
  GemmParams p0, p1;
  int bm, bn, nw, bm1, bn1, nw1;
  HxaWeight w0, w1;
  bool s0, s1;
  if (gemm_prepare(g0, p0, bm, bn, nw, w0, s0) != HXA_OK || s0 || g0.ksplit != 1 || g1.ksplit != 1) return false;
  if (!pair_tile(bm, bn) || (p0.tiles_m * p0.tiles_n) % 8) return false;
  HxaGemm g1f = g1;
  g1f.force_bm = bm;
  g1f.force_bn = bn;
  g1f.force_nw = nw;
  if (gemm_prepare(g1f, p1, bm1, bn1, nw1, w1, s1) != HXA_OK || s1 || w0.fmt != w1.fmt || (w0.z != nullptr) != (w1.z != nullptr))
    return false;
  const long n0 = (long)p0.tiles_m * p0.tiles_n, n1 = (long)p1.tiles_m * p1.tiles_n;
  const long c = num_cu();
  return (n0 + n1 + c - 1) / c == (n0 + c - 1) / c;
}

bool hxa_gemm_xattn_fits(int M, int N) {
  return (long)((M + 127) / 128) * ((N + 127) / 128) <= num_cu();
}

int hxa_gemm_xattn_launch(const HxaGemm &g, const HxaXAttn &a, hipStream_t st) {
  if (g.side != nullptr) return HXA_E_ARG;  // (no side GEMV: only hxa_gemm_launch hosts one)
  if (g.w == nullptr || (g.w->fmt & ~HXA_W_KTILED) != HXA_W_F16 || g.epi != HXA_EPI_STORE || g.ksplit != 1 ||
      g.hn_cols < g.w->N || g.hn_cos != nullptr || g.out_t != nullptr || g.pf_bytes > 0)
    return HXA_E_ARG;
  // (NKV % 8: a V^T chunk of 8 keys that starts below NKV ends within it)
  if (a.T <= 0 || a.T % 128 || g.M % a.T || g.w->N % 128 || a.NKV < 1 || a.NKV % 8 || a.nvalid < 1 || a.nvalid > a.NKV ||
      !a.k || !a.vt || !a.o)
    return HXA_E_ARG;
  if ((a.ldk % 8) || (a.ldvt % 8) || (a.ldo % 4) || a.ldvt < a.NKV || (((uintptr_t)a.k | (uintptr_t)a.vt) % 16) ||
      ((uintptr_t)a.o % 8) || (a.kb % 8) || (a.vb % 8) || a.ldk >= (1L << 24) || a.ldvt >= (1L << 23))
    return HXA_E_ARG;
  HxaGemm gf = g;
  gf.force_bm = 128;
  gf.force_bn = 128;
  gf.force_nw = 4;
  GemmParams p;
  int bm, bn, nw;
  HxaWeight w;
  bool split2;
  const int r = gemm_prepare(gf, p, bm, bn, nw, w, split2);
  if (r != HXA_OK) return r;
  p.xa_k = a.k;
  p.xa_vt = a.vt;
  p.xa_o = a.o;
  p.xa_ldk = a.ldk;
  p.xa_ldvt = a.ldvt;
  p.xa_ldo = a.ldo;
  p.xa_kb = a.kb;
  p.xa_vb = a.vb;
  p.xa_nkv = a.NKV;
  p.xa_nvalid = a.nvalid;
  p.xa_T = a.T;
  return launch_xattn(p, st) == hipSuccess ? HXA_OK : HXA_E_HIP;
}

int hxa_gemm_plan(const HxaGemm &g, int *bm, int *bn, int *nw, int *rounds) {
  GemmParams p;
  HxaWeight w;
  bool split2;
  const int r = gemm_prepare(g, p, *bm, *bn, *nw, w, split2);
  if (r != HXA_OK) return r;
  const long n = (long)p.tiles_m * p.tiles_n * g.ksplit;
  *rounds = (int)((n + num_cu() - 1) / num_cu());
  return HXA_OK;
}

int hxa_gemm_pair_launch(const HxaGemm &g0, const HxaGemm &g1, hipStream_t st) {
  if (g0.side != nullptr || g1.side != nullptr) return HXA_E_ARG;  // (only hxa_gemm_launch hosts a side GEMV)
  GemmParams p0, p1;
  int bm, bn, nw, bm1, bn1, nw1;
  HxaWeight w0, w1;
  bool s0, s1;
  int r = gemm_prepare(g0, p0, bm, bn, nw, w0, s0);
  if (r != HXA_OK) return r;
  hipError_t e = hipErrorInvalidValue;
  // paired on the 128x128 and 192x256 tiles; the second GEMM then takes the first
  // one's tile. The 192x256 pair only where the second GEMM's tiles fit in the CUs the first leaves idle: a
  // further round of 192x256 tiles is slower than the second GEMM's own launch (6144 x 2048 cross q + 512-row text
  // k / v: 79 us paired, 70 us as two launches)
  if (pair_tile(bm, bn) && !s0 && g0.ksplit == 1 && g1.ksplit == 1 && (p0.tiles_m * p0.tiles_n) % 8 == 0) {
    HxaGemm g1f = g1;
    g1f.force_bm = bm;
    g1f.force_bn = bn;
    g1f.force_nw = nw;
    r = gemm_prepare(g1f, p1, bm1, bn1, nw1, w1, s1);
    if (r != HXA_OK) return r;
    if (g0.epi == HXA_EPI_GELU_ERF) p0.erf_t2 = erf_table(st);
    if (g1.epi == HXA_EPI_GELU_ERF) p1.erf_t2 = erf_table(st);
    const long n0 = (long)p0.tiles_m * p0.tiles_n, n1 = (long)p1.tiles_m * p1.tiles_n;
    const long c = num_cu();
    const bool extra_round = (n0 + n1 + c - 1) / c > (n0 + c - 1) / c;
    if (w0.fmt == w1.fmt && (w0.z != nullptr) == (w1.z != nullptr) && !s1 && !(bn == 256 && extra_round)) {
      if (w0.fmt == HXA_W_F16) e = launch_pair_fmt<HXA_W_F16, false>(bm, bn, p0, p1, st);
      else if (w0.fmt == HXA_W_Q8) e = launch_pair_fmt<HXA_W_Q8, false>(bm, bn, p0, p1, st);
      else if (w0.z) e = launch_pair_fmt<HXA_W_Q4, true>(bm, bn, p0, p1, st);
      else e = launch_pair_fmt<HXA_W_Q4, false>(bm, bn, p0, p1, st);
    }
  }
  if (e == hipErrorInvalidValue) {  // not pairable: two launches, each on its own tile
    r = hxa_gemm_launch(g0, st);
    return r != HXA_OK ? r : hxa_gemm_launch(g1, st);
  }
  return e == hipSuccess ? HXA_OK : HXA_E_HIP;
}

// ---- int8 / int4 weights -> fp16, k-tiled [K/32][N][32] (the layout the fp16 kernels read) ----
// One 8-k slot of one row per thread (the 16-byte fragment unit of the main loops), dequantised with their own
// dq8_word / dq4_word, so the values are the same f16(q * s) (+ z) bits the fused path feeds its MFMAs. Reads
// w.w / w.s / w.z once (the weights with non-temporal loads), writes 2 N K bytes.
namespace {
template <int FMT, bool ASYM>
__global__ __launch_bounds__(256) void dequant_kernel(GemmParams p, hxa_h *out) {
  const long t = (long)blockIdx.x * 256 + threadIdx.x;  // 8-k slot c = t % 4 of group i = t / 4 (g = i / N, n = i % N)
  const long i = t >> 2;
  const int c = (int)(t & 3);
  if (i >= (long)(p.Ktot / 32) * p.N) return;
  const long g = i / p.N, n = i % p.N;
  const hxa_h s = p.S[i];
  const half2_t s2 = {s, s};
  const hxa_h z = ASYM ? p.Z[i] : (hxa_h)0.0f;
  const half2_t z2 = {z, z};
  const uint8_t *src = (const uint8_t *)p.W + n * p.w_rs + g * p.w_gs;
  uint32_t o[4];
  if constexpr (FMT == HXA_W_Q8) {
    const uint2_t v = __builtin_nontemporal_load((const uint2_t *)(src + 8 * c));
    dq8_word(v.x, s2, o[0], o[1]);
    dq8_word(v.y, s2, o[2], o[3]);
  } else {
    dq4_word<ASYM>(__builtin_nontemporal_load((const uint32_t *)(src + 4 * c)), s2, z2, o);
  }
  // lanes write consecutive 16-byte chunks: 1 KB per wave store
  *(uint4_t *)(out + i * 32 + c * 8) = (uint4_t){o[0], o[1], o[2], o[3]};
}
}  // namespace

int hxa_dequant_launch(const HxaWeight &w0, hxa_h *out, hipStream_t st) {
  HxaWeight w = w0;
  const int wkt = (w.fmt & HXA_W_KTILED) ? 1 : 0;
  w.fmt &= ~HXA_W_KTILED;
  if ((w.fmt != HXA_W_Q8 && w.fmt != HXA_W_Q4) || w.s == nullptr || w.N <= 0 || w.K <= 0 || w.K % 32 != 0)
    return HXA_E_ARG;
  if (((uintptr_t)w.w % 16) != 0 || ((uintptr_t)out % 16) != 0) return HXA_E_ARG;
  GemmParams p{};
  p.W = w.w;
  p.S = w.s;
  p.Z = w.z;
  p.N = w.N;
  p.Ktot = w.K;
  const long cb = w.fmt == HXA_W_Q4 ? 16 : 32;
  p.w_rs = wkt ? cb : (long)w.K / 32 * cb;
  p.w_gs = wkt ? cb * w.N : cb;
  const long slots = (long)(w.K / 32) * w.N * 4;
  const dim3 grid((unsigned)((slots + 255) / 256));
  if (w.fmt == HXA_W_Q8) hxa_launch((dequant_kernel<HXA_W_Q8, false>), grid, dim3(256), 0, st, p, out);
  else if (w.z) hxa_launch((dequant_kernel<HXA_W_Q4, true>), grid, dim3(256), 0, st, p, out);
  else hxa_launch((dequant_kernel<HXA_W_Q4, false>), grid, dim3(256), 0, st, p, out);
  return hipGetLastError() == hipSuccess ? HXA_OK : HXA_E_HIP;
}

// ---- split-K linear: fp32 slice sums added in order and rounded once
// out[m][n] = f16(p[0] + p[1] + ... + p[S-1]) at element (m, n) of each slice; one thread per 8 columns of a row
__global__ __launch_bounds__(256) void sum_partials_kernel(const float *__restrict__ p, int S, long zstride, long ldp,
                                                           int M, int N, hxa_h *__restrict__ out, long ldo) {
  const int c8 = N / 8;
  const long c = (long)blockIdx.x * 256 + threadIdx.x;
  if (c >= (long)M * c8) return;
  const int m = (int)(c / c8), n = (int)(c % c8) * 8;
  const float *src = p + (long)m * ldp + n;
  float4_t a0 = *(const float4_t *)src, a1 = *(const float4_t *)(src + 4);
  for (int z = 1; z < S; z++) {
    const float *q = src + (long)z * zstride;
    a0 += *(const float4_t *)q;
    a1 += *(const float4_t *)(q + 4);
  }
  const half8_t o = {(hxa_h)a0[0], (hxa_h)a0[1], (hxa_h)a0[2], (hxa_h)a0[3],
                     (hxa_h)a1[0], (hxa_h)a1[1], (hxa_h)a1[2], (hxa_h)a1[3]};
  *(half8_t *)(out + (long)m * ldo + n) = o;
}

int hxa_sum_partials_launch(const float *p, int S, long zstride, long ldp, int M, int N, hxa_h *out, long ldo,
                            hipStream_t st) {
  if (!p || !out || S < 1 || M <= 0 || N <= 0 || N % 8 || ldp < N || ldo < N || ldp % 4 || ldo % 8 ||
      (S > 1 && zstride < (long)M * ldp) || zstride % 4 || ((uintptr_t)p | (uintptr_t)out) % 16)
    return HXA_E_ARG;
  const long chunks = (long)M * (N / 8);
  hxa_launch(sum_partials_kernel, dim3((unsigned)((chunks + 255) / 256)), dim3(256), 0, st, p, S, zstride, ldp, M, N,
             out, ldo);
  return hipGetLastError() == hipSuccess ? HXA_OK : HXA_E_HIP;
}

// gemm_skinny_kernel's cost model, like kTiles: rounds * (a * K / 1000 + b) + c us, fitted to 16 - 1562 rows x 35 shapes
// per format (cold weights, row counts up to 3 rounds; int4 to 132 shapes since its dequantisation takes 13 operations)
constexpr struct {
  int bm;
  double a[3], b[3], c[3];
} kSkinny[] = {{64, {2.18, 2.00, 1.95}, {3.19, 3.48, 2.40}, {0.0, 0.0, 1.19}},
               {32, {1.57, 1.59, 1.57}, {2.52, 2.39, 1.89}, {0.63, 1.05, 1.33}}};
// the row count (64, 32) of the skinny tile whose modelled time is below t us, else 0
static int skinny_rows(int M, int N, int K, int fmt, double t) {
  if (K % 64 != 0) return 0;
  int bm = 0;
  for (const auto &c : kSkinny) {
    const long tiles = (long)((M + c.bm - 1) / c.bm) * ((N + 31) / 32), ncu = num_cu();
    const double ts = (double)((tiles + ncu - 1) / ncu) * (c.a[fmt] * 1e-3 * K + c.b[fmt]) + c.c[fmt];
    if (ts < t) {
      t = ts;
      bm = c.bm;
    }
  }
  return bm;
}
int hxa_skinny_rows(int M, int N, int K, int fmt) {
  fmt &= ~HXA_W_KTILED;
  if (M <= 0 || N <= 0 || K <= 0 || N % 8 || fmt < 0 || fmt > HXA_W_Q4) return 0;
  return skinny_rows(M, N, K, fmt, tile_time(M, N, K, 1, fmt));
}
// The form hxa_linear runs a linear in. *bm: the rows of gemm_skinny_kernel's tile where its modelled time is within 5% of
// the other forms' (their model is the more optimistic one: over 105 (M, N, K, format) of 16 - 1562 rows the choice is
// within 1% of the fastest form, geometric mean; without the skinny kernel 18%), else 0. Result: the K slices, 1 (one launch, fp16 store) or S in {2, 4} (fp32 slices, then their sum)
// when the tile model's time for S slices plus the slices' round trip through memory is below the one-launch time.
int hxa_linear_form(int M, int N, int K, int fmt, int *bm) {
  *bm = 0;
  fmt &= ~HXA_W_KTILED;
  if (M <= 0 || N <= 0 || K <= 0 || N % 8 || fmt < 0 || fmt > HXA_W_Q4) return 1;
  const double t1 = tile_time(M, N, K, 1, fmt);
  int best = 1;
  double tb = t1;
  for (int S = 2; S <= 4; S *= 2) {
    if (K % (32 * S) != 0) continue;
    // slices written by the GEMM and read back by the sum, fp16 out, and the second launch
    const double bytes = 2.0 * S * M * (double)N * 4.0 + 2.0 * M * (double)N;
    const double t = tile_time(M, N, K, S, fmt) + kSumLaunchUs + bytes / kSumBytesPerUs;
    if (t < tb * (S == 4 && best == 2 && fmt != HXA_W_F16 ? 1.02 : kSplitGain)) {
      tb = t;
      best = S;
    }
  }
  *bm = skinny_rows(M, N, K, fmt, 1.05 * tb);
  return *bm ? 1 : best;
}
