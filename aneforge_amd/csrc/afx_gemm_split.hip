// C-ABI entry points, plan and finishing sum of the split GEMM (kernel: afx_gemm_split.h).
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include "afx_gemm_split.h"

namespace afx {

constexpr int kSplitMaxS = 16;

static long long split_row_bytes_of(int fmt, int K) { return fmt == FMT_F16 ? 2LL * K : fmt == FMT_I8 || fmt == FMT_BW ? K : K / 2; }
static long long split_side_bytes_of(int fmt, int K) {
  return fmt == FMT_Q4 || fmt == FMT_BW ? K / 32 * 2 : fmt == FMT_Q4K ? K / 256 * 20 : fmt == FMT_Q6K ? K / 32 * 12 : 0;
}

bool split_supported(int fmt, int N, int K) {
  if (fmt < 0 || fmt > 6 || N < 16 || N % 16 != 0 || K < kSK || K % (fmt == FMT_Q4K || fmt == FMT_Q6K ? 256 : kSK) != 0) return false;
  // a tile's weight rows (up to 256 for the formats with tiles of 256 features) in 31-bit offsets
  return (fmt == FMT_I8 || fmt == FMT_Q4 ? 256 : 128) * split_row_bytes_of(fmt, K) < (1ll << 31);
}

// Whether two workgroups share a CU: at most 128 registers a thread and 80 KB of LDS, as the kernels are
// built.  Counting on two where one fits cost the row tiles of 48 to 96 rows x 128 features of these formats
// a round of workgroups: with the right count Q4_K 22016 x 4096 at 200 rows takes 92 us for 113, blockwise
// 11008 x 2048 at 200 rows 27 for 36, fp16 4096 x 4096 at 128 rows 15 for 19.
static bool split_two_per_cu(int fmt, int mt, int nw) {
  if (nw > 4 || mt > 6) return false;
  switch (fmt) {
    case FMT_I8: return !(mt == 3 && nw == 4);
    case FMT_F16: case FMT_BW: case FMT_Q6K: return nw == 2 || mt <= 2;
    case FMT_Q4K: return mt <= 2 || (nw == 2 && mt == 6);
    default: return true;
  }
}
// Microseconds of one workgroup and K chunk by row tile (16 * mt rows) and features (32 * nw), measured on
// MI355X; `busy` with every CU taken, where the taller tiles, one workgroup per CU, slow down (not for the
// formats whose shorter tiles are alone on a CU too).  Tiles of 64 features take 0.7 of 128, taller ones
// more (their four K groups meet in LDS).
// dec: what decoding a format's 128 features adds (none for int8 codes, two fp32 steps per weight for the
// K-quants; fp16: twice the bytes).
static float split_chunk_us(int fmt, int mt, int nw, bool busy) {
  const int i = mt <= 4 ? mt - 1 : mt <= 6 ? 4 : 5;
  static const float c4[6] = {0.35f, 0.45f, 0.53f, 0.62f, 0.74f, 0.87f};
  static const float c8[6] = {0.0f, 0.0f, 0.0f, 1.01f, 1.13f, 1.35f};
  static const float dec[7] = {0.0f, 0.05f, 0.05f, 0.1f, 0.15f, 0.45f, 0.3f};
  const bool alone = fmt == FMT_BW || fmt == FMT_Q4K || fmt == FMT_Q6K;
  const float slow = busy && ((mt == 8 && !alone) || nw == 8) ? 1.08f : 1.0f;
  return nw == 8 ? (c8[i] + 2.0f * dec[fmt]) * slow : (c4[i] + dec[fmt]) * slow * (nw == 4 ? 1.0f : mt <= 4 ? 0.7f : mt <= 6 ? 0.78f : 0.84f);
}
static int split_rows_kept(int M) { return M < 16 ? M : 16; }
static long long split_ws_bytes(const SplitPlan& p, int M, int S) {
  return (long long)S * p.tiles_m * p.tiles_n * p.mt * p.nw * 128 * split_rows_kept(M);
}
static double weight_mb(int fmt, int N, int K) {
  return (double)N * (split_row_bytes_of(fmt, K) + split_side_bytes_of(fmt, K)) * 1e-6;
}

// The tile and slice count with the least predicted time: rounds of workgroups over the CUs x chunks x the
// chunk time, longer by 6% a round up to three (a chip that stays full), a tile's fill and drain, half of the
// weight stream's 5 TB/s time (the other half overlaps), and a second launch and about 0.5 us per MB of
// partials when K is sliced.  An XCD takes whole (feature tile, slice) pairs with all their row tiles, so
// its 32 CUs may get a round more than the chip's average (int8 5120 x 3072 at 1500 rows: 240 workgroups of
// 256 features, 36 on four of the XCDs, 102 us where 128 features take 63): the rounds are those of the XCD
// with the most.  Where two workgroups share a CU the second costs 0.85 of a round.  Nine of ten of 2940
// measured shapes (7 formats, 17 to 2048 rows, K 1024 to 11008) are within 15% of their prediction.
// 4096 x 4096 at 64, 128 and 300 rows takes 13.9, 16.5 and 24.8 us where the 128 x 128 tiles of afx_gemm
// take 42.5, 43.5 and 43.6.
// fs, fn, fm: only these slices (as many of them as fit), features / 32 and rows / 16; 0: any.
static SplitPlan split_search(int fmt, int M, int N, int K, long long ws_bytes, int fs, int fn, int fm) {
  static const int mts[6] = {1, 2, 3, 4, 6, 8};
  const int nk = K / kSK, t16 = (M + 15) / 16;
  const double stream = 4.5 + weight_mb(fmt, N, K) / 10.0;
  SplitPlan best = {};
  best.us = 1e30f;
  for (int im = 0; im < 6; ++im) {
    const int mt = mts[im];
    if (fm ? mt != fm : im > 0 && mts[im - 1] >= t16) continue;      // no tile taller than needed
    for (int nw = 2; nw <= 8; nw *= 2) {
      if (!split_built(fmt, mt, nw)) continue;
      if (fn && nw != fn) continue;
      SplitPlan p = {mt, nw, (t16 + mt - 1) / mt, (N + 32 * nw - 1) / (32 * nw), 1, 0.0f};
      const double part = (double)p.tiles_m * p.tiles_n * mt * nw * 2048e-6;   // MB of one slice's partials
      const bool two = split_two_per_cu(fmt, mt, nw);
      const double chunk[2] = {split_chunk_us(fmt, mt, nw, false), split_chunk_us(fmt, mt, nw, true)};
      // a tile's epilogue (its K groups meet, then the stores) grows with its registers
      const double tail = 0.0016 * (mt * nw) * (mt * nw), idle = two ? 1.0 : 2.5;
      int smax = nk < kSplitMaxS ? nk : kSplitMaxS;
      while (smax > 1 && split_ws_bytes(p, M, smax) > ws_bytes) --smax;
      if (fs && fs < smax) smax = fs;
      for (int S = fs ? smax : 1; S <= smax; ++S) {
        if (!fs && S > 1 && nk < 2 * S) break;
        const long long wgs = 8LL * ((p.tiles_n * S + 7) / 8) * p.tiles_m;   // as if every XCD had the most of them
        const int n = wgs <= 256 ? 1 : (int)((wgs + 255) / 256);
        const double rounds = n > 1 && two ? 0.7 * n + 0.05 + 0.15 * wgs / 256 : n;
        const double sustained = 1.0 + 0.06 * (n < 4 ? n - 1 : 3);
        const double us = stream + rounds * tail + (rounds - 1.0) * idle + sustained * rounds * ((nk + S - 1) / S) * chunk[wgs > 200] +
                          (S > 1 ? 3.0 + 0.5 * S * part : 0.22 * (mt * nw) * (wgs < 256 ? wgs / 256.0 : 1.0));
        if (us < best.us) {
          best = p;
          best.S = S;
          best.us = (float)us;
        }
      }
    }
  }
  return best;
}
SplitPlan split_plan(int fmt, int M, int N, int K, long long ws_bytes) {
  const char* es = getenv("AFX_GEMM_SPLIT");       // "S", "S.nw" or "S.nw.mt": a fixed choice (tests, tuning), read per call
  int fs = 0, fn = 0, fm = 0;
  if (es && sscanf(es, "%d.%d.%d", &fs, &fn, &fm) >= 1 && fs >= 0 && fn >= 0 && fm >= 0) {
    const SplitPlan p = split_search(fmt, M, N, K, ws_bytes, fs, fn, fm);
    if (p.S > 0) return p;                         // else no kernel of that tile is built for the format
  }
  return split_search(fmt, M, N, K, ws_bytes, 0, 0, 0);
}
// The same product on afx_gemm's tiles, after an expansion to fp16 (6 TB/s; the codebook and K-quant kernels
// 4 and 2) for formats it does not read.  Microseconds per K step of 64 by the 128 x 128 tiles of a CU on the
// XCD with the most; fp16's 256 x 256 tiles, where afx_gemm takes them, 1.9 a round.
static float gemm_tile_us(int fmt, int M, int N, int K) {
  const int tiles_m = (M + 127) / 128, tiles_n = (N + 127) / 128;
  const double x = 8.0 * ((tiles_n + 7) / 8) * tiles_m / 256, n = ceil(x);
  const bool i8 = fmt == FMT_I8;
  double step = n <= 1.0 ? 0.57 + 0.07 * x : n <= 2.0 ? (i8 ? 0.65 : 0.7) + 0.22 * x : (i8 ? 0.52 : 0.55) * n;
  const double rounds7 = ceil(8.0 * (((N + 255) / 256 + 7) / 8) * ((M + 255) / 256) / 256);
  if (!i8 && 10.0 * tiles_m * tiles_n >= 34 * 256 * rounds7) step = 1.9 * rounds7;
  double us = 4.5 + 3.0 * (x < 1.0 ? x : 1.0) + K / 64 * step + weight_mb(fmt, N, K) / 20.0;
  if (!i8 && fmt != FMT_F16) {
    const double tbs = fmt == FMT_Q6K ? 2.0 : fmt == FMT_Q4K || fmt == FMT_L4 ? 4.0 : 6.0;
    us += 2.0 + (2e-6 * N * K + weight_mb(fmt, N, K)) / tbs;
  }
  return (float)us;
}

// y = epilogue(sum of the S slices of ws in slice order), four output features of one row per thread;
// the slices hold the tiles in the kernel's own order.
__global__ __launch_bounds__(256) void gemm_split_finish_kernel(SplitArgs a) {
  const int nt = 2 * a.nw;
  const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long per = (long long)a.tiles_m * a.tiles_n * nt * a.mt * 4 * a.rp;   // f4 per slice
  if (idx >= per) return;
  const int gr = (int)(idx / a.rp), r = (int)(idx - (long long)gr * a.rp);
  const int q0 = gr >> 2, q1 = q0 / a.mt, tile = q1 / nt;
  const int n = (tile / a.tiles_m) * (16 * nt) + 16 * (q1 % nt) + 4 * (gr & 3);
  const int m = ((tile % a.tiles_m) * a.mt + q0 % a.mt) * 16 + r;
  if (n >= a.N || m >= a.M) return;
  const f4* w = (const f4*)a.ws + idx;
  float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int q = 0; q < a.S; q += 4) {               // four slices' loads in flight; slots past S re-read the first
    f4 t[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) t[u] = w[(q + u < a.S ? q + u : 0) * per];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (q + u < a.S) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] += t[u][i];
      }
  }
  split_store4(a, v, n, m);
}

static split_fn pick(int fmt, int mt, int nw) {
  switch (fmt) {
    case FMT_I8: return pick_split<FMT_I8>(mt, nw);
    case FMT_Q4: return pick_split<FMT_Q4>(mt, nw);
    case FMT_F16: return pick_split<FMT_F16>(mt, nw);
    case FMT_BW: return pick_split<FMT_BW>(mt, nw);
    case FMT_L4: return pick_split<FMT_L4>(mt, nw);
    case FMT_Q4K: return pick_split<FMT_Q4K>(mt, nw);
    default: return pick_split<FMT_Q6K>(mt, nw);
  }
}

// Experts: the row tile covers about 1.25 times the mean tokens of an expert, up to 96 rows, two workgroups
// per CU (a longer list takes several tiles: 1024 tokens of top-2 over 8 Q4_0 experts take 657 + 310 us in
// them, 755 + 369 in 128-row tiles); the grid holds the most row tiles T * topk entries can make.
int split_moe_launch(int fmt, SplitArgs& a, hipStream_t stream, const char* what) {
  AFX_REQUIRE(a.w && a.x && a.y && a.cnt && a.list, "%s: null pointer", what);
  AFX_REQUIRE(a.T >= 1 && a.topk >= 1 && a.E >= 1 && split_supported(fmt, a.N, a.K), "%s: bad sizes", what);
  AFX_REQUIRE(a.ldx % 8 == 0 && ((uintptr_t)a.x & 15) == 0 && ((uintptr_t)a.w & 15) == 0,
              "%s: x and weights must be 16-byte aligned", what);
  AFX_REQUIRE(fmt == FMT_F16 || a.scale, "%s: quantized weights need scales", what);
  const long long entries = (long long)a.T * a.topk, xrows = a.x_by_token ? a.T : entries;
  const long long xbytes = xrows * a.ldx * 2;
  AFX_REQUIRE(xbytes < 0x7fff0000LL, "%s: activations span %lld bytes (limit 2 GiB)", what, xbytes);
  a.xbytes = (int)xbytes;
  const double mean = 1.25 * entries / a.E / 16;   // in 16-row tiles
  int mt = mean <= 1 ? 1 : mean <= 2 ? 2 : mean <= 3 ? 3 : mean <= 4 ? 4 : 6;
  int nw = (double)((a.N + 127) / 128) * (a.E < entries ? a.E : entries) >= 256 ? 4 : 2;
  const char* es = getenv("AFX_GEMM_SPLIT");       // as split_plan's (the slice count does not apply)
  int fs = 0, fn = 0, fm = 0;
  if (es && sscanf(es, "%d.%d.%d", &fs, &fn, &fm) >= 2) {
    if (fn == 2 || fn == 4 || fn == 8) nw = fn;
    if (fm >= 1) mt = fm <= 4 ? fm : fm <= 6 ? 6 : 8;
    if (!split_built(fmt, mt, nw)) nw = 4;
  }
  a.S = 1; a.M = 0; a.mt = mt; a.nw = nw;
  a.tiles_n = (a.N + 32 * nw - 1) / (32 * nw);
  const long long tiles = entries / (16 * mt) + (a.E < entries ? a.E : entries);
  AFX_REQUIRE(tiles * a.tiles_n < (1ll << 31), "%s: too many tiles", what);
  const bool glu = a.epi == EPI_SWIGLU || a.epi == EPI_GEGLU;
  a.vec = glu ? a.ldy % 2 == 0 && ((uintptr_t)a.y & 3) == 0 : a.ldy % 4 == 0 && ((uintptr_t)a.y & 15) == 0;
  hipLaunchKernelGGL(pick(fmt, mt, nw), dim3((unsigned)(tiles * a.tiles_n)), dim3(512), 0, stream, a);
  return check_launch(what);
}

int split_launch(int fmt, SplitArgs& a, const SplitPlan& p, hipStream_t stream, const char* what) {
  a.S = p.S;
  a.tiles_m = p.tiles_m; a.tiles_n = p.tiles_n; a.mt = p.mt; a.nw = p.nw;
  a.rp = split_rows_kept(a.M);
  const bool glu = a.epi == EPI_SWIGLU || a.epi == EPI_GEGLU;
  a.vec = a.epi == EPI_F32 ? a.ldy % 4 == 0 && ((uintptr_t)a.y & 15) == 0
        : glu ? a.ldy % 2 == 0 && ((uintptr_t)a.y & 3) == 0
        : a.ldy % 4 == 0 && ((uintptr_t)a.y & 7) == 0 && (a.epi != EPI_RESID || ((uintptr_t)a.resid & 7) == 0);
  const long long xbytes = ((long long)(a.M - 1) * a.ldx + a.K) * 2;
  AFX_REQUIRE(xbytes < (1ll << 31), "%s: activations span %lld bytes (limit 2 GiB)", what, xbytes);
  a.xbytes = (int)xbytes;
  const long long blocks = ((long long)a.tiles_n * a.S + 7) / 8 * 8 * a.tiles_m;
  AFX_REQUIRE(blocks < (1ll << 31), "%s: %lld tiles", what, blocks);
  hipLaunchKernelGGL(pick(fmt, p.mt, p.nw), dim3((unsigned)blocks), dim3(512), 0, stream, a);
  const int rc = check_launch(what);
  if (rc || a.S == 1) return rc;
  const long long n = split_ws_bytes(p, a.M, 1) / 16;
  hipLaunchKernelGGL(gemm_split_finish_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, a);
  return check_launch(what);
}

}  // namespace afx

using namespace afx;

extern "C" {

int afx_gemm_split_plan(int fmt, int M, int N, int K, long long* ws_bytes) {
  if (ws_bytes) *ws_bytes = 0;
  AFX_REQUIRE(M >= 1 && split_supported(fmt, N, K), "afx_gemm_split_plan: fmt=%d M=%d N=%d K=%d is not afx_gemm_split's", fmt, M, N, K);
  const SplitPlan p = split_plan(fmt, M, N, K);
  if (ws_bytes) *ws_bytes = p.S > 1 ? split_ws_bytes(p, M, p.S) : 0;
  // Up to three of afx_gemm's row tiles the two predictions are taken as they are: int8 22016 x 4096 at 128
  // rows 52 -> 43 us, 11008 x 2048 at 300 34 -> 26.  Past that the two are closer and 5% have to be in it: of
  // 2940 measured shapes 6 come out more than 3% slower than on the other kernel (9% at most), 96 stay there
  // that would gain more than 5%.
  const float margin = M <= 384 ? 1.0f : 0.95f;
  // rows of up to 2 K elements apart stay inside the kernel's 2 GiB activation range
  return (long long)M * K < (1ll << 29) && p.us < margin * gemm_tile_us(fmt, M, N, K) ? 1 : 0;
}

int afx_gemm_split(int fmt, const void* w, const void* scale, const void* x, int ldx, void* y, int ldy, int M, int N,
                   int K, const void* bias, const void* residual, int epi, void* ws, long long ws_bytes,
                   void* stream) {
  AFX_REQUIRE(w && x && y, "afx_gemm_split: null pointer");
  AFX_REQUIRE(M >= 1 && split_supported(fmt, N, K),
              "afx_gemm_split: need M >= 1, N %% 16 == 0, K %% 128 == 0 (256 for K-quants), a tile's rows inside 2 GiB (fmt=%d M=%d N=%d K=%d)", fmt, M, N, K);
  AFX_REQUIRE(ldx >= K && ldx % 8 == 0 && ((uintptr_t)x & 15) == 0 && ((uintptr_t)w & 15) == 0,
              "afx_gemm_split: x and weights must be 16-byte aligned rows (ldx %% 8 == 0)");
  AFX_REQUIRE((epi >= 0 && epi <= 3) || epi == EPI_GEGLU, "afx_gemm_split: unknown epilogue %d", epi);
  AFX_REQUIRE(fmt == FMT_F16 || scale, "afx_gemm_split: quantized weights need scales");
  const int align = fmt == FMT_L4 ? 15 : fmt == FMT_I8 || fmt == FMT_F16 ? 1 : 3;
  AFX_REQUIRE(((uintptr_t)scale & align) == 0, "afx_gemm_split: scales must be %d-byte aligned", align + 1);
  AFX_REQUIRE(epi != EPI_RESID || residual, "afx_gemm_split: residual pointer required");
  const bool glu = epi == EPI_SWIGLU || epi == EPI_GEGLU;
  AFX_REQUIRE(glu ? ldy >= N / 2 : ldy >= N, "afx_gemm_split: ldy=%d too small", ldy);
  AFX_REQUIRE(!ws || ((uintptr_t)ws & 15) == 0, "afx_gemm_split: the workspace must be 16-byte aligned");
  SplitArgs a = {};
  a.w = w; a.scale = (const half_t*)scale; a.bias = (const half_t*)bias; a.x = (const half_t*)x; a.y = y;
  a.resid = (const half_t*)residual; a.ldx = ldx; a.ldy = ldy; a.M = M; a.N = N; a.K = K; a.epi = epi;
  a.ws = (float*)ws;
  return split_launch(fmt, a, split_plan(fmt, M, N, K, ws ? ws_bytes : 0), (hipStream_t)stream, "afx_gemm_split");
}

}  // extern "C"
