// Tiled MFMA GEMM over packed weights for a few to a few hundred activation rows: the linears of
// short prompts and verification rows, and the grouped MoE experts of a prompt.
//
//   Y[m, n] = epilogue( sum_k X[m, k] * W^[n, k] ),   X fp16 rows (stride ldx), W in any packed format.
//
// A 128 x 128 tile per workgroup leaves most of the chip idle here (N = 4096: 32 workgroups on 256
// CUs) and each K step waits out the memory latency.  So:
//  * Eight wavefronts share a tile of 16 MT rows x BN features: NW side by side in N (32 features
//    each), times KG = 8 / NW groups that take different MFMA steps of every staged K chunk and
//    meet in LDS at the end, so a tile of 64 features still fills a CU.
//  * K is cut further into S slices, one workgroup per (tile, slice); the slices' fp32 partials
//    meet in a caller workspace and a second launch sums them in slice order and applies the
//    epilogue (S = 1: the epilogue runs here).  Partials cost about 0.5 us per MB and the launch 3,
//    so S and the tile are the ones of least predicted time.
//  * Global loads are row-contiguous (the MFMA layout would have 16 lanes touch 16 rows: the same
//    bytes at a quarter of the rate) and run PD chunks ahead in registers; two LDS stages, one
//    barrier per 128-wide chunk.  Weights are staged in their packed format and decoded when a
//    wavefront reads its fragment, each by one wavefront only, with no separate dequantisation pass.
//  * LDS rows have their 16-byte chunks XOR-permuted by the row, so the fragment reads of 8 rows at
//    one k hit distinct banks.
// The weights are the A operand (row l % 16 = output feature, k slot l / 16) and X the B operand
// (column l % 16 = activation row): a lane's four results are four consecutive output features of
// one row, so stores are 8 or 16 bytes and a gate/up pair meets in one lane.  A k-permutation shared
// by A and B is free, so each lane decodes the k values of its own weight words.
#pragma once
#include "afx_gemv_impl.h"

namespace afx {

struct SplitArgs {
  const void* w;           // weights [E][N][row bytes]
  const half_t* scale;     // the format's scales / side words [E][N][..]
  long long w_es, s_es;    // per-expert strides (bytes of w, halves of scale)
  const half_t* x;         // activations, row r at x + r * ldx
  void* y;                 // output rows, stride ldy
  const half_t* bias;      // [N] or null
  const half_t* resid;     // EPI_RESID: [M][ldy] (may alias y)
  float* ws;               // S > 1: partials [S][M][N]
  const int* cnt;          // MoE: tokens per expert [E], else null
  const int* list;         // MoE: entries (token * topk + slot) per expert [E][T]
  int T, E, topk, x_by_token;   // MoE: tokens, experts, top-k, X row of an entry = entry / topk or the entry
  int ldx, ldy, M, N, K, epi;
  int S, tiles_n, tiles_m, mt, nw; // slices and tiles (MoE: one slice; row tiles are found from cnt)
  int rp;                  // rows of a 16-row tile kept in the workspace (M below 16 rows, else 16)
  int xbytes;              // bytes of X the loads may read (< 2^31)
  int vec;                 // y (and resid, bias) rows take 4-element accesses
};

constexpr int kSK = 128;                           // k per chunk

// Buffer loads: the lane's byte offset in a vector register, the chunk's in a scalar one; a resource
// of zero bytes makes a load past the last chunk return zeros without a memory access, so the loop
// has no branch around its loads (with one the compiler waits for every load in flight at the merge).
__device__ __forceinline__ u4 split_load16(__amdgpu_buffer_rsrc_t r, int vo, int so) {
  return __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(r, vo, so, 0));
}
__device__ __forceinline__ u2 split_load8(__amdgpu_buffer_rsrc_t r, int vo, int so) {
  return __builtin_bit_cast(u2, __builtin_amdgcn_raw_buffer_load_b64(r, vo, so, 0));
}
__device__ __forceinline__ uint32_t split_load4(__amdgpu_buffer_rsrc_t r, int vo, int so) {
  return __builtin_amdgcn_raw_buffer_load_b32(r, vo, so, 0);
}

// Per format: staged bytes of a weight row per chunk (kRB), of its side words (kSB), the A operand of
// MFMA step i = 0..3 of a chunk from the staged row, and the 16-byte X chunk (of 16) that lane group
// g pairs with it.  wchunk: LDS offset of a row's 16-byte chunk c.
template <int RB> __device__ __forceinline__ int wchunk(int row, int c) {
  return row * RB + ((RB == 256 ? c ^ (row & 15) : RB == 128 ? c ^ (row & 7) : c ^ ((row >> 1) & 3)) << 4);
}
template <int FMT> struct SW;

template <> struct SW<FMT_I8> {
  static constexpr int kRB = 128, kSB = 0;
  struct Ctx {};
  __device__ static Ctx make(const half_t*, int) { return {}; }
  __device__ static int xc(int g, int i) { return 8 * (i >> 1) + 2 * g + (i & 1); }
  __device__ static h8 codes(const unsigned char* w, int row, int g, int i) {
    const u2 v = *(const u2*)(w + wchunk<kRB>(row, 4 * (i >> 1) + g) + 8 * (i & 1));
    h2 a, b, c, d;
    i8x4_to_h2(v.x, a, b);
    i8x4_to_h2(v.y, c, d);
    return (h8){a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y};
  }
  __device__ static h8 frag(const unsigned char* w, const unsigned char*, const Ctx&, int row, int g, int i) {
    return codes(w, row, g, i);
  }
};
// blockwise: fp16(q * s); the block of k 64 (i / 2) + 16 g .. + 15 is 2 (i / 2) + g / 2 of the chunk's four
template <> struct SW<FMT_BW> : SW<FMT_I8> {
  static constexpr int kSB = 8;
  __device__ static h8 frag(const unsigned char* w, const unsigned char* sd, const Ctx&, int row, int g, int i) {
    const half_t s = *(const half_t*)(sd + row * kSB + 4 * (i >> 1) + 2 * (g >> 1));
    const h8 s8 = {s, s, s, s, s, s, s, s};
    return codes(w, row, g, i) * s8;
  }
};
template <> struct SW<FMT_F16> {
  static constexpr int kRB = 256, kSB = 0;
  struct Ctx {};
  __device__ static Ctx make(const half_t*, int) { return {}; }
  __device__ static int xc(int g, int i) { return 4 * i + g; }
  __device__ static h8 frag(const unsigned char* w, const unsigned char*, const Ctx&, int row, int g, int i) {
    return *(const h8*)(w + wchunk<kRB>(row, 4 * i + g));
  }
};
struct SW4 {                                       // 4-bit formats
  static constexpr int kRB = 64, kSB = 0;
  struct Ctx {};
  __device__ static Ctx make(const half_t*, int) { return {}; }
  __device__ static uint32_t word(const unsigned char* w, int row, int g, int i) {
    return *(const uint32_t*)(w + wchunk<kRB>(row, g) + 4 * i);
  }
};
// Q4_0: word i of 16-byte chunk g = elements 8 g .. + 7 of block i, fp16((nibble - 8) * d)
template <> struct SW<FMT_Q4> : SW4 {
  static constexpr int kSB = 8;
  __device__ static int xc(int g, int i) { return 4 * i + g; }
  __device__ static h8 frag(const unsigned char* w, const unsigned char* sd, const Ctx&, int row, int g, int i) {
    const half_t s = *(const half_t*)(sd + row * kSB + 2 * i);
    const h2 s2 = {s, s};
    h2 q[4];
    q4_word_to_h2(word(w, row, g, i), q);
#pragma unroll
    for (int k = 0; k < 4; ++k) q[k] = q[k] * s2;
    return (h8){q[0].x, q[0].y, q[1].x, q[1].y, q[2].x, q[2].y, q[3].x, q[3].y};
  }
};
// int4 codebook: word i of chunk g = columns 32 g + 8 i .. + 7; the lookup yields them as
// (0, 2, 4, 6, 1, 3, 5, 7), the order the X staging of this format writes
template <> struct SW<FMT_L4> : SW4 {
  typedef L4Ctx Ctx;
  __device__ static Ctx make(const half_t* s, int row) { return L4Ctx::make(s, row); }
  __device__ static int xc(int g, int i) { return 4 * g + i; }
  __device__ static h8 frag(const unsigned char* wl, const unsigned char*, const Ctx& t, int row, int g, int i) {
    const uint32_t w = word(wl, row, g, i);
    uint32_t la, ha, lb, hb;
    l4_lookup(t, w & 0x07070707u, l4_bit7_mask(w << 4), la, ha);
    l4_lookup(t, (w >> 4) & 0x07070707u, l4_bit7_mask(w), lb, hb);
    const u4 o = {__builtin_amdgcn_perm(ha, la, 0x05010400u), __builtin_amdgcn_perm(ha, la, 0x07030602u),
                  __builtin_amdgcn_perm(hb, lb, 0x05010400u), __builtin_amdgcn_perm(hb, lb, 0x07030602u)};
    return __builtin_bit_cast(h8, o);
  }
};
__device__ __forceinline__ u4 l4_x_order(u4 v) {   // (x0,x1) .. (x6,x7) -> (x0,x2) (x4,x6) (x1,x3) (x5,x7)
  return (u4){__builtin_amdgcn_perm(v.y, v.x, 0x05040100u), __builtin_amdgcn_perm(v.w, v.z, 0x05040100u),
              __builtin_amdgcn_perm(v.y, v.x, 0x07060302u), __builtin_amdgcn_perm(v.w, v.z, 0x07060302u)};
}
__device__ __forceinline__ h8 fma8(uint32_t a, uint32_t b, float ds, float off) {   // fp16(ds * byte + off)
  asm("" : "+v"(a), "+v"(b));                      // one v_cvt_f32_ubyte<n> per byte
  h8 o;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    o[k] = (half_t)__builtin_fmaf(ds, ubyte_f32(a, k), off);
    o[4 + k] = (half_t)__builtin_fmaf(ds, ubyte_f32(b, k), off);
  }
  return o;
}
// Q4_K: a chunk is half a super-block; 16-byte chunk g is half h = g % 2 of pair g / 2: low nibbles
// (i = 0, 1) are k 64 (g / 2) + 16 h + 8 i .., high nibbles (i = 2, 3) those + 32.  Staged side words:
// {d, dmin}, then the two pairs' scale and min bytes.
template <> struct SW<FMT_Q4K> : SW4 {
  static constexpr int kSB = 16;
  __device__ static int xc(int g, int i) { return 8 * (g >> 1) + 2 * (g & 1) + 4 * (i >> 1) + (i & 1); }
  __device__ static h8 frag(const unsigned char* w, const unsigned char* sd, const Ctx&, int row, int g, int i) {
    const h2 dd = *(const h2*)(sd + row * kSB);
    const uint32_t sm = *(const uint32_t*)(sd + row * kSB + 4 + 4 * (g >> 1));
    const u2 v = *(const u2*)(w + wchunk<kRB>(row, g) + 8 * (i & 1));
    const int b = i >> 1;
    const float ds = (float)dd.x * (float)((sm >> (8 * b)) & 0xFFu), dm = (float)dd.y * (float)((sm >> (16 + 8 * b)) & 0xFFu);
    return fma8((v.x >> (4 * b)) & 0x0F0F0F0Fu, (v.y >> (4 * b)) & 0x0F0F0F0Fu, ds, -dm);
  }
};
// Q6_K: 16-byte chunk g is the 32-weight block g, word i its elements 8 i .. + 7
template <> struct SW<FMT_Q6K> : SW4 {
  static constexpr int kSB = 48;
  __device__ static int xc(int g, int i) { return 4 * g + i; }
  __device__ static h8 frag(const unsigned char* wl, const unsigned char* sd, const Ctx&, int row, int g, int i) {
    const uint32_t* q = (const uint32_t*)(sd + row * kSB + 12 * g);
    const uint32_t H = q[i >> 1], sc = q[2], w = word(wl, row, g, i);
    const float ds = (float)as_h2(sc).y * (float)(int8_t)((sc >> (8 * (i >> 1))) & 0xFFu);
    const uint32_t lo = (w & 0x0F0F0F0Fu) | (((i & 1) ? H : H << 4) & 0x30303030u);
    const uint32_t hi = ((w >> 4) & 0x0F0F0F0Fu) | (((i & 1) ? H >> 2 : H << 2) & 0x30303030u);
    return fma8(lo, hi, ds, -32.0f * ds);
  }
};

template <int FMT> __host__ __device__ constexpr long long split_row_bytes(int K) {
  return FMT == FMT_F16 ? 2LL * K : FMT == FMT_I8 || FMT == FMT_BW ? K : K / 2;
}

// Output features n .. n + 3 (n % 4 == 0, all inside N) of y row yr: bias, epilogue, store.
__device__ __forceinline__ void split_store4(const SplitArgs& a, float (&v)[4], int n, int yr) {
  if (a.bias) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] += (float)a.bias[n + i];
  }
  const size_t o = (size_t)yr * a.ldy;
  if (a.epi == EPI_SWIGLU || a.epi == EPI_GEGLU) {
    const bool gelu = a.epi == EPI_GEGLU;
    half_t* yp = (half_t*)a.y + o + (n >> 1);
    h2 r;
    r.x = (half_t)(glu_act(gelu, (float)(half_t)v[0]) * (float)(half_t)v[1]);
    r.y = (half_t)(glu_act(gelu, (float)(half_t)v[2]) * (float)(half_t)v[3]);
    if (a.vec) *(uint32_t*)yp = as_u32(r);
    else { yp[0] = r.x; yp[1] = r.y; }
  } else if (a.epi == EPI_F32) {
    float* yp = (float*)a.y + o + n;
    if (a.vec) *(f4*)yp = (f4){v[0], v[1], v[2], v[3]};
    else {
#pragma unroll
      for (int i = 0; i < 4; ++i) yp[i] = v[i];
    }
  } else {
    half_t* yp = (half_t*)a.y + o + n;
    const half_t* rp = a.resid + o + n;
    h4 r;
    if (a.epi == EPI_RESID) {
      h4 b;
      if (a.vec) b = *(const h4*)rp;
      else b = (h4){rp[0], rp[1], rp[2], rp[3]};
#pragma unroll
      for (int i = 0; i < 4; ++i) r[i] = (half_t)((float)b[i] + (float)(half_t)v[i]);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) r[i] = (half_t)v[i];
    }
    if (a.vec) *(h4*)yp = r;
    else {
#pragma unroll
      for (int i = 0; i < 4; ++i) yp[i] = r[i];
    }
  }
}

template <int B> struct Buf { static constexpr int value = B; };

template <int FMT> __host__ __device__ constexpr long long split_side_bytes(int K) {   // per row of weights
  return FMT == FMT_Q4 || FMT == FMT_BW ? K / 32 * 2 : FMT == FMT_Q4K ? K / 256 * 20 : FMT == FMT_Q6K ? K / 32 * 12 : 0;
}

template <int FMT, int MT, int NW, int NT> struct SplitGeo {
  typedef SW<FMT> F;
  static constexpr int KG = 8 / NW, BN = 16 * NT * NW;
  static constexpr int kX = MT * 4096, kW = BN * F::kRB, kS = BN * F::kSB, kStage = kX + kW + kS;
  static constexpr int kRed = KG / 2 * NW * MT * NT * 1024;          // the K groups' meeting place, after the loop
  static constexpr int kLds = 2 * kStage > kRed ? 2 * kStage : kRed;
  static constexpr int NX = (MT + 1) / 2;                            // 16-byte chunks per thread and K chunk: X,
  static constexpr int NL = kW / 16 < 512 ? 1 : kW / 16 / 512;       // weights
  static constexpr int PD = MT <= 4 && NT == 2 ? 4 : 2;              // K chunks in flight in registers
};

template <int FMT, int MT, int NW, int NT>
__global__ __launch_bounds__(512, 2) void gemm_split_kernel(SplitArgs a) {
  typedef SW<FMT> F;
  typedef SplitGeo<FMT, MT, NW, NT> G;
  constexpr int KG = G::KG, BN = G::BN, NX = G::NX, NL = G::NL, PD = G::PD, RB = F::kRB;
  __shared__ __align__(16) unsigned char lds[G::kLds];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave % NW, kg = wave / NW;
  const int r = lane & 15, g = lane >> 4;
  int id = blockIdx.x, rows = a.M, m0, n0, e = 0, slice = 0;
  const int* lst = nullptr;
  if (a.cnt) {
    // row tile id / tiles_n of the experts' tiles in expert order, found from the token counts
    int left = id / a.tiles_n;
    n0 = (id - left * a.tiles_n) * BN;
    for (e = -1, m0 = 0; e < 0; m0 += 64) {        // 64 experts a pass; m0: the pass's first expert
      if (m0 >= a.E) return;                       // past the last tile (whole workgroup: no barrier reached)
      const int c = m0 + lane < a.E ? a.cnt[m0 + lane] : 0;
      int t = (c + MT * 16 - 1) / (MT * 16);       // tiles of this lane's expert, then their running sum
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int u = __shfl_up(t, d, 64);
        if (lane >= d) t += u;
      }
      const unsigned long long past = __ballot(t > left);
      if (past) {
        const int l = __ffsll(past) - 1;
        const int before = l > 0 ? __builtin_amdgcn_readlane(t, l - 1) : 0;
        rows = __builtin_amdgcn_readlane(c, l);
        e = m0 + l;
        left -= before;
      } else {
        left -= __builtin_amdgcn_readlane(t, 63);
      }
    }
    m0 = left * (MT * 16);
    lst = a.list + (size_t)e * a.T;
  } else {
    // an XCD (dispatch is round-robin over 8) takes every row tile of its (feature tile, slice) pairs, one
    // after the other: the weights leave memory once, and with 8 slices an XCD reads one K slice of X
    const int local = id >> 3, pair = (local / a.tiles_m) * 8 + (id & 7);
    const int nt = pair / a.S, mt = local % a.tiles_m;
    if (nt >= a.tiles_n) return;
    slice = pair - nt * a.S;
    m0 = mt * (MT * 16);
    n0 = nt * BN;
    id = nt * a.tiles_m + mt;
  }
  const int tile = id;
  const int N = a.N, K = a.K, nk = K / kSK;        // chunks of the row; the slice's are [t0, t1)
  const int t0 = (int)((long long)nk * slice / a.S), t1 = (int)((long long)nk * (slice + 1) / a.S);

  // X staging: thread t carries 16-byte chunk t % 16 of rows t / 16 + 32 i (with MT odd, the last i of half the threads)
  const int xrow = tid >> 4, xp = tid & 15;
  int xo[NX], xl[NX];                              // byte offsets; rows past the end repeat the last one (not stored)
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    int m = m0 + xrow + 32 * i;
    m = m < rows ? m : rows - 1;
    if (lst) {
      m = lst[m];
      if (a.x_by_token) m /= a.topk;
    }
    xo[i] = m * (a.ldx * 2) + xp * 16;
    xl[i] = wchunk<256>(xrow + 32 * i, xp);
  }
  const bool xlast = MT % 2 == 0 || wave < 4;      // wavefront-uniform
  // weight staging: 16-byte chunk c % CPR of row c / CPR for c = t + 512 i
  constexpr int CPR = RB / 16;
  const int nrows = N - n0 < BN ? N - n0 : BN;
  const unsigned char* wb = (const unsigned char*)a.w + (size_t)e * a.w_es + (size_t)n0 * split_row_bytes<FMT>(K);
  const int wbytes = nrows * (int)split_row_bytes<FMT>(K);
  const half_t* sb = a.scale ? a.scale + (size_t)e * a.s_es : nullptr;
  const unsigned char* sdb = (const unsigned char*)sb + (size_t)n0 * split_side_bytes<FMT>(K);
  const int sbytes = nrows * (int)split_side_bytes<FMT>(K);
  int wo[NL], wl[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int c = tid + 512 * i, row = c / CPR;
    wo[i] = row * (int)split_row_bytes<FMT>(K) + (c % CPR) * 16;     // a row past N is out of the buffer's range: zeros
    wl[i] = wchunk<RB>(row, c % CPR);
  }
  const bool wok = BN * CPR >= 512 || wave < BN * CPR / 64;
  // side words: thread t carries piece t % kSP of row t / kSP
  constexpr int kSP = FMT == FMT_Q6K ? 3 : 1;
  static_assert(F::kSB == 0 || BN * kSP <= 512, "one side piece per thread");
  const int srow = tid / kSP, spc = tid % kSP;
  const bool sok = F::kSB > 0 && tid < BN * kSP;
  const int so = srow * (int)split_side_bytes<FMT>(K) + spc * 16;

  u4 xq[PD][NX], wq[PD][NL], sq[PD];
  auto load = [&](auto b, int t) {
    constexpr int B = decltype(b)::value;
    const bool ok = t < t1;
    const __amdgpu_buffer_rsrc_t ws = make_rsrc(wb, ok ? wbytes : 0), xs = make_rsrc(a.x, ok ? a.xbytes : 0);
#pragma unroll
    for (int i = 0; i < NL; ++i) wq[B][i] = split_load16(ws, wo[i], t * RB);
    if constexpr (F::kSB > 0) {
      const __amdgpu_buffer_rsrc_t ss = make_rsrc(sdb, ok ? sbytes : 0);
      if constexpr (FMT == FMT_Q6K) sq[B] = split_load16(ss, so, t * 48);
      else if constexpr (FMT == FMT_Q4K) {
        const u2 p = split_load8(ss, so + 4, (t >> 1) * 20 + 8 * (t & 1));
        sq[B] = (u4){split_load4(ss, so, (t >> 1) * 20), p.x, p.y, 0u};
      } else {
        const u2 p = split_load8(ss, so, t * 8);
        sq[B] = (u4){p.x, p.y, 0u, 0u};
      }
    }
#pragma unroll
    for (int i = 0; i < NX; ++i) xq[B][i] = split_load16(xs, xo[i], t * 256);
  };
  auto stage = [&](auto b, int s) {
    constexpr int B = decltype(b)::value;
    unsigned char* base = lds + s * G::kStage;
#pragma unroll
    for (int i = 0; i < NX; ++i)
      if (i + 1 < NX || xlast) *(u4*)(base + xl[i]) = FMT == FMT_L4 ? l4_x_order(xq[B][i]) : xq[B][i];
    if (wok) {
#pragma unroll
      for (int i = 0; i < NL; ++i) *(u4*)(base + G::kX + wl[i]) = wq[B][i];
    }
    if constexpr (F::kSB > 0) {
      if (sok) {
        unsigned char* sp = base + G::kX + G::kW + srow * F::kSB + spc * 16;
        if constexpr (F::kSB == 8) *(u2*)sp = (u2){sq[B].x, sq[B].y};
        else *(u4*)sp = sq[B];
      }
    }
  };
  const int wrow = wn * (16 * NT) + r;
  typename F::Ctx ctx[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int n = n0 + wrow + 16 * j;
    ctx[j] = F::make(sb, n < N ? n : N - 1);
  }
  f4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = (f4){0.0f, 0.0f, 0.0f, 0.0f};

  auto compute = [&](int s) {
    const unsigned char* base = lds + s * G::kStage;
#pragma unroll
    for (int q = 0; q < 4 / KG; ++q) {
      const int i = kg * (4 / KG) + q;             // this group's MFMA steps of the chunk
      h8 wf[NT], xf[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) xf[m] = *(const h8*)(base + m * 4096 + wchunk<256>(r, F::xc(g, i)));
#pragma unroll
      for (int j = 0; j < NT; ++j) wf[j] = F::frag(base + G::kX, base + G::kX + G::kW, ctx[j], wrow + 16 * j, g, i);
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          acc[m][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf[j], xf[m], acc[m][j], 0, 0, 0);
    }
  };
  // chunk t is in LDS stage t & 1 (counted from t0), chunks t + 1 .. t + PD - 1 in registers, t + PD issued
  auto step = [&](auto b, int t, int s) {
    constexpr int B = decltype(b)::value;
    load(b, t + PD);
    if (FMT != FMT_L4 || t < t1) compute(s);       // a zero chunk's codes would still name codebook entry 0, which may be infinite
    stage(Buf<(B + 1) % PD>{}, s ^ 1);             // last read before the previous barrier
    __syncthreads();
  };
  load(Buf<0>{}, t0);
  load(Buf<1>{}, t0 + 1);
  if constexpr (PD == 4) {
    load(Buf<2>{}, t0 + 2);
    load(Buf<3>{}, t0 + 3);
  }
  stage(Buf<0>{}, 0);
  __syncthreads();
  for (int t = t0; t < t1; t += PD) {              // chunks past t1 are zeros
    step(Buf<0>{}, t, 0);
    step(Buf<1>{}, t + 1, 1);
    if constexpr (PD == 4) {
      if (t + 2 >= t1) break;                      // uniform
      step(Buf<2>{}, t + 2, 0);
      step(Buf<3>{}, t + 3, 1);
    }
  }

  // the K groups' tiles, halved until group 0 holds the sum
  f4* red = (f4*)lds;
  constexpr int NP = MT * NT;
#pragma unroll
  for (int h = KG / 2; h >= 1; h >>= 1) {
    if (kg >= h && kg < 2 * h) {
#pragma unroll
      for (int p = 0; p < NP; ++p) red[(((kg - h) * NW + wn) * NP + p) * 64 + lane] = acc[p / NT][p % NT];
    }
    __syncthreads();
    if (kg < h) {
#pragma unroll
      for (int p = 0; p < NP; ++p) acc[p / NT][p % NT] += red[((kg * NW + wn) * NP + p) * 64 + lane];
    }
    if (h > 1) __syncthreads();
  }
  if (kg > 0) return;
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int n = n0 + wn * (16 * NT) + 16 * j + 4 * g;
    if (n >= N) continue;
    float sc[4] = {1.0f, 1.0f, 1.0f, 1.0f};
    if constexpr (FMT == FMT_I8) {
#pragma unroll
      for (int i = 0; i < 4; ++i) sc[i] = (float)sb[n + i];
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int mr = m0 + 16 * m + r;
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = acc[m][j][i] * sc[i];
      if (a.S > 1) {
        if (r < a.rp)
          ((f4*)a.ws)[(((((size_t)slice * a.tiles_m * a.tiles_n + tile) * (NW * NT) + wn * NT + j) * MT + m) * 4 + g) * a.rp + r] =
              (f4){v[0], v[1], v[2], v[3]};
      } else if (mr < rows) split_store4(a, v, n, lst ? lst[mr] : mr);
    }
  }
}

typedef void (*split_fn)(SplitArgs);
// The kernels built, by row tiles mt and feature tiles of 32 * nw: nw = 8 is four wavefronts of 64 features.
template <int FMT, int NW> split_fn pick_split_mt(int mt) {
  return mt <= 1 ? gemm_split_kernel<FMT, 1, NW, 2> : mt <= 2 ? gemm_split_kernel<FMT, 2, NW, 2> : mt <= 3 ? gemm_split_kernel<FMT, 3, NW, 2>
       : mt <= 4 ? gemm_split_kernel<FMT, 4, NW, 2> : mt <= 6 ? gemm_split_kernel<FMT, 6, NW, 2> : gemm_split_kernel<FMT, 8, NW, 2>;
}
inline bool split_built(int fmt, int mt, int nw) {
  // 256 features: int8 and Q4_0, where the X traffic saved shows and the registers hold (Q4_0 up to mt = 6)
  return nw < 8 || (mt >= 4 && (fmt == FMT_I8 || (fmt == FMT_Q4 && mt <= 6)));
}
template <int FMT> split_fn pick_split(int mt, int nw) {
  if constexpr (FMT == FMT_I8 || FMT == FMT_Q4) {
    if (nw == 8 && mt <= 4) return gemm_split_kernel<FMT, 4, 4, 4>;
    if (nw == 8 && (mt <= 6 || FMT == FMT_Q4)) return gemm_split_kernel<FMT, 6, 4, 4>;
    if (nw == 8) return gemm_split_kernel<FMT_I8, 8, 4, 4>;
  }
  return nw == 2 ? pick_split_mt<FMT, 2>(mt) : pick_split_mt<FMT, 4>(mt);
}
extern template split_fn pick_split<FMT_I8>(int, int);
extern template split_fn pick_split<FMT_Q4>(int, int);
extern template split_fn pick_split<FMT_F16>(int, int);
extern template split_fn pick_split<FMT_BW>(int, int);
extern template split_fn pick_split<FMT_L4>(int, int);
extern template split_fn pick_split<FMT_Q4K>(int, int);
extern template split_fn pick_split<FMT_Q6K>(int, int);

// Row tiles (16 * mt rows each), features per tile (32 * nw) and K slices of a dense [M][K] x [N][K] product,
// as many slices as a workspace of ws_bytes holds.
struct SplitPlan {
  int mt, nw, tiles_m, tiles_n, S;
  float us;                // its predicted time
};
bool split_supported(int fmt, int N, int K);
// afx_gemm_split's launches by plan p (made for a.ws), `a` filled in but for the plan's fields; w, x and ws
// 16-byte aligned.
int split_launch(int fmt, SplitArgs& a, const SplitPlan& p, hipStream_t stream, const char* what);
SplitPlan split_plan(int fmt, int M, int N, int K, long long ws_bytes = 1ll << 62);
// The grouped experts (a.cnt set): a's pointers, strides, T, E, topk, N, K and epi filled in by the caller.
int split_moe_launch(int fmt, SplitArgs& a, hipStream_t stream, const char* what);

}  // namespace afx
