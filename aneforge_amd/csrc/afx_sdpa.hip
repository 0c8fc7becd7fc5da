// Attention of many queries over head-major q [H][Sq][D], k/v [Hkv][Skv][D] (af.sdpa at prompt or encoder
// shapes, aneforge/graph.py:993-1040), plain or causal, fp32 scores and softmax.
//
// The decode kernel takes one query a row and streams the keys through VALU dot products: 512 queries of
// 32 heads (8 kv, head dim 128) read every key 512 times (130 us).  Here both products run on
// MFMA with keys staged once per 64 queries (18 us, causal or not):
//  * S^T = K Q^T (keys are the A rows): a query's scores sit in four lanes, so row maxima and sums are
//    lane-local but for two exchanges, and the probabilities are already the B operand of O^T = V^T P^T.
//  * The probabilities keep their fp32 bits: p = the sum of three fp16 values, each multiplied with V, so
//    a product has the decode kernel's fp32 weight; with two (22 bits) differences of near weights came out
//    ten times further from 64 bits, for 16.2 us instead of 17.7.  The three hold p * 2^14, exactly down to
//    p = 2^-14 and to 2^-39 below; the power of two leaves with the sum's reciprocal.
//  * Eight wavefronts: 64 queries x two halves of the keys, each half with its own double-buffered
//    stages, merged through LDS, so the longest serial chain is half the key blocks (causal tiles are
//    dispatched longest first).
// V is staged row-major and read through ds_read_b64_tr_b16; a query may see no key of its half (its
// maximum stays -inf, its weights 0).  A V row with an infinity or NaN would turn a hidden key's zero
// weight into NaN, and the infinity of a visible one too (its weight's low part may be zero or negative),
// so a block that holds one adds its visible keys one by one, each with its fp32 weight.  Looking for them
// takes three VALU operations per two values as they are staged.
#include "afx_common.h"

namespace afx {

constexpr int kSQ = 64, kSB = 64;        // queries per workgroup, keys per block
constexpr float kPScale = 16384.0f;      // the probabilities' scale: the largest is 1, and 2^14 an fp16 number

struct SdpaArgs {
  const half_t *q, *k, *v;
  half_t* o;
  int H, Hkv, Sq, Skv, tiles, causal;
  float scale_log2;
};

typedef short v4s __attribute__((ext_vector_type(4)));
typedef short v8s __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) v4s lds_v4s;

template <int D> __device__ __forceinline__ int v_at(int row, int ch) {   // byte of 16-byte chunk ch of a staged V row
  return row * (2 * D) + ((ch ^ ((row & (D / 16 - 1)) << 1)) << 4);
}

template <int D>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void sdpa_kernel(SdpaArgs a) {
  constexpr int KR = 2 * D + 16, VR = 2 * D, KS = D / 32, ND = D / 16;
  constexpr int kKB = kSB * KR, kVB = kSB * VR, kX = 4 * ND + 2;
  __shared__ __align__(16) unsigned char lds[4 * kKB + 4 * kVB];
  __shared__ int odd[2][4];              // [half][block % 4]: the staged V holds an infinity or NaN
  static_assert(4 * 64 * kX * 4 <= 4 * kKB, "the handover fits in the K stages");
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hf = wave >> 2, w4 = wave & 3, htid = tid & 255;
  const int fr = lane & 15, fg = lane >> 4;
  unsigned char* const Kh = lds + hf * 2 * kKB;
  unsigned char* const Vh = lds + 4 * kKB + hf * 2 * kVB;
  const int t = a.tiles - 1 - (int)blockIdx.x / a.H, h = (int)blockIdx.x % a.H;
  const int kvh = h / (a.H / a.Hkv), m0 = t * kSQ, off = a.Skv - a.Sq;
  const int mlast = (m0 + kSQ < a.Sq ? m0 + kSQ : a.Sq) - 1;
  const int nkeys = a.causal ? mlast + off + 1 : a.Skv;               // keys some query of the tile sees
  const int nkb = (nkeys + kSB - 1) / kSB, nb0 = nkb >> 1;
  const int kb0 = hf ? nb0 : 0, kb1 = hf ? nkb : nb0, trips = nkb - nb0;   // the second half has the longer range
  const int mw = m0 + 16 * w4, mq = mw + fr;
  const int seen = a.causal ? mq + off + 1 : a.Skv;                   // keys this lane's query sees
  const int wfirst = a.causal ? mw + off + 1 : a.Skv;                 // ... the wavefront's first query
  const int wmost = mw < a.Sq ? (a.causal ? (mw + 15 < a.Sq ? mw + 15 : a.Sq - 1) + off + 1 : a.Skv) : 0;
  const half_t* kbase = a.k + (size_t)kvh * a.Skv * D;
  const half_t* vbase = a.v + (size_t)kvh * a.Skv * D;
  constexpr int NC = D / 32;              // 16-byte chunks per thread: 64 rows x D / 8 over 256 threads
  u4 kr[NC], vr[NC];
  auto load = [&](int key0) {
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = htid + 256 * i, row = c / (D / 8), ch = c % (D / 8);
      const int key = key0 + row;
      const bool in = key < a.Skv;       // rows past the keys are zeros
      const size_t at = (size_t)(in ? key : 0) * D + ch * 8;
      kr[i] = *(const u4*)(kbase + at);
      vr[i] = *(const u4*)(vbase + at);
      if (!in) { kr[i] = (u4){0u, 0u, 0u, 0u}; vr[i] = kr[i]; }
    }
  };
  auto stage = [&](int s, int i4) {
    uint32_t bad = 0;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = htid + 256 * i, row = c / (D / 8), ch = c % (D / 8);
      *(u4*)(Kh + s * kKB + row * KR + ch * 16) = kr[i];
      *(u4*)(Vh + s * kVB + v_at<D>(row, ch)) = vr[i];
      const uint32_t w[4] = {vr[i].x, vr[i].y, vr[i].z, vr[i].w};
#pragma unroll
      for (int j = 0; j < 4; ++j) bad |= ((w[j] & 0x7C007C00u) + 0x04000400u) & 0x80008000u;   // a full exponent carries into its sign
    }
    if (bad) odd[hf][i4] = 1;
  };
  if (tid < 8) odd[tid >> 2][tid & 3] = 0;
  if (kb0 < kb1) load(kb0 * kSB);
  h8 qf[KS];
  {
    const half_t* qrow = a.q + ((size_t)h * a.Sq + (mq < a.Sq ? mq : a.Sq - 1)) * D;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = __builtin_bit_cast(h8, *(const u4*)(qrow + ks * 32 + 8 * fg));
  }
  f4 acc[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d) acc[d] = (f4){0.0f, 0.0f, 0.0f, 0.0f};
  float mrow = -INFINITY, lrow = 0.0f;
  __syncthreads();                       // odd is cleared
  if (kb0 < kb1) stage(0, 0);
  __syncthreads();
  for (int i = 0; i < trips; ++i) {
    const int kb = kb0 + i, s = i & 1, key0 = kb * kSB;
    const bool mine = kb < kb1, more = kb + 1 < kb1;   // uniform over the half
    if (more) load(key0 + kSB);
    if (mine && key0 < wmost) {
      f4 st[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        st[j] = (f4){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const h8 kf = __builtin_bit_cast(h8, *(const u4*)(Kh + s * kKB + (j * 16 + fr) * KR + (ks * 32 + 8 * fg) * 2));
          st[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, qf[ks], st[j], 0, 0, 0);
        }
      }
      const bool hidden = key0 + kSB > (wfirst < a.Skv ? wfirst : a.Skv);   // some key of the block is masked (uniform)
      float bm = -INFINITY;
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          st[j][e] *= a.scale_log2;
          if (hidden && key0 + j * 16 + 4 * fg + e >= seen) st[j][e] = -INFINITY;
          bm = fmaxf(bm, st[j][e]);
        }
      bm = swap32_max(swap16_max(bm));
      const float mn = fmaxf(mrow, bm), me = mn == -INFINITY ? 0.0f : mn;
      const bool grew = mn > mrow;
      const float alpha = __builtin_amdgcn_exp2f(mrow - me);
      mrow = mn;
      float rs = 0.0f;
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          st[j][e] = __builtin_amdgcn_exp2f(st[j][e] - me);
          rs += st[j][e];
        }
      lrow = lrow * alpha + swap32_sum(swap16_sum(rs));
      if (__builtin_amdgcn_ballot_w64(grew)) {
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[d][e] *= alpha;
      }
      if (!odd[hf][i & 3]) {
        h8 pf[2][3];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            float p = st[2 * ks + (e >> 2)][e & 3] * kPScale;
#pragma unroll
            for (int i = 0; i < 3; ++i) {
              pf[ks][i][e] = (half_t)p;
              p -= (float)pf[ks][i][e];                // exact
            }
          }
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
          for (int ks = 0; ks < 2; ++ks) {
            // lane (fr, fg) asks for dims 16 d + 4 (fr & 3) .. of key 32 ks + 4 fg + fr / 4 and receives
            // dim 16 d + fr of keys 32 ks + 4 fg + 0..3; the second read takes keys + 16
            const int row = ks * 32 + 4 * fg + (fr >> 2);
            unsigned char* const vp = Vh + s * kVB + v_at<D>(row, 2 * d + ((fr >> 1) & 1)) + (fr & 1) * 8;
            const v4s a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)vp);
            const v4s a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(vp + 16 * VR));
            const h8 vf = __builtin_bit_cast(h8, (v8s){a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]});
#pragma unroll
            for (int i = 2; i >= 0; --i) acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, pf[ks][i], acc[d], 0, 0, 0);
          }
      } else {
        // key by key: the weight from the lane that holds it, only where the query sees the key
#pragma unroll 1
        for (int key = 0; key < kSB; ++key) {
          float p = 0.0f;
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (j * 4 + e == (key >> 4) * 4 + (key & 3)) p = st[j][e];
          p = __shfl(p, fr + 16 * ((key >> 2) & 3), 64) * kPScale;
          if (key0 + key < seen) {
#pragma unroll
            for (int d = 0; d < ND; ++d) {
              const half_t* vk = (const half_t*)(Vh + s * kVB + v_at<D>(key, 2 * d + (fg >> 1)) + (fg & 1) * 8);
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[d][e] = __builtin_fmaf(p, (float)vk[e], acc[d][e]);
            }
          }
        }
      }
    }
    if (htid == 0) odd[hf][(i + 2) & 3] = 0;           // last read two blocks ago
    if (more) stage(s ^ 1, (i + 1) & 3);   // the stage was last read before the previous barrier
    __syncthreads();
  }
  // the second half hands over through the idle K stages, lane-major
  float* const xw = (float*)lds + w4 * kX * 64 + lane;
  if (hf) {
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
      for (int e = 0; e < 4; ++e) xw[(d * 4 + e) * 64] = acc[d][e];
    xw[(4 * ND) * 64] = mrow;
    xw[(4 * ND + 1) * 64] = lrow;
  }
  __syncthreads();
  if (hf || mq >= a.Sq) return;
  const float mb = xw[(4 * ND) * 64], lb = xw[(4 * ND + 1) * 64];
  const float mn = fmaxf(mrow, mb);
  const float sa = mrow == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mrow - mn);
  const float sb = mb == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mb - mn);
  const float inv = 1.0f / (lrow * sa + lb * sb) * (1.0f / kPScale);
  half_t* orow = a.o + ((size_t)h * a.Sq + mq) * D + 4 * fg;
#pragma unroll
  for (int d = 0; d < ND; ++d) {
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = (acc[d][e] * sa + xw[(d * 4 + e) * 64] * sb) * inv;   // a half without keys: 0 * 0
    const h2 lo = {(half_t)v[0], (half_t)v[1]}, hi = {(half_t)v[2], (half_t)v[3]};
    *(u2*)(orow + d * 16) = (u2){as_u32(lo), as_u32(hi)};
  }
}

}  // namespace afx

using namespace afx;

extern "C" {

int afx_sdpa(const void* q, const void* k, const void* v, void* o, int H, int Hkv, int Sq, int Skv, int D, int causal,
             float scale, void* stream) {
  AFX_REQUIRE(q && k && v && o, "afx_sdpa: null pointer");
  AFX_REQUIRE(D == 64 || D == 128, "afx_sdpa: head dim %d not supported (64, 128)", D);
  AFX_REQUIRE(Hkv >= 1 && H >= Hkv && H % Hkv == 0, "afx_sdpa: bad heads H=%d Hkv=%d", H, Hkv);
  AFX_REQUIRE(Sq >= 1 && Skv >= 1 && (!causal || Skv >= Sq), "afx_sdpa: bad lengths Sq=%d Skv=%d", Sq, Skv);
  AFX_REQUIRE(Sq < (1 << 30) && Skv < (1 << 30) && (long long)H * ((Sq + kSQ - 1) / kSQ) < (1ll << 31), "afx_sdpa: too large");
  AFX_REQUIRE((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)o) & 15) == 0, "afx_sdpa: buffers must be 16-byte aligned");
  SdpaArgs a = {(const half_t*)q, (const half_t*)k, (const half_t*)v, (half_t*)o, H, Hkv, Sq, Skv, (Sq + kSQ - 1) / kSQ, causal,
                scale * 1.4426950408889634f};
  const dim3 grid((unsigned)(a.tiles * H));
  if (D == 64) hipLaunchKernelGGL(sdpa_kernel<64>, grid, dim3(512), 0, (hipStream_t)stream, a);
  else hipLaunchKernelGGL(sdpa_kernel<128>, grid, dim3(512), 0, (hipStream_t)stream, a);
  return check_launch("afx_sdpa");
}

}  // extern "C"
