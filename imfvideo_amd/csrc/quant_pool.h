// INT8 quantisation and router pooling of q and k tiles: the body that
// quant_pool_kernel and quant_states_kernel run.  Every fp32 product and sum
// rounds separately, in the order written, whatever the translation unit's
// contraction mode.
#pragma once

#include "common.h"

namespace sla2h {

constexpr int kTile = 64;  // E = D = 64

struct QuantPoolArgs {
  const uint16_t* x[2];   // (BH, L, 64) 16-bit
  int8_t* xq[2];          // (BH, L, 64)
  float* xs[2];           // (BH, Nb)
  float* pool[2];         // q: (BH, Nb, 64); k: (BH, 64, npool) transposed; may be null
  const float* proj[2];   // (64, 64) or null
  int npool[2];           // number of leading blocks to pool
  int64_t pool_len[2];    // rows that count for pooling (L for q, Np*E for k)
  int transposed[2];
  float* kb[2];           // (BH, Nb) or null: bound on the tile's dequantised row norms
  int BH;
  int64_t L;
  int Nb;
};

// Both of q and k, as sla2h_quant_pool_qk takes them
inline QuantPoolArgs quant_pool_qk_args(const void* q, const void* k, int BH, int64_t L, int Np,
                                        const float* proj_q, const float* proj_k, int8_t* q8,
                                        float* qs, int8_t* k8, float* ks, float* qpool,
                                        float* kpool_t, float* kbound) {
  QuantPoolArgs a = {};
  a.BH = BH;
  a.L = L;
  a.Nb = (int)((L + kTile - 1) / kTile);
  a.x[0] = static_cast<const uint16_t*>(q);
  a.x[1] = static_cast<const uint16_t*>(k);
  a.xq[0] = q8;
  a.xq[1] = k8;
  a.xs[0] = qs;
  a.xs[1] = ks;
  a.pool[0] = qpool;
  a.pool[1] = kpool_t;
  a.proj[0] = proj_q;
  a.proj[1] = proj_k;
  a.npool[0] = a.Nb;
  a.npool[1] = Np;
  a.pool_len[0] = L;
  a.pool_len[1] = (int64_t)Np * kTile;
  a.transposed[0] = 0;
  a.transposed[1] = 1;
  a.kb[1] = kbound;
  return a;
}

// Exact quotient fl(x / s) without a division per element (Markstein's
// correction): with r = fl(1 / s) correctly rounded and q0 = fl(x r) within an
// ulp of x / s, e = x - q0 s is exact under the FMA and fl(q0 + e r) is the
// correctly rounded quotient (checked against IEEE division for every 16-bit
// x and tile maximum: equal except for denormal x, whose quotients both
// round to 0).
__device__ inline float quotient(float x, float s, float r) {
#pragma clang fp contract(off)
  const float q0 = x * r;
  return __builtin_fmaf(__builtin_fmaf(-q0, s, x), r, q0);
}

// Round half away from zero of the quotient q = quotient(x, s, 1/s):
// trunc(fl(q + sign(x) (0.5 - 2^-25))).  The constant just below 0.5 keeps
// q = 0.5 - 2^-25 at 0 (q + 0.5 would round up to 1 there), and exact ties
// k + 0.5 still round away (the sum rounds up to k + 1).  With x and the tile
// maximum both 16-bit values this equals (int)roundf(fl(x / s)) for every
// pair (exhaustive check: tests/quant_law_check.c).
__device__ inline int round_away(float q, float x) {
#pragma clang fp contract(off)
  return (int)(q + __builtin_copysignf(0x1.fffffep-2f, x));
}
// Low bytes of four int32 values packed into one word (three v_perm_b32)
__device__ inline uint32_t pack_bytes(int b0, int b1, int b2, int b3) {
  const uint32_t lo = __builtin_amdgcn_perm((uint32_t)b1, (uint32_t)b0, 0x0c0c0400u);
  const uint32_t hi = __builtin_amdgcn_perm((uint32_t)b3, (uint32_t)b2, 0x0c0c0400u);
  return __builtin_amdgcn_perm(hi, lo, 0x05040100u);
}

// Tiles are numbered i = (tensor * BH + bh) * Nb + blk.  Each workgroup of 256
// threads takes tiles i = i0, + G, ... and keeps the
// loads of the next kQuantSets - 1 tiles in flight while it quantises the
// current one: kQuantSets register sets, each reloaded with the tile
// kQuantSets G further on as soon as its data is consumed (the loop is
// unrolled over the sets, so no set is ever copied -- a register copy would
// wait for its load).  Thread tid owns row tid / 4, channels 16 (tid % 4) ..
// +15.  The pooling sums run in wave 0 from a double-buffered LDS copy of the
// tile, so one barrier per tile.
constexpr int kQuantSets = 3;

struct QuantPoolLds {
  uint16_t tile[2][kTile][kTile];  // 16-byte aligned
  float red[2][4];
  float rnorm[2][4];
  float vec[2][kTile];
};

template <typename T16>
__device__ __forceinline__ void quant_pool_tiles(const QuantPoolArgs& a, int ntiles, int i0, int G,
                                                 QuantPoolLds& s_) {
#pragma clang fp contract(off)
  auto& tile = s_.tile;
  auto& red = s_.red;
  auto& rnorm = s_.rnorm;
  auto& vec = s_.vec;
  const int tid = threadIdx.x;
  const int r = tid >> 2;
  const int c0 = (tid & 3) * 16;
  auto load = [&](int i, uint4 (&u)[2]) {
    if (i >= ntiles) return;
    const int blk = i % a.Nb;
    const int y = i / a.Nb;
    const int t = y / a.BH, bh = y - t * a.BH;
    const int64_t row = (int64_t)blk * kTile + r;
    if (row < a.L) {
      const uint4* src = reinterpret_cast<const uint4*>(a.x[t] + ((int64_t)bh * a.L + row) * kTile + c0);
      u[0] = src[0];
      u[1] = src[1];
    } else {
      u[0] = u[1] = make_uint4(0, 0, 0, 0);
    }
  };
  int buf = 0;
  auto body = [&](int i, uint4 (&u)[2]) {
#pragma clang fp contract(off)
    const int blk = i % a.Nb;
    const int y = i / a.Nb;
    const int t = y / a.BH, bh = y - t * a.BH;
    const int64_t row = (int64_t)blk * kTile + r;

    const uint32_t wv[8] = {u[0].x, u[0].y, u[0].z, u[0].w, u[1].x, u[1].y, u[1].z, u[1].w};
    float xv[16];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      xv[2 * k] = T16::to_f32((uint16_t)(wv[k] & 0xffff));
      xv[2 * k + 1] = T16::to_f32((uint16_t)(wv[k] >> 16));
    }
    // tile absmax (max is order-independent, so any reduction tree is exact)
    float am = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) am = fmaxf(am, fabsf(xv[k]));
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) am = fmaxf(am, __shfl_xor(am, m, 64));
    if ((tid & 63) == 0) red[buf][tid >> 6] = am;
    // largest squared row norm of the tile (the bound below needs no exact
    // sum: rounding only moves a softmax shift)
    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) ss = __builtin_fmaf(xv[k], xv[k], ss);
    ss = ss + __shfl_xor(ss, 1, 64);
    ss = ss + __shfl_xor(ss, 2, 64);
#pragma unroll
    for (int m = 4; m <= 32; m <<= 1) ss = fmaxf(ss, __shfl_xor(ss, m, 64));
    if ((tid & 63) == 0) rnorm[buf][tid >> 6] = ss;
    const bool pooled = a.pool[t] != nullptr && blk < a.npool[t];
    if (pooled) {
      *reinterpret_cast<uint4*>(&tile[buf][r][c0]) = u[0];
      *reinterpret_cast<uint4*>(&tile[buf][r][c0 + 8]) = u[1];
    }
    load(i + kQuantSets * G, u);  // this set's data is consumed: refill it
    __syncthreads();
    am = fmaxf(fmaxf(red[buf][0], red[buf][1]), fmaxf(red[buf][2], red[buf][3]));
    const float s = am / 127.0f + 1e-12f;  // IEEE division, then add
    const float rs = 1.0f / s;             // correctly rounded reciprocal

    uint32_t w[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      int qv[4];
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const float x = xv[4 * k + b];
        qv[b] = round_away(quotient(x, s, rs), x);
      }
      w[k] = pack_bytes(qv[0], qv[1], qv[2], qv[3]);
    }
    if (row < a.L)
      *reinterpret_cast<uint4*>(a.xq[t] + ((int64_t)bh * a.L + row) * kTile + c0) =
          make_uint4(w[0], w[1], w[2], w[3]);
    if (tid == 0) a.xs[t][(int64_t)bh * a.Nb + blk] = s;
    // kb >= max_j ||x8_j|| s over the tile's rows: each element of x8 s is
    // within s / 2 of x, so ||x8_j s - x_j|| <= 4 s over 64 channels
    if (tid == 0 && a.kb[t] != nullptr) {
      const float mx = fmaxf(fmaxf(rnorm[buf][0], rnorm[buf][1]), fmaxf(rnorm[buf][2], rnorm[buf][3]));
      a.kb[t][(int64_t)bh * a.Nb + blk] = __builtin_sqrtf(mx) * 1.000001f + 4.f * s;
    }

    // ---- pooling (wave 0): sequential per-channel fp32 sum over the real rows ----
    if (pooled && tid < kTile) {
      const int64_t rem = a.pool_len[t] - (int64_t)blk * kTile;
      const int cnt = rem < kTile ? (int)rem : kTile;
      float acc = 0.f;
      int rr = 0;
      for (; rr + 16 <= cnt; rr += 16) {  // 16 LDS reads in flight, then the adds in row order
        float xr[16];
#pragma unroll
        for (int uu = 0; uu < 16; ++uu) xr[uu] = T16::to_f32(tile[buf][rr + uu][tid]);
#pragma unroll
        for (int uu = 0; uu < 16; ++uu) acc = acc + xr[uu];
      }
      for (; rr < cnt; ++rr) acc = acc + T16::to_f32(tile[buf][rr][tid]);
      const float mean = acc / (float)cnt;
      float outv = mean;
      if (a.proj[t] != nullptr) {
        vec[buf][tid] = mean;
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const float* pr = a.proj[t] + tid * kTile;  // row e of proj: out[e] = sum_d x[d] P[e,d]
        float p = 0.f;
        for (int d = 0; d < kTile; ++d) p = p + vec[buf][d] * pr[d];
        outv = p;
      }
      if (a.transposed[t])
        a.pool[t][((int64_t)bh * kTile + tid) * a.npool[t] + blk] = outv;
      else
        a.pool[t][((int64_t)bh * a.Nb + blk) * kTile + tid] = outv;
    }
    buf ^= 1;
  };
  uint4 u0[2], u1[2], u2[2];
  static_assert(kQuantSets == 3, "one register set per unrolled body below");
  load(i0, u0);
  load(i0 + G, u1);
  load(i0 + 2 * G, u2);
  for (int i = i0; i < ntiles; i += 3 * G) {
    body(i, u0);
    if (i + G >= ntiles) break;
    body(i + G, u1);
    if (i + 2 * G >= ntiles) break;
    body(i + 2 * G, u2);
  }
}

}  // namespace sla2h
