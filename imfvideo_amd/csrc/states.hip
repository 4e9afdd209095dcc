// Linear-branch states (phi(K)^T V per video tile, their tangents and global
// sums), the transposed value tiles used by the attention kernel, and the
// per-query-block complement records.
//
// Reference semantics:
//   phi / states   models/sla2_cube_qat.py:911-958 (_phi_states_kernel)
//   global sums    models/sla2_cube_qat.py:645-648
//   complement     models/sla2_cube_qat.py:510-523, 570-578
#include "common.h"
#include "quant_pool.h"
#include "train_setup.h"

#include <mutex>

namespace sla2h {

constexpr int kT = 64;          // E = D = 64
constexpr int kLds = kT + 8;    // padded LDS row (16-bit elements)
constexpr size_t kRecBytes = 2 * 16384 + 2 * 256;

// One tile (b,h,n) per workgroup.  n < Np: phi, states; every n < Nb: the
// attention kernel's operand tiles, in MFMA fragment order so that each wave
// load there is one contiguous 1 KB (rows past L are zero).  With lane
// (g, r) = (lane/16, lane%16), wave w = keys 16w..16w+15, column tile ct:
//   vt, tangent: [ct][w][lane] 16 B = V[16w+4g+0..3][16ct+r] | dV[same]
//   vt, primal:  [ct][w][lane]  8 B = V[16w+4g+0..3][16ct+r]
//   kt (tangent only): [w][ks][lane] 16 B = K[16w+r][32ks+8g+0..7] for ks 0,1,
//                      dK[16w+r][32(ks-2)+8g+0..7] for ks 2,3
//
// Products phi^T V run on 16-bit MFMA with phi split into hi + lo halves of
// the input's 16-bit type (about 16 significant bits), fp32 accumulate.
// ROUND (training forward): phi is rounded to the 16-bit type first, as the
// reference's softmax(K).to(dtype) (models/sla2_cube_qat.py:728), and the lo
// half vanishes.  RH (the inference states of _hblocks): H is stored
// rounded to the 16-bit type, as the reference keeps HALL in V's dtype.  The
// value operand tiles are written when vt is not NULL.
//
// HBM-bound at scale, by the LDS pipe and latency below.  Rows go to LDS as
// they are (16-byte writes) and the operands, the fragment-ordered value tile
// included, come out transposed (ds_read_b64_tr_b16); the column sums exchange
// 15 values per lane; H is computed as H^T for 16-byte stores.  Against 2-byte
// transposed LDS writes (4-way bank conflicts), 64 cross-lane exchanges per
// sum and 4-byte stores, us: 8 heads x 468 tiles with tangent 68.6 -> 62.0 (370
// MB, 6.0 TB/s), primal 35.1 -> 28.7, training 16 x 468 60.5 -> 44.4, 4 x 64 with
// tangent 13.1 -> 10.2.
template <bool TAN>
struct StatesLds {  // 16-byte aligned
  // phi rows (hi, lo), then (tangent, second phase) dphi rows: one buffer keeps
  // the LDS footprint at four workgroups per CU
  uint16_t ph[2][kT][kLds];   // [hi/lo][r][d]
  uint16_t vs[kT][kLds];      // [r][c]
  uint16_t dvs[TAN ? kT : 1][kLds];
  float zred[2][4][kT];
};

template <typename T16, bool TAN, bool ROUND, bool RH>
__device__ __forceinline__ void linear_states_tile(
    const uint16_t* __restrict__ K, const uint16_t* __restrict__ dK,
    const uint16_t* __restrict__ V, const uint16_t* __restrict__ dV, int64_t L, int Np, int Nb,
    float* __restrict__ Hb, float* __restrict__ dHb, float* __restrict__ zb,
    float* __restrict__ dzb, uint16_t* __restrict__ vt, uint16_t* __restrict__ kt, int n, int bh,
    StatesLds<TAN>& lds) {
  auto& ph = lds.ph;
  auto& vs = lds.vs;
  auto& dvs = lds.dvs;
  auto& zred = lds.zred;
  const int tid = threadIdx.x;
  const int r = tid >> 2;
  const int c0 = (tid & 3) * 16;
  const int w = tid >> 6, l = tid & 63, lr = l & 15, g = l >> 4;
  const int64_t row = (int64_t)n * kT + r;
  const bool valid = row < L;
  const int64_t off = ((int64_t)bh * L + row) * kT + c0;

  struct Row16 {  // 16 consecutive 16-bit values of one row
    u32x4 u[2];
  };
  auto load16 = [&](const uint16_t* src) {
    Row16 x;
#pragma unroll
    for (int k = 0; k < 2; ++k)
      x.u[k] = valid ? reinterpret_cast<const u32x4*>(src + off)[k] : u32x4{0, 0, 0, 0};
    return x;
  };
  auto store16 = [&](uint16_t* dst, const Row16& x) {
    reinterpret_cast<u32x4*>(dst)[0] = x.u[0];
    reinterpret_cast<u32x4*>(dst)[1] = x.u[1];
  };
  auto val = [](const Row16& x, int i) {
    return T16::to_f32((uint16_t)(x.u[i >> 3][(i >> 1) & 3] >> (16 * (i & 1))));
  };

  const bool states = n < Np;  // uniform over the workgroup
  const Row16 vb = load16(V);
  Row16 dvb, kb, dkb;
  if (TAN) dvb = load16(dV);
  if (states || TAN) {
    kb = load16(K);
    if (TAN) dkb = load16(dK);
  }
  store16(&vs[r][c0], vb);
  if (TAN) {
    store16(&dvs[r][c0], dvb);
    // key-operand fragments of this thread's 16 columns: 2 x (K, dK) chunks
    const int kw = r >> 4, rr = r & 15, ksd = c0 >> 5, g0 = (c0 & 31) >> 3;
    unsigned char* base = reinterpret_cast<unsigned char*>(kt) + ((int64_t)bh * Nb + n) * 16384;
#pragma unroll
    for (int h2 = 0; h2 < 2; ++h2) {
      const int lane = (g0 + h2) * 16 + rr;
      *reinterpret_cast<u32x4*>(base + ((kw * 4 + ksd) * 64 + lane) * 16) = kb.u[h2];
      *reinterpret_cast<u32x4*>(base + ((kw * 4 + ksd + 2) * 64 + lane) * 16) = dkb.u[h2];
    }
  }
  // x rows as hi + lo halves of the 16-bit type
  auto store_split = [&](const float (&x)[16]) {
    Row16 hi, lo;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t hw = pack_pair<T16>(x[2 * e], x[2 * e + 1]);
      hi.u[e >> 2][e & 3] = hw;
      lo.u[e >> 2][e & 3] = pack_pair<T16>(x[2 * e] - T16::to_f32((uint16_t)(hw & 0xffff)),
                                           x[2 * e + 1] - T16::to_f32((uint16_t)(hw >> 16)));
    }
    store16(&ph[0][r][c0], hi);
    if (!ROUND) store16(&ph[1][r][c0], lo);
  };
  // Column sums over the wave's 16 rows: a lane holds 16 columns of one row, so
  // each step halves both the rows to add and the columns a lane keeps (15
  // exchanges instead of 64), leaving one column per lane: c0 + 8 b5 + 4 b4 + 2
  // b3 + b2 of its lane bits.
  auto col_sum = [&](const float (&x)[16]) {
    float a8[8], a4[4], a2[2];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const auto s = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, x[i]),
                                                      __builtin_bit_cast(unsigned, x[i + 8]), false, false);
      a8[i] = __builtin_bit_cast(float, (unsigned)s[0]) + __builtin_bit_cast(float, (unsigned)s[1]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const auto s = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a8[i]),
                                                      __builtin_bit_cast(unsigned, a8[i + 4]), false, false);
      a4[i] = __builtin_bit_cast(float, (unsigned)s[0]) + __builtin_bit_cast(float, (unsigned)s[1]);
    }
    const bool b3 = (l & 8) != 0, b2 = (l & 4) != 0;
#pragma unroll
    for (int i = 0; i < 2; ++i)
      a2[i] = (b3 ? a4[i + 2] : a4[i]) + __shfl_xor(b3 ? a4[i] : a4[i + 2], 8, 64);
    return (b2 ? a2[1] : a2[0]) + __shfl_xor(b2 ? a2[0] : a2[1], 4, 64);
  };
  const int zcol = c0 + ((l >> 5) & 1) * 8 + ((l >> 4) & 1) * 4 + ((l >> 3) & 1) * 2 + ((l >> 2) & 1);

  float dphi[16];
  if (states) {
    float x[16], phi[16];
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      x[i] = val(kb, i);
      mx = fmaxf(mx, x[i]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 1, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 2, 64));
    float den = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      phi[i] = __expf(x[i] - mx);
      den += phi[i];
    }
    den += __shfl_xor(den, 1, 64);
    den += __shfl_xor(den, 2, 64);
#pragma unroll
    for (int i = 0; i < 16; ++i) phi[i] = phi[i] / den;
    if (TAN) {
      float dot = 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) dot += phi[i] * val(dkb, i);
      dot += __shfl_xor(dot, 1, 64);
      dot += __shfl_xor(dot, 2, 64);
#pragma unroll
      for (int i = 0; i < 16; ++i) dphi[i] = phi[i] * (val(dkb, i) - dot);
    }
    if (!valid) {  // padding rows of a ragged last tile stay inert
#pragma unroll
      for (int i = 0; i < 16; ++i) phi[i] = dphi[i] = 0.f;
    }
    if (ROUND) {
#pragma unroll
      for (int i = 0; i < 16; ++i) phi[i] = T16::to_f32(T16::from_f32(phi[i]));
    }
    store_split(phi);
    zred[0][w][zcol] = col_sum(phi);
    if (TAN) zred[1][w][zcol] = col_sum(dphi);
  }
  __syncthreads();

  // Four consecutive rows 16 vw + 4 g .. + 3 of one column 16 ct + lr, read
  // transposed: half a K = 32 operand (rows 4 g .. and 16 + 4 g .. of a 32-row
  // step are the K slots of lane group g, in both operands).
  auto quad = [&](const uint16_t (*m)[kLds], int ct, int vw) {
    return lds_read_tr16(&m[16 * vw + 4 * g + (lr >> 2)][16 * ct + 4 * (lr & 3)]);
  };
  auto frag = [&](const uint16_t (*m)[kLds], int ct, int ks) {
    const u32x2 lo = quad(m, ct, 2 * ks), hi = quad(m, ct, 2 * ks + 1);
    return u32x4{lo.x, lo.y, hi.x, hi.y};
  };

  // value-operand tile in fragment order: wave w writes column tile w
  if (vt != nullptr) {
    unsigned char* base = reinterpret_cast<unsigned char*>(vt) +
                          ((int64_t)bh * Nb + n) * (TAN ? 16384 : 8192);
#pragma unroll
    for (int vw = 0; vw < 4; ++vw) {
      const u32x2 a = quad(vs, w, vw);
      if (TAN) {
        const u32x2 b = quad(dvs, w, vw);
        *reinterpret_cast<u32x4*>(base + ((w * 4 + vw) * 64 + l) * 16) = u32x4{a.x, a.y, b.x, b.y};
      } else {
        *reinterpret_cast<u32x2*>(base + ((w * 4 + vw) * 64 + l) * 8) = a;
      }
    }
  }
  if (!states) return;

  if (tid < kT) {
    const int64_t zo = ((int64_t)bh * Np + n) * kT + tid;
    zb[zo] = (zred[0][0][tid] + zred[0][1][tid]) + (zred[0][2][tid] + zred[0][3][tid]);
    if (TAN) dzb[zo] = (zred[1][0][tid] + zred[1][1][tid]) + (zred[1][2][tid] + zred[1][3][tid]);
  }

  // Hb[d][v] = sum_r phi[r][d] V[r][v] as H^T = V^T phi: wave w owns d 16w ..
  // 16w + 15, lane (g, lr) holds v = 16 ct + 4 g .. + 3 of d = 16w + lr (16-byte
  // stores).
  f32x4 acc[4], dacc[4];
#pragma unroll
  for (int ct = 0; ct < 4; ++ct) acc[ct] = dacc[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
  // phase 1: H = phi^T V and the phi^T dV half of dH
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const u32x4 bh_ = frag(ph[0], w, ks);
    u32x4 bl = bh_;
    if (!ROUND) bl = frag(ph[1], w, ks);
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
      const u32x4 av = frag(vs, ct, ks);
      acc[ct] = mfma_16x16x32<T16>(av, bh_, acc[ct]);
      if (!ROUND) acc[ct] = mfma_16x16x32<T16>(av, bl, acc[ct]);
      if (TAN) {
        const u32x4 adv = frag(dvs, ct, ks);
        dacc[ct] = mfma_16x16x32<T16>(adv, bh_, dacc[ct]);
        dacc[ct] = mfma_16x16x32<T16>(adv, bl, dacc[ct]);
      }
    }
  }
  if (TAN) {  // phase 2: dphi replaces phi; dH += dphi^T V
    __syncthreads();
    store_split(dphi);
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const u32x4 bh_ = frag(ph[0], w, ks), bl = frag(ph[1], w, ks);
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) {
        const u32x4 av = frag(vs, ct, ks);
        dacc[ct] = mfma_16x16x32<T16>(av, bh_, dacc[ct]);
        dacc[ct] = mfma_16x16x32<T16>(av, bl, dacc[ct]);
      }
    }
  }
  const int64_t hbase = ((int64_t)bh * Np + n) * kT * kT + (16 * w + lr) * kT + 4 * g;
#pragma unroll
  for (int ct = 0; ct < 4; ++ct) {
    f32x4 x = acc[ct];
    if (RH) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float e = x[i];
        x[i] = T16::to_f32(T16::from_f32(e));
      }
    }
    *reinterpret_cast<f32x4*>(Hb + hbase + 16 * ct) = x;
    if (TAN) *reinterpret_cast<f32x4*>(dHb + hbase + 16 * ct) = dacc[ct];
  }
}

template <typename T16, bool TAN, bool ROUND = false, bool RH = false>
__global__ __launch_bounds__(256) void linear_states_kernel(
    const uint16_t* __restrict__ K, const uint16_t* __restrict__ dK,
    const uint16_t* __restrict__ V, const uint16_t* __restrict__ dV, int64_t L, int Np, int Nb,
    float* __restrict__ Hb, float* __restrict__ dHb, float* __restrict__ zb,
    float* __restrict__ dzb, uint16_t* __restrict__ vt, uint16_t* __restrict__ kt) {
  __shared__ __align__(16) StatesLds<TAN> lds;
  linear_states_tile<T16, TAN, ROUND, RH>(K, dK, V, dV, L, Np, Nb, Hb, dHb, zb, dzb, vt, kt,
                                          blockIdx.x, blockIdx.y, lds);
}

// (batch, head, block) tiles that one grid of three workgroups each holds (2^32
// threads).  No call comes near: their fp32 states alone would take 69 GB, the
// whole primal call over 400 GB.
constexpr int64_t kFusedStatesTiles = 1 << 22;

// The states and, independent of them, the INT8 quantisation and pooling of q
// and k in one launch: workgroups 0 .. BH Nb - 1 take a states tile each (the
// longer ones first), the others a quantisation tile.  The quantisation is bound
// by its barrier and pooling chain, the states by HBM, so they fill each other's
// gaps, and a small call saves a launch.  As two launches -> one, us: 4 heads x 5
// tiles 11.1 -> 6.0, 4 x 64 13.0 -> 8.2, 8 x 130 27.8 -> 22.1, 8 x 468 91.3 -> 86.3,
// 16 x 218 93.6 -> 89.7 (tangent); primal 8 x 468 49.6 -> 47.8.
template <typename T16, bool TAN>
__global__ __launch_bounds__(256) void quant_states_kernel(
    QuantPoolArgs a, int ntiles, const uint16_t* __restrict__ K, const uint16_t* __restrict__ dK,
    const uint16_t* __restrict__ V, const uint16_t* __restrict__ dV, int Np,
    float* __restrict__ Hb, float* __restrict__ dHb, float* __restrict__ zb,
    float* __restrict__ dzb, uint16_t* __restrict__ vt, uint16_t* __restrict__ kt) {
  constexpr size_t kBytes = sizeof(StatesLds<TAN>) > sizeof(QuantPoolLds) ? sizeof(StatesLds<TAN>)
                                                                          : sizeof(QuantPoolLds);
  __shared__ __align__(16) unsigned char lds[kBytes];
  const int ns = a.BH * a.Nb, i = blockIdx.x;
  if (i < ns)
    linear_states_tile<T16, TAN, false, false>(K, dK, V, dV, a.L, Np, a.Nb, Hb, dHb, zb, dzb, vt, kt,
                                               i % a.Nb, i / a.Nb,
                                               *reinterpret_cast<StatesLds<TAN>*>(lds));
  else
    quant_pool_tiles<T16>(a, ntiles, i - ns, gridDim.x - ns, *reinterpret_cast<QuantPoolLds*>(lds));
}

// The training states and, independent of them, the call's setup (2.9 us as a
// launch of its own): workgroups BH Nb .. take 256 of its elements each.
template <typename T16>
__global__ __launch_bounds__(256) void states_setup_kernel(
    const uint16_t* __restrict__ K, const uint16_t* __restrict__ V, int64_t L, int Nb, int ns,
    float* __restrict__ Hb, float* __restrict__ zb, uint16_t* __restrict__ vt, TrainSetup setup) {
  __shared__ __align__(16) StatesLds<false> lds;
  const int i = blockIdx.x;
  if (i < ns)
    linear_states_tile<T16, false, true, false>(K, nullptr, V, nullptr, L, Nb, Nb, Hb, nullptr, zb,
                                                nullptr, vt, nullptr, i % Nb, i / Nb, lds);
  else
    train_setup(setup, (int64_t)(i - ns) * 256 + threadIdx.x);
}

// Global sums over the Np tiles in a fixed order (deterministic): eight partial
// sums of a column, partial w over tiles 32 c + 4 w .. + 3 of every group c of 32
// in order, four at a time as (x0 + x1) + (x2 + x3); then ((p0 + p1) + (p2 + p3))
// + ((p4 + p5) + (p6 + p7)).  It is the order in which comp_gemm_kernel sums
// (SUM below), so both give the same bits.  64 columns per workgroup of 256
// threads, two partials a thread.
// Column index e spans [Hb 4096 | dHb 4096 | zb 64 | dzb 64].
__global__ __launch_bounds__(256) void states_sum_kernel(const float* __restrict__ Hb,
                                                        const float* __restrict__ dHb,
                                                        const float* __restrict__ zb,
                                                        const float* __restrict__ dzb, int Np,
                                                        float* __restrict__ Hall,
                                                        float* __restrict__ dHall,
                                                        float* __restrict__ zall,
                                                        float* __restrict__ dzall) {
  __shared__ float part[8][64];
  const int c = threadIdx.x & 63, part_id = threadIdx.x >> 6;
  const int e = blockIdx.x * 64 + c;
  const int bh = blockIdx.y;
  const float* src;
  float* dst;
  int stride, col;
  if (e < 4096) {
    src = Hb; dst = Hall; stride = 4096; col = e;
  } else if (e < 8192) {
    src = dHb; dst = dHall; stride = 4096; col = e - 4096;
  } else if (e < 8256) {
    src = zb; dst = zall; stride = 64; col = e - 8192;
  } else {
    src = dzb; dst = dzall; stride = 64; col = e - 8256;
  }
  if (src == nullptr) return;  // uniform: a workgroup never spans two parts
  const float* p = src + (int64_t)bh * Np * stride + col;
  float acc[2] = {0.f, 0.f};
  auto at = [&](int n) { return n < Np ? p[(int64_t)n * stride] : 0.f; };
#pragma unroll 4
  for (int n0 = 4 * part_id; n0 < Np; n0 += 32)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int n = n0 + 16 * u;
      acc[u] += (at(n) + at(n + 1)) + (at(n + 2) + at(n + 3));
    }
  part[part_id][c] = acc[0];
  part[part_id + 4][c] = acc[1];
  __syncthreads();
  if (part_id == 0)
    dst[(int64_t)bh * stride + col] =
        ((part[0][c] + part[1][c]) + (part[2][c] + part[3][c])) +
        ((part[4][c] + part[5][c]) + (part[6][c] + part[7][c]));
}

// ---------------------------------------------------------------------------
// Complement records.  For each query block m of a head:
//   Hc[m] = sum over the video tiles n NOT routed for m of Hb[n]   (and dHc, zc, dzc)
// computed as a GEMM per head, C = Mc . S, with Mc[m][n] = 1 - sel(m, n)
// (Mb x Np, 0/1) and S = [Hb | dHb | zb | dzb] (Np x 8320 columns, fp32).  S
// is split into bf16 hi + lo halves (about 16 significant bits) and the
// products accumulate in fp32 on MFMA; the mask is exact in bf16.  The H
// columns run in comp_gemm_kernel, the z columns in comp_mask_kernel (small
// calls: all of it in comp_gemm_kernel, see kFusedMaskWords).
//
// Record of (b,h,m), kRecBytes bytes, fp32:
//   [0, 16384) Hc[d][v] row-major, [16384, 32768) dHc, [32768, 33024) zc,
//   [33024, 33280) dzc.
// ---------------------------------------------------------------------------
constexpr int kMaskSub = 32;  // 16-row mask sub-tiles per GEMM workgroup (512 rows)
constexpr int kCompCols = 64;  // state columns per GEMM workgroup
constexpr int kCompThreads = 512;  // 8 waves
// One launch for masks, z and H columns where that is the faster one: the
// workgroups of each column tile build the same mask, so it pays while the
// launch it saves costs more than that.  Measured (two launches -> one, us; 130
// workgroups a head with tangent, 65 without):
//   heads x query blocks   4, tangent     6            8            12
//   5, T = 2 of 4        7.3 ->  5.3   7.9 ->  6.0   8.7 ->  7.3  10.3 ->  9.6
//   32, T = 3 of 32      7.4 ->  5.9   8.6 ->  7.0   9.5 ->  8.5  11.5 -> 11.1
//   64, T = 6 of 64      8.8 ->  7.7  11.0 ->  9.3  12.3 -> 12.3  15.9 -> 16.3
//   64, T = 16 of 64     9.2 ->  9.1  10.9 -> 10.2  12.1 -> 13.4  15.6 -> 17.4
//   96, T = 10 of 96    10.5 -> 10.8  13.8 -> 12.6  15.9 -> 16.4  20.3 -> 21.6
// (primal: the same at twice the heads, within 0.8), so up to 780 workgroups; the
// two launches' GEMM is at its best at 512, two a CU.  Past the other lines, 2048
// LUT entries a workgroup, 4 x 64, T = 32 of 64, 9.3 -> 11.3; four mask words, 8 x
// 130, T = 12 of 128, 12.9 -> 14.4; 8 x 300, T = 3 of 32, 12.7 -> 13.1.
constexpr int kFusedMaskWords = 3;        // 32 tiles each
constexpr int kFusedMaskRows = 96;        // query blocks
constexpr int kFusedMaskEntries = 1024;   // LUT entries of a workgroup's rows
constexpr int kFusedMaskGroups = 780;     // workgroups

// 8 mask bits -> the 8 bf16 A-operand slots (1.0 where set)
__device__ __forceinline__ u32x4 expand_mask8(uint32_t b) {
  u32x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t v = (b >> (2 * e)) & 3u;
    o[e] = ((v & 1u) | ((v & 2u) << 15)) * 0x3F80u;
  }
  return o;
}

// Complement bit masks cbits[bh][kc][m] (m < 16 MT): bit j of word (kc, m) is
// 1 where tile n = 32 kc + j < Np is not routed for query block m < Mb.
// With zb given, the workgroup also writes the zc (and, with dzb, dzc) parts
// of its 16 query blocks' records: the same 0/1-mask product as the GEMM
// below (bf16 hi + lo halves of zb, chunks of 32 tiles in the same order).
// Wave w owns columns 16 (w % 4) .. + 15 of zc (w < 4) or of dzc (w >= 4,
// eight waves with the tangent).  This keeps the 64- and 128-column z parts
// out of the GEMM's grid.
__global__ __launch_bounds__(512) void comp_mask_kernel(const int32_t* __restrict__ lut, int Mb,
                                                      int Np, int T, int MT, int NC,
                                                      uint32_t* __restrict__ cbits,
                                                      const float* __restrict__ zb,
                                                      const float* __restrict__ dzb,
                                                      unsigned char* __restrict__ comp) {
  extern __shared__ uint32_t selbits[];  // [16][NC]
  const int mt = blockIdx.x, bh = blockIdx.y, tid = threadIdx.x;
  const int nthr = blockDim.x;
  for (int i = tid; i < 16 * NC; i += nthr) selbits[i] = 0u;
  __syncthreads();
  for (int i = tid; i < 16 * T; i += nthr) {
    const int row = i / T, jj = i % T;
    const int m = mt * 16 + row;
    if (m >= Mb) continue;
    const int n = lut[((int64_t)bh * Mb + m) * T + jj];
    if ((unsigned)n < (unsigned)Np) atomicOr(&selbits[row * NC + (n >> 5)], 1u << (n & 31));
  }
  __syncthreads();
  for (int i = tid; i < NC * 16; i += nthr) {
    const int kc = i >> 4, row = i & 15;
    const int m = mt * 16 + row;
    const int nv = Np - 32 * kc;  // real tiles in this word
    const uint32_t valid = nv >= 32 ? 0xffffffffu : ((1u << nv) - 1u);
    cbits[((int64_t)bh * NC + kc) * (MT * 16) + m] = m < Mb ? (~selbits[row * NC + kc] & valid) : 0u;
  }
  if (zb == nullptr) return;

  const int w = tid >> 6, l = tid & 63, r = l & 15, g = l >> 4;
  const int part = w >> 2, cw = w & 3;  // part 0: zc from zb, 1: dzc from dzb
  const bool rowok = mt * 16 + r < Mb;
  // tiles n >= Np read as 0 (buffer range check); four chunks of loads in flight
  const auto rz = make_rsrc((part ? dzb : zb) + (int64_t)bh * Np * kT, (int64_t)Np * kT * 4);
  const int coff = (16 * cw + r) * 4;
  auto split = [](const float* x, u32x4& hi, u32x4& lo) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t h = pack_pair<BF16>(x[2 * e], x[2 * e + 1]);
      hi[e] = h;
      lo[e] = pack_pair<BF16>(x[2 * e] - __builtin_bit_cast(float, h << 16),
                              x[2 * e + 1] - __builtin_bit_cast(float, h & 0xffff0000u));
    }
  };
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int kU = 4;
  for (int kc0 = 0; kc0 < NC; kc0 += kU) {
    float x[kU][8];
#pragma unroll
    for (int u = 0; u < kU; ++u)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int off = (32 * (kc0 + u) + 8 * g + j) * (kT * 4) + coff;
        x[u][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rz, off, 0, 0));
      }
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int kc = kc0 + u;
      if (kc >= NC) break;
      const int nv = Np - 32 * kc;
      const uint32_t valid = nv >= 32 ? 0xffffffffu : ((1u << nv) - 1u);
      const uint32_t word = rowok ? (~selbits[r * NC + kc] & valid) : 0u;
      const u32x4 am = expand_mask8((word >> (8 * g)) & 0xffu);
      u32x4 hi, lo;
      split(x[u], hi, lo);
      acc = mfma_bf16_16x16x32(am, hi, acc);
      acc = mfma_bf16_16x16x32(am, lo, acc);
    }
  }
  // lane (g, r) element i = C[query block 16 mt + 4g + i][column 16 cw + r]
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = mt * 16 + 4 * g + i;
    if (m >= Mb) continue;
    unsigned char* rec = comp + ((int64_t)bh * Mb + m) * kRecBytes;
    reinterpret_cast<float*>(rec + 32768 + 256 * part)[16 * cw + r] = acc[i];
  }
}

// One workgroup of 8 waves: 64 state columns x up to 512 query blocks of one
// head (wave w owns the 16-row tiles w, w+8, w+16, w+24, so 64 accumulator
// registers per lane and four waves per SIMD).  The contraction over video
// tiles runs in chunks of 32, double-buffered in LDS and prefetched two
// chunks ahead.  Staging: thread (wave w, column c) loads rows 4w..4w+3 of
// column c, splits them into bf16 hi + lo and writes half a B-operand
// fragment of each with one 8-byte LDS store.  The A operand (0/1 mask)
// comes from the row's mask byte, one 16-entry nibble table read per half.
//
// MASK: the workgroup builds the mask words of its rows itself, in LDS, from
// the LUT (and the one of column tile 0 also stores them to cbits_out), and the
// z columns are two more column tiles: no comp_mask_kernel before it.
//
// SUM (training): the column sums over all tiles as well, Hall and (may be NULL)
// zall, in fp32 from the rows that the staging holds anyway, where
// states_sum_kernel read them again: 16 heads x 468 tiles 25 us, 4 x 64 tiles
// 4 us and a launch; the GEMM takes the same time.  Its first workgroup also copies
// the call's finished lse maxima to the caller's buffer (stats, may be NULL).
template <bool TAN, bool MASK, bool SUM = false>
__global__ __launch_bounds__(kCompThreads, 4) void comp_gemm_kernel(
    const float* __restrict__ Hb, const float* __restrict__ dHb, const float* __restrict__ zb,
    const float* __restrict__ dzb, const uint32_t* __restrict__ cbits, int Mb, int Np, int MT,
    int NC, unsigned char* __restrict__ comp, const int32_t* __restrict__ lut, int T,
    uint32_t* __restrict__ cbits_out, float* __restrict__ Hall, float* __restrict__ zall,
    const float* __restrict__ lse_max, float* __restrict__ stats, int nstats) {
  __shared__ float psum[SUM ? 2 : 1][SUM ? 8 : 1][kCompCols];
  extern __shared__ uint32_t lbits[];  // MASK: [kc][local row], 16 kMaskSub rows
  __shared__ __align__(16) uint16_t sb[2][2][kCompCols][40];  // [buf][hi/lo][column][n] (+pad)
  __shared__ __align__(16) uint32_t mw[2][MASK ? 1 : 16 * kMaskSub];  // [buf][local row] mask words
  // mask nibble -> four bf16 operand slots: 16 entries of 8 bytes occupy 32 distinct LDS
  // banks, so lanes reading different entries never conflict
  __shared__ __align__(16) u32x2 mexp[16];

  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l = tid & 63, r = l & 15, g = l >> 4;
  const int c0 = blockIdx.x * kCompCols;
  const int bh = blockIdx.y;
  const int mt0 = blockIdx.z * kMaskSub;
  const int MTp = MT * 16;
  const int m0 = mt0 * 16;

  // column tile -> source tensor (boundaries are multiples of 64)
  const float* src;
  int stride, col0, part;  // part: 0 Hc, 1 dHc, 2 zc, 3 dzc
  const int zbase = TAN ? 8192 : 4096;
  if (c0 < 4096) {
    src = Hb; stride = 4096; col0 = c0; part = 0;
  } else if (TAN && c0 < 8192) {
    src = dHb; stride = 4096; col0 = c0 - 4096; part = 1;
  } else if (c0 < zbase + 64) {
    src = zb; stride = 64; col0 = c0 - zbase; part = 2;
  } else {
    src = dzb; stride = 64; col0 = c0 - zbase - 64; part = 3;
  }
  // tile rows n >= Np and mask words past the head read as 0 (buffer range check)
  const auto rs = make_rsrc(src + (int64_t)bh * Np * stride, (int64_t)Np * stride * 4);
  const auto rb = make_rsrc(MASK ? reinterpret_cast<const uint32_t*>(lut)
                                 : cbits + (int64_t)bh * NC * MTp, (int64_t)NC * MTp * 4);

  if (tid < 16) {
    const u32x4 e = expand_mask8(tid);
    mexp[tid] = u32x2{e[0], e[1]};
  }

  if constexpr (MASK) {
    constexpr int kRows = 16 * kMaskSub;
    const int rows = min(kRows, MTp - m0);
    for (int i = tid; i < NC * kRows; i += kCompThreads) lbits[i] = 0u;
    __syncthreads();
    const int real = min(rows, Mb - m0);  // rows of real query blocks
    const int32_t* lrow = lut + ((int64_t)bh * Mb + m0) * T;
    for (int i = tid; i < real * T; i += kCompThreads) {
      const int row = i / T;
      const int n = lrow[i];
      if ((unsigned)n < (unsigned)Np) atomicOr(&lbits[(n >> 5) * kRows + row], 1u << (n & 31));
    }
    __syncthreads();
    for (int i = tid; i < NC * kRows; i += kCompThreads) {
      const int kc = i / kRows, row = i - kc * kRows;
      const int nv = Np - 32 * kc;  // real tiles in this word
      const uint32_t valid = nv >= 32 ? 0xffffffffu : ((1u << nv) - 1u);
      const uint32_t wd = row < real ? (~lbits[i] & valid) : 0u;
      lbits[i] = wd;
      if (c0 == 0 && row < rows) cbits_out[((int64_t)bh * NC + kc) * MTp + m0 + row] = wd;
    }
  }

  f32x4 acc[4][4];
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) acc[s][ct] = f32x4{0.f, 0.f, 0.f, 0.f};

  struct Chunk {
    float x[4];
    uint32_t mk;
  };
  const int xoff = (col0 + l) * 4 + 4 * w * stride * 4;
  auto load_chunk = [&](int kc, Chunk& c) {
    kc = min(kc, NC - 1);  // past the end: a harmless reload, never stored
#pragma unroll
    for (int j = 0; j < 4; ++j)
      c.x[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                             rs, xoff + (32 * kc + j) * stride * 4, 0, 0));
    if (!MASK) c.mk = __builtin_amdgcn_raw_buffer_load_b32(rb, (kc * MTp + m0 + tid) * 4, 0, 0);
  };
  float sum = 0.f;
  auto store_chunk = [&](int buf, const Chunk& c, int kc) {
    if (SUM && kc < NC) sum += (c.x[0] + c.x[1]) + (c.x[2] + c.x[3]);
    u32x2 hi, lo;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const uint32_t h = pack_pair<BF16>(c.x[2 * e], c.x[2 * e + 1]);
      hi[e] = h;
      lo[e] = pack_pair<BF16>(c.x[2 * e] - __builtin_bit_cast(float, h << 16),
                              c.x[2 * e + 1] - __builtin_bit_cast(float, h & 0xffff0000u));
    }
    *reinterpret_cast<u32x2*>(&sb[buf][0][l][4 * w]) = hi;
    *reinterpret_cast<u32x2*>(&sb[buf][1][l][4 * w]) = lo;
    if (!MASK) mw[buf][tid] = c.mk;
  };
  const unsigned char* mwb = reinterpret_cast<const unsigned char*>(MASK ? lbits : &mw[0][0]);
  auto compute = [&](int buf, int kc) {
    u32x4 bhi[4], blo[4];
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
      bhi[ct] = *reinterpret_cast<const u32x4*>(&sb[buf][0][ct * 16 + r][8 * g]);
      blo[ct] = *reinterpret_cast<const u32x4*>(&sb[buf][1][ct * 16 + r][8 * g]);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int lt = w + 8 * s;  // local 16-row tile; uniform per wave
      if (mt0 + lt < MT) {
        const uint32_t mb = mwb[((MASK ? kc : buf) * 16 * kMaskSub + lt * 16 + r) * 4 + g];
        const u32x2 alo = mexp[mb & 15u], ahi = mexp[mb >> 4];
        const u32x4 am = u32x4{alo.x, alo.y, ahi.x, ahi.y};
#pragma unroll
        for (int ct = 0; ct < 4; ++ct) {
          acc[s][ct] = mfma_bf16_16x16x32(am, bhi[ct], acc[s][ct]);
          acc[s][ct] = mfma_bf16_16x16x32(am, blo[ct], acc[s][ct]);
        }
      }
    }
  };

  Chunk ca, cb;
  load_chunk(0, ca);
  load_chunk(1, cb);
  store_chunk(0, ca, 0);
  __syncthreads();
  for (int kc = 0; kc < NC; kc += 2) {
    // chunk kc in buffer 0, chunk kc+1 in registers cb
    load_chunk(kc + 2, ca);
    compute(0, kc);
    store_chunk(1, cb, kc + 1);  // buffer 1 was last read before the previous barrier
    __syncthreads();
    if (kc + 1 >= NC) break;
    load_chunk(kc + 3, cb);
    compute(1, kc + 1);
    store_chunk(0, ca, kc + 2);
    __syncthreads();
  }

  if constexpr (SUM) {
    if (stats != nullptr && blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0)
      for (int i = tid; i < nstats; i += kCompThreads) stats[i] = lse_max[i];
    // with the masks the z columns are a column tile of their own; otherwise the
    // first column tile's workgroup sums them too
    const bool zsum = !MASK && c0 == 0 && zall != nullptr;
    psum[0][w][l] = sum;
    if (zsum) {
      const auto rz = make_rsrc(zb + (int64_t)bh * Np * 64, (int64_t)Np * 256);
      float zs = 0.f;
#pragma unroll 4
      for (int kc = 0; kc < NC; ++kc) {
        float x[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
          x[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                               rz, (32 * kc + 4 * w + j) * 256 + 4 * l, 0, 0));
        zs += (x[0] + x[1]) + (x[2] + x[3]);
      }
      psum[1][w][l] = zs;
    }
    __syncthreads();
    if (w < 2 && blockIdx.z == 0) {
      float* dst = w == 0 ? (part == 0 ? Hall + (int64_t)bh * 4096 + col0
                                       : (zall != nullptr ? zall + (int64_t)bh * 64 : nullptr))
                          : (zsum ? zall + (int64_t)bh * 64 : nullptr);
      if (dst != nullptr) {
        const auto& p = psum[w];
        dst[l] = ((p[0][l] + p[1][l]) + (p[2][l] + p[3][l])) +
                 ((p[4][l] + p[5][l]) + (p[6][l] + p[7][l]));
      }
    }
  }

  // records: lane (g, r) element i = C[16 mt + 4g + i][c0 + 16 ct + r]; 16
  // consecutive columns of one record per 16 lanes
  const int pbase = part < 2 ? part * 16384 : 32768 + (part - 2) * 256;
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int mt = mt0 + w + 8 * s;
    if (mt >= MT) break;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = mt * 16 + 4 * g + i;
      if (m >= Mb) continue;
      float* rec = reinterpret_cast<float*>(comp + ((int64_t)bh * Mb + m) * kRecBytes + pbase);
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) rec[col0 + ct * 16 + r] = acc[s][ct][i];
    }
  }
}

}  // namespace sla2h

using namespace sla2h;

extern "C" size_t sla2h_complement_record_bytes(int D) { return D == kT ? kRecBytes : 0; }

extern "C" int sla2h_linear_states(const void* k, const void* dk, const void* v, const void* dv,
                                   int dtype, int B, int H, int64_t L, int D, int E, int Np,
                                   float* Hb, float* dHb, float* zb, float* dzb, float* Hall,
                                   float* dHall, float* zall, float* dzall, void* vt, void* kt,
                                   void* stream) {
  SLA2H_CHECK_ARG(k && v && Hb && zb && vt);
  SLA2H_CHECK_ARG((Hall == nullptr) == (zall == nullptr));
  SLA2H_CHECK_ARG(D == kT && E == kT);
  SLA2H_CHECK_ARG(dtype == SLA2H_DTYPE_F16 || dtype == SLA2H_DTYPE_BF16);
  SLA2H_CHECK_ARG(B > 0 && H > 0 && B * H <= 65535);
  // Np * E <= L for cube video tiles; Np = Nb (every tile, the last one
  // possibly partial) for 1-D key blocks
  SLA2H_CHECK_ARG(Np > 0 && (int64_t)(Np - 1) * E < L);
  const bool tan = dk != nullptr;
  if (tan) SLA2H_CHECK_ARG(dv && dHb && dzb && kt);
  if (tan && Hall) SLA2H_CHECK_ARG(dHall && dzall);
  const int Nb = (int)((L + E - 1) / E);
  hipStream_t st = static_cast<hipStream_t>(stream);
  dim3 grid(Nb, B * H);
  auto K = static_cast<const uint16_t*>(k);
  auto dK = static_cast<const uint16_t*>(dk);
  auto V = static_cast<const uint16_t*>(v);
  auto dV = static_cast<const uint16_t*>(dv);
  auto VT = static_cast<uint16_t*>(vt);
  auto KT = static_cast<uint16_t*>(kt);
  if (dtype == SLA2H_DTYPE_BF16) {
    if (tan)
      linear_states_kernel<BF16, true><<<grid, 256, 0, st>>>(K, dK, V, dV, L, Np, Nb, Hb, dHb, zb, dzb, VT, KT);
    else
      linear_states_kernel<BF16, false><<<grid, 256, 0, st>>>(K, dK, V, dV, L, Np, Nb, Hb, dHb, zb, dzb, VT, KT);
  } else {
    if (tan)
      linear_states_kernel<F16, true><<<grid, 256, 0, st>>>(K, dK, V, dV, L, Np, Nb, Hb, dHb, zb, dzb, VT, KT);
    else
      linear_states_kernel<F16, false><<<grid, 256, 0, st>>>(K, dK, V, dV, L, Np, Nb, Hb, dHb, zb, dzb, VT, KT);
  }
  int err = (int)hipGetLastError();
  if (err || Hall == nullptr) return err;
  dim3 g2(8320 / 64, B * H);
  states_sum_kernel<<<g2, 256, 0, st>>>(Hb, tan ? dHb : nullptr, zb, tan ? dzb : nullptr, Np, Hall,
                                        dHall, zall, dzall);
  return (int)hipGetLastError();
}

namespace sla2h {

// sla2h_linear_states_qat without the sums over the tiles, and a training
// forward's setup
int states_and_setup(const void* k, const void* v, int dtype, int B, int H, int64_t L, float* Hb,
                     float* zb, void* vt, const TrainSetup& setup, void* stream) {
  SLA2H_CHECK_ARG(k && v && Hb && zb);
  SLA2H_CHECK_ARG(dtype == SLA2H_DTYPE_F16 || dtype == SLA2H_DTYPE_BF16);
  SLA2H_CHECK_ARG(B > 0 && H > 0 && B * H <= 65535 && L > 0);
  const int Nb = (int)((L + kT - 1) / kT);
  const int64_t ns = (int64_t)B * H * Nb;
  int64_t n = setup.nl > setup.na ? setup.nl : setup.na;
  if (setup.stats != nullptr && n < setup.H) n = setup.H;
  const int64_t grid = ns + (n + 255) / 256;
  SLA2H_CHECK_ARG(grid < (1 << 24));  // 2^32 threads
  hipStream_t st = static_cast<hipStream_t>(stream);
  auto K = static_cast<const uint16_t*>(k);
  auto V = static_cast<const uint16_t*>(v);
  auto VT = static_cast<uint16_t*>(vt);
  if (dtype == SLA2H_DTYPE_BF16)
    states_setup_kernel<BF16><<<(unsigned)grid, 256, 0, st>>>(K, V, L, Nb, (int)ns, Hb, zb, VT, setup);
  else
    states_setup_kernel<F16><<<(unsigned)grid, 256, 0, st>>>(K, V, L, Nb, (int)ns, Hb, zb, VT, setup);
  return (int)hipGetLastError();
}

}  // namespace sla2h

extern "C" int sla2h_linear_states_qat(const void* k, const void* v, int dtype, int B, int H,
                                       int64_t L, int D, int E, float* Hb, float* zb, float* Hall,
                                       float* zall, void* vt, void* stream) {
  SLA2H_CHECK_ARG(k && v && Hb && zb && Hall && zall);
  SLA2H_CHECK_ARG(D == kT && E == kT);
  SLA2H_CHECK_ARG(dtype == SLA2H_DTYPE_F16 || dtype == SLA2H_DTYPE_BF16);
  SLA2H_CHECK_ARG(B > 0 && H > 0 && B * H <= 65535 && L > 0);
  const int Nb = (int)((L + E - 1) / E);
  hipStream_t st = static_cast<hipStream_t>(stream);
  dim3 grid(Nb, B * H);
  auto K = static_cast<const uint16_t*>(k);
  auto V = static_cast<const uint16_t*>(v);
  if (dtype == SLA2H_DTYPE_BF16)
    linear_states_kernel<BF16, false, true><<<grid, 256, 0, st>>>(K, nullptr, V, nullptr, L, Nb, Nb, Hb, nullptr, zb, nullptr, static_cast<uint16_t*>(vt), nullptr);
  else
    linear_states_kernel<F16, false, true><<<grid, 256, 0, st>>>(K, nullptr, V, nullptr, L, Nb, Nb, Hb, nullptr, zb, nullptr, static_cast<uint16_t*>(vt), nullptr);
  const int err = (int)hipGetLastError();
  if (err) return err;
  dim3 g2(8320 / 64, B * H);
  states_sum_kernel<<<g2, 256, 0, st>>>(Hb, nullptr, zb, nullptr, Nb, Hall, nullptr, zall, nullptr);
  return (int)hipGetLastError();
}

// Inference states of the 1-D SLA2 (_hblocks through complement_linear_states,
// models/sla2_vendor/kernel_linear.py:396-427, 496-504): phi(K) rounded to the
// 16-bit type, HALL_j = phi(K_j)^T V_j rounded to the 16-bit type (held as
// fp32 values), ZALL_j = colsum phi(K_j) in fp32, for every key block; the
// sums over the blocks when Hall / zall are given; the primal value operand
// tiles of the 16-bit sparse kernel when vt is given.
extern "C" int sla2h_hblocks_states(const void* k, const void* v, int dtype, int B, int H,
                                    int64_t L, int D, int E, float* Hb, float* zb, float* Hall,
                                    float* zall, void* vt, void* stream) {
  SLA2H_CHECK_ARG(k && v && Hb && zb);
  SLA2H_CHECK_ARG((Hall == nullptr) == (zall == nullptr));
  SLA2H_CHECK_ARG(D == kT && E == kT);
  SLA2H_CHECK_ARG(dtype == SLA2H_DTYPE_F16 || dtype == SLA2H_DTYPE_BF16);
  SLA2H_CHECK_ARG(B > 0 && H > 0 && B * H <= 65535 && L > 0);
  const int Nb = (int)((L + E - 1) / E);
  hipStream_t st = static_cast<hipStream_t>(stream);
  dim3 grid(Nb, B * H);
  auto K = static_cast<const uint16_t*>(k);
  auto V = static_cast<const uint16_t*>(v);
  if (dtype == SLA2H_DTYPE_BF16)
    linear_states_kernel<BF16, false, true, true><<<grid, 256, 0, st>>>(K, nullptr, V, nullptr, L, Nb, Nb, Hb, nullptr, zb, nullptr, static_cast<uint16_t*>(vt), nullptr);
  else
    linear_states_kernel<F16, false, true, true><<<grid, 256, 0, st>>>(K, nullptr, V, nullptr, L, Nb, Nb, Hb, nullptr, zb, nullptr, static_cast<uint16_t*>(vt), nullptr);
  int err = (int)hipGetLastError();
  if (err || Hall == nullptr) return err;
  dim3 g2(8320 / 64, B * H);
  states_sum_kernel<<<g2, 256, 0, st>>>(Hb, nullptr, zb, nullptr, Nb, Hall, nullptr, zall, nullptr);
  return (int)hipGetLastError();
}

// Backward complement.  sel[bh][n][kc] bit j = 1 where query block
// m = 32 kc + j routes tile n (augmented LUT); the GEMM above then runs with
// the roles swapped: rows = tiles n, contraction over query blocks m, mask
// = NOT sel, operands = the per-query-block partials [P | Pz].
__global__ __launch_bounds__(256) void fill_u32_kernel(uint32_t* __restrict__ p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = 0u;
}

__global__ __launch_bounds__(256) void sel_scatter_kernel(const int32_t* __restrict__ lut, int Mb,
                                                         int Mq, int qshift, int J, int NCq,
                                                         uint32_t* __restrict__ sel) {
  const int bh = blockIdx.y;
  const int idx = blockIdx.x * 256 + threadIdx.x;  // over 64-row query blocks x J
  if (idx >= Mb * J) return;
  const int m = idx / J;
  const int n = lut[((int64_t)bh * Mq + (m >> qshift)) * J + (idx - m * J)];
  if ((unsigned)n < (unsigned)Mb)
    atomicOr(&sel[((int64_t)bh * Mb + n) * NCq + (m >> 5)], 1u << (m & 31));
}

__global__ __launch_bounds__(256) void sel_complement_kernel(const uint32_t* __restrict__ sel,
                                                            int Mb, int NCq, int MTp,
                                                            uint32_t* __restrict__ cbits) {
  const int bh = blockIdx.y;
  const int idx = blockIdx.x * 256 + threadIdx.x;  // over NCq * MTp
  if (idx >= NCq * MTp) return;
  const int kc = idx / MTp, n = idx - kc * MTp;
  uint32_t wd = 0u;
  if (n < Mb) {
    const int nv = Mb - 32 * kc;
    const uint32_t valid = nv >= 32 ? 0xffffffffu : ((1u << nv) - 1u);
    wd = ~sel[((int64_t)bh * Mb + n) * NCq + kc] & valid;
  }
  cbits[(int64_t)bh * NCq * MTp + idx] = wd;
}

namespace sla2h {
// The mask GEMM of the backward: records of Mb key tiles from the partial states
// [P | Pz] of Mb query blocks and the masks cbits.
int complement_gemm_bwd(const float* P, const float* Pz, const uint32_t* cbits, int BH, int Mb,
                        void* comp, void* stream) {
  const int MT = (Mb + 15) / 16, NC = (Mb + 31) / 32;
  dim3 grid(4160 / kCompCols, BH, (MT + kMaskSub - 1) / kMaskSub);
  comp_gemm_kernel<false, false><<<grid, kCompThreads, 0, static_cast<hipStream_t>(stream)>>>(
      P, nullptr, Pz, nullptr, cbits, Mb, Mb, MT, NC, static_cast<unsigned char*>(comp), nullptr, 0,
      nullptr, nullptr, nullptr, nullptr, nullptr, 0);
  return (int)hipGetLastError();
}
}  // namespace sla2h

extern "C" int sla2h_complement_bwd(const float* P, const float* Pz, const int32_t* lut_aug,
                                    int B, int H, int Mb, int bq, int J, void* workspace,
                                    uint32_t* sel, void* comp, void* stream) {
  SLA2H_CHECK_ARG(P && Pz && lut_aug && workspace && sel && comp);
  SLA2H_CHECK_ARG(B > 0 && H > 0 && B * H <= 65535 && Mb > 0 && Mb <= 4096 && J >= 1);
  SLA2H_CHECK_ARG(bq == 64 || bq == 128 || bq == 256);
  const int qshift = bq == 64 ? 0 : (bq == 128 ? 1 : 2);
  const int Mq = (Mb + (1 << qshift) - 1) >> qshift;
  const int MT = (Mb + 15) / 16, NC = (Mb + 31) / 32;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int64_t nsel = (int64_t)B * H * Mb * NC;
  fill_u32_kernel<<<(unsigned)((nsel + 255) / 256), 256, 0, st>>>(sel, nsel);
  sel_scatter_kernel<<<dim3((Mb * J + 255) / 256, B * H), 256, 0, st>>>(lut_aug, Mb, Mq, qshift, J,
                                                                       NC, sel);
  auto cbits = static_cast<uint32_t*>(workspace);
  sel_complement_kernel<<<dim3((NC * MT * 16 + 255) / 256, B * H), 256, 0, st>>>(sel, Mb, NC,
                                                                               MT * 16, cbits);
  int err = (int)hipGetLastError();
  if (err) return err;
  return complement_gemm_bwd(P, Pz, cbits, B * H, Mb, comp, stream);
}

extern "C" size_t sla2h_complement_workspace_bytes(int B, int H, int Mb, int Np) {
  if (B <= 0 || H <= 0 || Mb <= 0 || Np <= 0) return 0;
  const size_t MT = (size_t)(Mb + 15) / 16, NC = (size_t)(Np + 31) / 32;
  return (size_t)B * H * NC * MT * 16 * 4;
}

// ---------------------------------------------------------------------------
// Allocation-free complement: the bit-mask workspace lives in this file-scope
// device array (one copy per GPU, held until the process ends).  Host code
// never uses the array's name as an address: the device address of each GPU's
// copy comes from hipGetSymbolAddress, taken once per device on the first
// call with that device current, and is kept here.  The mask kernel writes
// every word the GEMM reads, so nothing needs clearing between calls; calls
// that overlap on one GPU (several streams or threads) race on the array.
// ---------------------------------------------------------------------------
static __device__ __align__(256) unsigned char scratch[SLA2H_COMPLEMENT_SCRATCH_BYTES];

namespace {
constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxScratchDevices] = {};

int complement_scratch(void** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= kMaxScratchDevices) return (int)hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    if (ptr == nullptr) return (int)hipErrorInvalidSymbol;
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return 0;
}
}  // namespace

namespace sla2h {

// sla2h_complement; with Hall (primal only) the sums of Hb and, where zall is
// given, of zb over the tiles as well, and with stats (H) a copy of lse_max there
int complement_sums(const float* Hb, const float* dHb, const float* zb, const float* dzb,
                    const int32_t* lut, int B, int H, int Mb, int Np, int D, int T,
                    void* workspace, void* comp, float* Hall, float* zall, const float* lse_max,
                    float* stats, void* stream) {
  SLA2H_CHECK_ARG(Hb && zb && lut && comp && workspace);
  SLA2H_CHECK_ARG(!stats || (Hall && lse_max));
  SLA2H_CHECK_ARG(D == kT);
  SLA2H_CHECK_ARG(B > 0 && H > 0 && B * H <= 65535 && Mb > 0 && Np > 0 && Np <= 4096);
  SLA2H_CHECK_ARG(T >= 1 && T <= Np);
  const bool tan = dHb != nullptr;
  if (tan) SLA2H_CHECK_ARG(dzb && !Hall);
  const int MT = (Mb + 15) / 16, NC = (Np + 31) / 32;
  hipStream_t st = static_cast<hipStream_t>(stream);
  auto cbits = static_cast<uint32_t*>(workspace);
  auto out = static_cast<unsigned char*>(comp);
  const unsigned groups = (unsigned)((MT + kMaskSub - 1) / kMaskSub);
  const int tiles = (tan ? 8320 : 4160) / kCompCols;
  if (NC <= kFusedMaskWords && Mb <= kFusedMaskRows && (int64_t)Mb * T <= kFusedMaskEntries &&
      (int64_t)tiles * B * H <= kFusedMaskGroups) {  // so one group of rows
    dim3 grid(tiles, B * H, groups);
    const size_t shmem = (size_t)NC * 16 * kMaskSub * 4;
    if (tan)
      comp_gemm_kernel<true, true><<<grid, kCompThreads, shmem, st>>>(
          Hb, dHb, zb, dzb, nullptr, Mb, Np, MT, NC, out, lut, T, cbits, nullptr, nullptr,
          nullptr, nullptr, 0);
    else if (Hall)
      comp_gemm_kernel<false, true, true><<<grid, kCompThreads, shmem, st>>>(
          Hb, nullptr, zb, nullptr, nullptr, Mb, Np, MT, NC, out, lut, T, cbits, Hall, zall,
          lse_max, stats, H);
    else
      comp_gemm_kernel<false, true><<<grid, kCompThreads, shmem, st>>>(
          Hb, nullptr, zb, nullptr, nullptr, Mb, Np, MT, NC, out, lut, T, cbits, nullptr, nullptr,
          nullptr, nullptr, 0);
    return (int)hipGetLastError();
  }
  // mask bits plus the z parts of the records; the GEMM takes the H parts only
  // (128 or 64 column tiles per head: whole rounds of workgroups)
  comp_mask_kernel<<<dim3(MT, B * H), tan ? 512 : 256, (size_t)16 * NC * 4, st>>>(
      lut, Mb, Np, T, MT, NC, cbits, zb, dzb, out);
  int err = (int)hipGetLastError();
  if (err) return err;
  dim3 grid((tan ? 8192 : 4096) / kCompCols, B * H, groups);
  if (tan)
    comp_gemm_kernel<true, false><<<grid, kCompThreads, 0, st>>>(
        Hb, dHb, zb, dzb, cbits, Mb, Np, MT, NC, out, nullptr, 0, nullptr, nullptr, nullptr,
        nullptr, nullptr, 0);
  else if (Hall)
    comp_gemm_kernel<false, false, true><<<grid, kCompThreads, 0, st>>>(
        Hb, nullptr, zb, nullptr, cbits, Mb, Np, MT, NC, out, nullptr, 0, nullptr, Hall, zall,
        lse_max, stats, H);
  else
    comp_gemm_kernel<false, false><<<grid, kCompThreads, 0, st>>>(
        Hb, nullptr, zb, nullptr, cbits, Mb, Np, MT, NC, out, nullptr, 0, nullptr, nullptr, nullptr,
        nullptr, nullptr, 0);
  return (int)hipGetLastError();
}

}  // namespace sla2h

extern "C" int sla2h_complement(const float* Hb, const float* dHb, const float* zb,
                                const float* dzb, const int32_t* lut, int B, int H, int Mb,
                                int Np, int D, int T, void* workspace, void* comp,
                                void* stream) {
  return complement_sums(Hb, dHb, zb, dzb, lut, B, H, Mb, Np, D, T, workspace, comp, nullptr,
                         nullptr, nullptr, nullptr, stream);
}

namespace sla2h {

// sla2h_quant_pool_qk (a) and sla2h_linear_states without the global sums, in one
// launch.
int quant_states(const QuantPoolArgs& a, const void* k, const void* dk, const void* v,
                 const void* dv, int dtype, int Np, float* Hb, float* dHb, float* zb, float* dzb,
                 void* vt, void* kt, void* stream) {
  const int64_t ns = (int64_t)a.BH * a.Nb;
  SLA2H_CHECK_ARG(ns <= kFusedStatesTiles);
  SLA2H_CHECK_ARG(k && v && Hb && zb && vt && Np > 0 && (int64_t)Np * kT <= a.L);
  SLA2H_CHECK_ARG(dtype == SLA2H_DTYPE_F16 || dtype == SLA2H_DTYPE_BF16);
  if (dk) SLA2H_CHECK_ARG(dv && dHb && dzb && kt);
  auto run = [&](auto kernel) {
    kernel<<<(unsigned)(3 * ns), 256, 0, static_cast<hipStream_t>(stream)>>>(
        a, (int)(2 * ns), static_cast<const uint16_t*>(k), static_cast<const uint16_t*>(dk),
        static_cast<const uint16_t*>(v), static_cast<const uint16_t*>(dv), Np, Hb, dHb, zb, dzb,
        static_cast<uint16_t*>(vt), static_cast<uint16_t*>(kt));
    return (int)hipGetLastError();
  };
  if (dtype == SLA2H_DTYPE_BF16)
    return dk ? run(quant_states_kernel<BF16, true>) : run(quant_states_kernel<BF16, false>);
  return dk ? run(quant_states_kernel<F16, true>) : run(quant_states_kernel<F16, false>);
}

}  // namespace sla2h

extern "C" int sla2h_complement_noalloc(const float* Hb, const float* dHb, const float* zb,
                                        const float* dzb, const int32_t* lut, int B, int H,
                                        int Mb, int Np, int D, int T, void* comp, void* stream) {
  SLA2H_CHECK_ARG(Hb && zb && lut && comp);
  SLA2H_CHECK_ARG(B > 0 && H > 0 && Mb > 0 && Np > 0);
  SLA2H_CHECK_ARG(sla2h_complement_workspace_bytes(B, H, Mb, Np) <=
                  (size_t)SLA2H_COMPLEMENT_SCRATCH_BYTES);
  void* ws = nullptr;
  const int err = complement_scratch(&ws);
  if (err) return err;
  return sla2h_complement(Hb, dHb, zb, dzb, lut, B, H, Mb, Np, D, T, ws, comp, stream);
}
