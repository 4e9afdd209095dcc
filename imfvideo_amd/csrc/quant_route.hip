// INT8 block quantisation, router tile pooling and block top-k for gfx950.
//
// This translation unit is compiled with -ffp-contract=off: every fp32
// product and sum below rounds separately, in the order written, so the
// results are bit-identical to the CPU restatement in oracle/.
//
// Reference semantics:
//   quantisation  models/sla2_vendor/kernel_sparse_qat.py:120-151
//   tile pooling  models/mla_video_sparse_jvp.py:506-529, 545-562
//   scores+top-k  models/mla_video_sparse_jvp.py:563-565, 292-294
#include "common.h"
#include "quant_pool.h"

#include <type_traits>

namespace sla2h {

// fp32 input "storage tag" (16-bit tags: common.h)
struct F32In {
  __device__ static inline float to_f32(float f) { return f; }
};

template <typename T16>
__global__ __launch_bounds__(256) void quant_pool_kernel(QuantPoolArgs a, int ntiles) {
  __shared__ __align__(16) QuantPoolLds lds;
  quant_pool_tiles<T16>(a, ntiles, blockIdx.x, gridDim.x, lds);
}

// Training-forward quantisation (semantics of the in-kernel quantisation of
// _attn_fwd_qat, models/sla2_vendor/kernel_sparse_qat.py:56-58, 88-90,
// 106-107): s = max|x| / 127 + 1e-12 per 64 x 64 tile, q = (int) fl(fl(x / s)
// + 0.5 sign(x)) truncated toward zero (sign(+-0) = +1).  Q and K keep the
// row-major (BH, L, 64) int8 layout; V is written as INT8 MFMA A-operand
// fragments of O^T = V8^T P8^T: per tile [ct][lane][16 B], byte s of lane
// (g, rr) of column tile ct = V8[16 (s >> 2) + 4 g + (s & 3)][16 ct + rr].
struct QuantTrainArgs {
  const uint16_t* x[3];  // q, k, v (BH, L, 64)
  int8_t* xq[3];         // q8, k8 (BH, L, 64); v8f (BH, Nb, 4096)
  float* xs[3];          // (BH, Nb)
  int BH;
  int64_t L;
  int Nb;
  int t0;                // first tensor of the grid (blockIdx.y / BH counts from it)
};

// RND: the round-half-away law of quantize_qkv instead (the inference INT8
// path, sla2h_quantize_v8f).
template <typename T16, bool RND = false>
__global__ __launch_bounds__(256) void quant_train_kernel(QuantTrainArgs a) {
  __shared__ float red[4];
  __shared__ __align__(16) int8_t q8t[kTile][kTile + 16];

  const int tid = threadIdx.x;
  const int blk = blockIdx.x;
  const int t = a.t0 + blockIdx.y / a.BH;
  const int bh = blockIdx.y % a.BH;
  const int r = tid >> 2;
  const int c0 = (tid & 3) * 16;
  const int64_t row = (int64_t)blk * kTile + r;
  const bool valid = row < a.L;
  const int64_t off = ((int64_t)bh * a.L + row) * kTile + c0;

  float xv[16];
  if (valid) {
    const uint4* src = reinterpret_cast<const uint4*>(a.x[t] + off);
    uint4 u0 = src[0], u1 = src[1];
    uint32_t w[8] = {u0.x, u0.y, u0.z, u0.w, u1.x, u1.y, u1.z, u1.w};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      xv[2 * i] = T16::to_f32((uint16_t)(w[i] & 0xffff));
      xv[2 * i + 1] = T16::to_f32((uint16_t)(w[i] >> 16));
    }
  } else {
#pragma unroll
    for (int i = 0; i < 16; ++i) xv[i] = 0.f;
  }
  float am = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) am = fmaxf(am, fabsf(xv[i]));
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) am = fmaxf(am, __shfl_xor(am, m, 64));
  if ((tid & 63) == 0) red[tid >> 6] = am;
  __syncthreads();
  am = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const float s = am / 127.0f + 1e-12f;

  uint32_t w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t acc = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const float x = xv[4 * i + b];
      int qv;
      if (RND) {
        qv = (int)roundf(x / s);  // round half away from zero
      } else {
        const float y = x / s + (x >= 0.f ? 0.5f : -0.5f);  // two roundings (no contraction)
        qv = (int)y;
      }
      acc |= ((uint32_t)(qv & 0xff)) << (8 * b);
    }
    w[i] = acc;
  }
  if (tid == 0) a.xs[t][(int64_t)bh * a.Nb + blk] = s;
  if (t < 2) {
    if (valid) *reinterpret_cast<uint4*>(a.xq[t] + off) = make_uint4(w[0], w[1], w[2], w[3]);
    return;
  }
  // V: transpose to the fragment order through LDS (rows past L are zero)
  *reinterpret_cast<uint4*>(&q8t[r][c0]) = make_uint4(w[0], w[1], w[2], w[3]);
  __syncthreads();
  const int ct = tid >> 6, lane = tid & 63, g = lane >> 4, rr = lane & 15;
  uint32_t f[4];
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    uint32_t acc = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      acc |= ((uint32_t)(uint8_t)q8t[16 * kb + 4 * g + i][16 * ct + rr]) << (8 * i);
    f[kb] = acc;
  }
  *reinterpret_cast<uint4*>(a.xq[2] + ((int64_t)bh * a.Nb + blk) * 4096 + tid * 16) =
      make_uint4(f[0], f[1], f[2], f[3]);
}

// Everything done to q, k and v before the INT8 attention, in one pass: token
// layout and 16-bit cast (rows_in_kernel's), the INT8 law (truncating as
// quant_train_kernel, or with RND half away from zero as quant_rows_kernel) and
// the router's pooled and projected blocks of q and k (pool_pair_kernel's), equal
// to the bit.  q in blocks of 64 NB rows, k and v of 64; one (tensor, head, block)
// per workgroup, heads fastest, thread tid = rows tid / 4 + 64 c, channels 16
// (tid % 4) .. + 15; the pooling sums run in wave 0 from an LDS copy.  HBM-bound:
// each element is read once.  Training, against three launches that wrote the
// rows and read them twice more: 2 x 8 heads x 29,952 fp16 tokens 153 -> 122 us,
// 8 heads x 8,269 bf16 tokens 33.9 -> 15.4 us.
struct OperandArgs {
  const void* x[3];              // (B, L, H, 64), strides below
  int64_t sb[3], st[3], sh[3];
  const int64_t* idx;            // token of row l, or null
  uint16_t* rows[3];             // (B, H, L, 64) 16-bit, or null
  int8_t* xq[3];                 // q8, k8 (B, H, L, 64); v8f (B, H, Nb, 4096)
  float* xs[3];                  // (B, H, blocks)
  float* pool[2];                // (B, H, Mq, 64); (B, H, 64, Np)
  const float* proj[2];
  int B, H, Nb, Np, Mq;
  int64_t L;
};

// TS: storage type of x, TR: the 16-bit type it is rounded to
template <typename TS, typename Raw, typename TR, bool RND, int NB>
__global__ __launch_bounds__(256) void operand_kernel(OperandArgs a) {
  __shared__ __align__(16) uint16_t tile[64 * NB][kTile];
  __shared__ __align__(16) int8_t q8t[kTile][kTile + 16];
  __shared__ float red[4];
  __shared__ float vec[kTile];
  const int tid = threadIdx.x;
  int i = blockIdx.x;
  const int nq = a.B * a.H * a.Mq, nk = a.B * a.H * a.Nb;
  const int t = i < nq ? 0 : (i < nq + nk ? 1 : 2);
  i -= t == 0 ? 0 : (t == 1 ? nq : nq + nk);
  const int nblk = t == 0 ? a.Mq : a.Nb;  // blocks of this tensor per head
  const int per = t == 0 ? kTile * NB : kTile;  // rows per block
  const int h = i % a.H, i1 = i / a.H;
  const int n = i1 % nblk, b = i1 / nblk;
  const int r = tid >> 2, c0 = (tid & 3) * 16;
  const int64_t bh = (int64_t)b * a.H + h;
  const int64_t row0 = (int64_t)n * per + r;
  const int64_t off = (bh * a.L + row0) * kTile + c0;
  const bool pooled = t == 0 || (t == 1 && n < a.Np);

  float xv[NB][16];
  float am = 0.f;
#pragma unroll
  for (int c = 0; c < NB; ++c) {
    if (c > 0 && t != 0) break;  // uniform
    const int64_t row = row0 + 64 * c;
    uint32_t w16[8] = {0, 0, 0, 0, 0, 0, 0, 0};  // the row segment in 16 bits
    if (row < a.L) {
      int64_t tok = row;
      if (a.idx != nullptr) {
        tok = a.idx[row];
        tok = tok < 0 ? 0 : (tok >= a.L ? a.L - 1 : tok);
      }
      const Raw* src = static_cast<const Raw*>(a.x[t]) + b * a.sb[t] + tok * a.st[t] + h * a.sh[t] + c0;
      if constexpr (sizeof(Raw) == 4) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float4 v = reinterpret_cast<const float4*>(src)[k];
          w16[2 * k] = pack_pair<TR>(v.x, v.y);
          w16[2 * k + 1] = pack_pair<TR>(v.z, v.w);
        }
      } else {
        const uint4 u0 = reinterpret_cast<const uint4*>(src)[0], u1 = reinterpret_cast<const uint4*>(src)[1];
        const uint32_t w[8] = {u0.x, u0.y, u0.z, u0.w, u1.x, u1.y, u1.z, u1.w};
#pragma unroll
        for (int k = 0; k < 8; ++k)
          w16[k] = std::is_same<TS, TR>::value
                       ? w[k]
                       : pack_pair<TR>(TS::to_f32((uint16_t)(w[k] & 0xffff)),
                                       TS::to_f32((uint16_t)(w[k] >> 16)));
      }
    }
    const uint4 lo = make_uint4(w16[0], w16[1], w16[2], w16[3]);
    const uint4 hi = make_uint4(w16[4], w16[5], w16[6], w16[7]);
    if (row < a.L && a.rows[t] != nullptr) {
      uint4* dst = reinterpret_cast<uint4*>(a.rows[t] + off + 64 * c * kTile);
      dst[0] = lo;
      dst[1] = hi;
    }
    if (pooled) {
      *reinterpret_cast<uint4*>(&tile[r + 64 * c][c0]) = lo;
      *reinterpret_cast<uint4*>(&tile[r + 64 * c][c0 + 8]) = hi;
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      xv[c][2 * k] = TR::to_f32((uint16_t)(w16[k] & 0xffff));
      xv[c][2 * k + 1] = TR::to_f32((uint16_t)(w16[k] >> 16));
    }
#pragma unroll
    for (int k = 0; k < 16; ++k) am = fmaxf(am, fabsf(xv[c][k]));
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) am = fmaxf(am, __shfl_xor(am, m, 64));
  if ((tid & 63) == 0) red[tid >> 6] = am;
  __syncthreads();
  am = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const float s = am / 127.0f + 1e-12f;  // IEEE division, then add
  const float rs = 1.0f / s;
  if (tid == 0) a.xs[t][bh * nblk + n] = s;
  uint4 q4;
#pragma unroll
  for (int c = 0; c < NB; ++c) {
    if (c > 0 && t != 0) break;
    uint32_t w8[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      int qv[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = xv[c][4 * k + e];
        const float y = quotient(x, s, rs);
        qv[e] = RND ? round_away(y, x) : (int)(y + (x >= 0.f ? 0.5f : -0.5f));
      }
      w8[k] = pack_bytes(qv[0], qv[1], qv[2], qv[3]);
    }
    q4 = make_uint4(w8[0], w8[1], w8[2], w8[3]);
    if (t < 2 && row0 + 64 * c < a.L)
      *reinterpret_cast<uint4*>(a.xq[t] + off + 64 * c * kTile) = q4;
  }
  if (t < 2) {
    if (!pooled || tid >= kTile) return;
    const int64_t rem = (t == 0 ? a.L : min(a.L, (int64_t)a.Np * kTile)) - (int64_t)n * per;
    const int cnt = rem < per ? (int)rem : per;
    float acc = 0.f;
    int rr = 0;
    for (; rr + 16 <= cnt; rr += 16) {  // 16 LDS reads in flight, then the adds in row order
      float xr[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) xr[u] = TR::to_f32(tile[rr + u][tid]);
#pragma unroll
      for (int u = 0; u < 16; ++u) acc = acc + xr[u];
    }
    for (; rr < cnt; ++rr) acc = acc + TR::to_f32(tile[rr][tid]);
    float outv = acc / (float)cnt;
    if (a.proj[t] != nullptr) {
      vec[tid] = outv;
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      const float* pr = a.proj[t] + tid * kTile;  // out[e] = sum_d mean[d] P[e][d]
      float p = 0.f;
#pragma unroll 16
      for (int d = 0; d < kTile; ++d) p = p + vec[d] * pr[d];
      outv = p;
    }
    if (t)
      a.pool[1][(bh * kTile + tid) * a.Np + n] = outv;
    else
      a.pool[0][(bh * a.Mq + n) * kTile + tid] = outv;
    return;
  }
  // V: transpose to the fragment order through LDS (rows past L are zero)
  *reinterpret_cast<uint4*>(&q8t[r][c0]) = q4;
  __syncthreads();
  const int ct = tid >> 6, lane = tid & 63, g = lane >> 4, rr = lane & 15;
  uint32_t f[4];
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    uint32_t acc = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      acc |= ((uint32_t)(uint8_t)q8t[16 * kb + 4 * g + e][16 * ct + rr]) << (8 * e);
    f[kb] = acc;
  }
  *reinterpret_cast<uint4*>(a.xq[2] + (bh * a.Nb + n) * 4096 + tid * 16) =
      make_uint4(f[0], f[1], f[2], f[3]);
}

// quantize_qkv / _quant_blocks (models/sla2_vendor/kernel_sparse_qat.py:
// 120-151) for blocks of E = 32..256 rows: one block per workgroup, thread t
// holds E/4 consecutive elements (a segment of one row), s = max|x| / 127 +
// 1e-12, q = round half away from zero of x / s.  TRUNC: the training
// kernel's law instead, q = (int) fl(fl(x / s) + 0.5 sign(x)) (the in-kernel
// Q quantisation of _attn_fwd_qat, kernel_sparse_qat.py:56-58, for BLOCK_M =
// bq rows).
template <typename T16, int E, bool TRUNC = false>
__global__ __launch_bounds__(256) void quant_rows_kernel(const uint16_t* __restrict__ x, int64_t L,
                                                         int Nb, int8_t* __restrict__ xq,
                                                         float* __restrict__ xs) {
  constexpr int PER = E / 4;
  __shared__ float red[4];
  const int tid = threadIdx.x;
  const int blk = blockIdx.x;
  const int bh = blockIdx.y;
  const int e0 = tid * PER;
  const bool valid = (int64_t)blk * E + e0 / kTile < L;
  const int64_t off = ((int64_t)bh * L + (int64_t)blk * E) * kTile + e0;
  float xv[PER];
#pragma unroll
  for (int c = 0; c < PER / 8; ++c) {
    const uint4 u = valid ? reinterpret_cast<const uint4*>(x + off)[c] : make_uint4(0, 0, 0, 0);
    const uint32_t wd[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      xv[8 * c + 2 * i] = T16::to_f32((uint16_t)(wd[i] & 0xffff));
      xv[8 * c + 2 * i + 1] = T16::to_f32((uint16_t)(wd[i] >> 16));
    }
  }
  float am = 0.f;
#pragma unroll
  for (int i = 0; i < PER; ++i) am = fmaxf(am, fabsf(xv[i]));
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) am = fmaxf(am, __shfl_xor(am, m, 64));
  if ((tid & 63) == 0) red[tid >> 6] = am;
  __syncthreads();
  am = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const float s = am / 127.0f + 1e-12f;  // IEEE division, then add
  uint32_t w[PER / 4];
#pragma unroll
  for (int i = 0; i < PER / 4; ++i) {
    uint32_t acc = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const float xx = xv[4 * i + b];
      const int qv = TRUNC ? (int)(xx / s + (xx >= 0.f ? 0.5f : -0.5f)) : (int)roundf(xx / s);
      acc |= ((uint32_t)(qv & 0xff)) << (8 * b);
    }
    w[i] = acc;
  }
  if (valid) {
    if (PER == 8) {
      *reinterpret_cast<uint2*>(xq + off) = make_uint2(w[0], w[1]);
    } else {
#pragma unroll
      for (int c = 0; c < PER / 16; ++c)
        reinterpret_cast<uint4*>(xq + off)[c] =
            make_uint4(w[4 * c], w[4 * c + 1], w[4 * c + 2], w[4 * c + 3]);
    }
  }
  if (tid == 0) xs[(int64_t)bh * Nb + blk] = s;
}

// Orderable 64-bit key: high word = monotone map of the fp32 score
// (NaN -> +NaN, the largest, as torch.topk orders; -0 -> +0), low word =
// ~index so that equal scores rank the lower index first.
__device__ inline uint64_t score_key(float sc, int n) {
  uint32_t u = __builtin_bit_cast(uint32_t, sc);
  if (sc != sc) u = 0x7fc00000u;
  if (u == 0x80000000u) u = 0u;
  const uint32_t ord = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
  return ((uint64_t)ord << 32) | (uint64_t)(0xffffffffu - (uint32_t)n);
}

// ROWS query blocks of one (b,h) per workgroup: scores into LDS, one
// bitonic sort (descending) per row over P2 = next_pow2(Np) keys, emit top T.
template <int ROWS>
__global__ __launch_bounds__(256) void route_topk_kernel(const float* __restrict__ qpool,
                                                         const float* __restrict__ kpool_t,
                                                         int Mb, int Np, int T, float scale,
                                                         int P2, int32_t* __restrict__ lut,
                                                         uint8_t* __restrict__ mask) {
  extern __shared__ __align__(16) unsigned char smem[];
  uint64_t* keys = reinterpret_cast<uint64_t*>(smem);                 // ROWS * P2
  float* qsh = reinterpret_cast<float*>(smem + (size_t)ROWS * P2 * 8);  // ROWS * 64
  uint8_t* sel = smem + (size_t)ROWS * P2 * 8 + ROWS * kTile * 4;      // ROWS * P2

  const int tid = threadIdx.x;
  const int bh = blockIdx.y;
  const int m0 = blockIdx.x * ROWS;

  for (int idx = tid; idx < ROWS * kTile; idx += 256) {
    const int rr = idx / kTile, d = idx % kTile;
    const int m = m0 + rr;
    qsh[idx] = (m < Mb) ? qpool[((int64_t)bh * Mb + m) * kTile + d] : 0.f;
  }
  for (int idx = tid; idx < ROWS * P2; idx += 256) sel[idx] = 0;
  __syncthreads();

  const float* kt = kpool_t + (int64_t)bh * kTile * Np;
  for (int n = tid; n < P2; n += 256) {
    if (n < Np) {
      float acc[ROWS];
#pragma unroll
      for (int rr = 0; rr < ROWS; ++rr) acc[rr] = 0.f;
      for (int d = 0; d < kTile; ++d) {
        const float kv = kt[(int64_t)d * Np + n];
#pragma unroll
        for (int rr = 0; rr < ROWS; ++rr) acc[rr] = acc[rr] + qsh[rr * kTile + d] * kv;
      }
#pragma unroll
      for (int rr = 0; rr < ROWS; ++rr) keys[rr * P2 + n] = score_key(acc[rr] * scale, n);
    } else {
#pragma unroll
      for (int rr = 0; rr < ROWS; ++rr) keys[rr * P2 + n] = 0ull;  // below every real key
    }
  }
  __syncthreads();

  const int half = P2 >> 1;
  for (int k = 2; k <= P2; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int idx = tid; idx < ROWS * half; idx += 256) {
        const int rr = idx / half, h = idx % half;
        const int i = (h / j) * 2 * j + (h % j);
        const int l = i + j;
        uint64_t* row = keys + rr * P2;
        const uint64_t ki = row[i], kl = row[l];
        const bool desc = (i & k) == 0;  // overall order: descending
        if (desc ? (ki < kl) : (ki > kl)) {
          row[i] = kl;
          row[l] = ki;
        }
      }
      __syncthreads();
    }
  }

  for (int idx = tid; idx < ROWS * T; idx += 256) {
    const int rr = idx / T, jj = idx % T;
    const int m = m0 + rr;
    const uint32_t n = 0xffffffffu - (uint32_t)(keys[rr * P2 + jj] & 0xffffffffull);
    if (m < Mb) lut[((int64_t)bh * Mb + m) * T + jj] = (int32_t)n;
    sel[rr * P2 + n] = 1;
  }
  if (mask == nullptr) return;
  __syncthreads();
  for (int idx = tid; idx < ROWS * Np; idx += 256) {
    const int rr = idx / Np, n = idx % Np;
    const int m = m0 + rr;
    if (m < Mb) mask[((int64_t)bh * Mb + m) * Np + n] = sel[rr * P2 + n];
  }
}

// Top-T of each row by wave-wide radix selection (T <= CAP): one wave per query
// block, NK keys per lane (tile n = lane + 64 i).
//   1. scores, same sequential fp32 order as route_topk_kernel;
//   2. a score word s* that exactly T keys reach, by a 32-bit binary search
//      with ballot counts (it ends at the first bit where the count is T: with
//      distinct scores about half-way); if several keys share the T-th
//      largest word, the lowest indices among them fill up to T (a 13-bit
//      binary search over n);
//   3. the T winners are compacted through LDS and each is written at its
//      rank, the number of winners with a larger 64-bit key (score word, then
//      lower index first).
// Bound by the wave's dependent chains (scores, ballots, ranks), not by
// memory: NK is the smallest that holds Np, and rank counting replaced a
// 64-lane bitonic sort (21 cross-lane exchanges whatever T) and, for T > 64,
// the full sort of every row in LDS.  Heads x rows x Np, T: 4 x 5 x 4, 2:
// 13.2 -> 4.2 us; 16 x 218 x 216, 6: 23.4 -> 11.9; 8 x 468 x 468, 46: 22.9 -> 20.3.
template <int NK, int CAP, bool V4>
__global__ __launch_bounds__(256) void route_select_kernel(const float* __restrict__ qpool,
                                                           const float* __restrict__ kpool_t,
                                                           int Mb, int Np, int T, float scale,
                                                           int32_t* __restrict__ lut,
                                                           uint8_t* __restrict__ mask) {
  // pooled keys of the head, staged in chunks of DC channels (at most 32 KB)
  // that the four waves share
  constexpr int DC = NK == 1 ? kTile : 128 / NK;
  __shared__ float ksh[DC][64 * NK];
  __shared__ uint64_t win[4][CAP];
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int bh = blockIdx.y;
  const int m = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + w);
  const bool active = m < Mb;  // uniform per wave; every wave takes the barriers

  const float* kt = kpool_t + (int64_t)bh * kTile * Np;
  float acc[NK];
#pragma unroll
  for (int i = 0; i < NK; ++i) acc[i] = 0.f;
  // lane d holds q[row][d] (broadcast with readlane).  Key slots past Np
  // need no guard: their scores are never selected (ord = 0 below); the
  // buffer range check returns 0 past the end of this head's pooled keys.
  const float qlane = active ? qpool[((int64_t)bh * Mb + m) * kTile + lane] : 0.f;
  const auto rk = make_rsrc(kt, (int64_t)kTile * Np * 4);
  for (int d0 = 0; d0 < kTile; d0 += DC) {
    __syncthreads();  // the previous chunk is consumed
    if constexpr (V4) {
      // Np % 4 == 0: a channel's row of Np floats is 16-byte aligned, so one
      // 16-byte load carries 4 keys (a load at n < Np lies inside the row)
#pragma unroll
      for (int k = 0; k < DC * 16 * NK / 256; ++k) {
        const int e = tid + 256 * k;
        const int dd = e / (16 * NK), n = 4 * (e % (16 * NK));
        *reinterpret_cast<u32x4*>(&ksh[dd][n]) = buf_load16(rk, ((d0 + dd) * Np + n) * 4, 0);
      }
    } else {
#pragma unroll
      for (int k = 0; k < DC * 64 * NK / 256; ++k) {
        const int e = tid + 256 * k;
        const int dd = e / (64 * NK), n = e % (64 * NK);
        ksh[dd][n] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                   rk, ((d0 + dd) * Np + n) * 4, 0, 0));
      }
    }
    __syncthreads();
    if (active) {
#pragma unroll
      for (int dd = 0; dd < DC; ++dd) {
        const float qv = __builtin_bit_cast(
            float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, qlane), d0 + dd));
#pragma unroll
        for (int i = 0; i < NK; ++i) acc[i] = acc[i] + qv * ksh[dd][lane + 64 * i];
      }
    }
  }
  if (!active) return;  // whole wave; no workgroup barrier below

  uint32_t ord[NK];
#pragma unroll
  for (int i = 0; i < NK; ++i) {
    const int n = lane + 64 * i;
    ord[i] = n < Np ? (uint32_t)(score_key(acc[i] * scale, n) >> 32) : 0u;  // 0: below all
  }
  // wave-wide sum of per-lane counts 0..NK: one ballot per count bit
  constexpr int kBits = NK == 1 ? 1 : NK == 2 ? 2 : NK == 4 ? 3 : NK == 8 ? 4
                      : NK == 16 ? 5 : NK == 32 ? 6 : 7;
  auto wave_sum = [&](int cl) {
    int c = 0;
#pragma unroll
    for (int b = 0; b < kBits; ++b) c += __popcll(__ballot((cl >> b) & 1)) << b;
    return c;
  };
  uint32_t sstar = 0, nstar = 0xffffffffu;  // keys at s* with n <= nstar are taken
  bool exact = false;
  for (int b = 31; b >= 0 && !exact; --b) {
    const uint32_t cand = sstar | (1u << b);
    int cl = 0;
#pragma unroll
    for (int i = 0; i < NK; ++i) cl += ord[i] >= cand ? 1 : 0;
    const int c = wave_sum(cl);
    if (c >= T) sstar = cand;
    exact = c == T;
  }
  if (!exact) {
    int l_gt = 0, l_eq = 0;
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      l_gt += ord[i] > sstar ? 1 : 0;
      l_eq += ord[i] == sstar ? 1 : 0;
    }
    const int c_gt = wave_sum(l_gt), c_eq = wave_sum(l_eq);
    const int need = T - c_gt;  // 1 <= need <= c_eq
    if (need < c_eq) {
      uint32_t pre = 0;
      for (int b = 12; b >= 0; --b) {
        const uint32_t cand = pre | (1u << b);
        int cl = 0;
#pragma unroll
        for (int i = 0; i < NK; ++i) cl += (ord[i] == sstar && (uint32_t)(lane + 64 * i) < cand) ? 1 : 0;
        if (wave_sum(cl) < need) pre = cand;
      }
      nstar = pre;
    }
  }
  // compact the T winners (any order)
  int base = 0;
#pragma unroll
  for (int i = 0; i < NK; ++i) {
    const uint32_t n = lane + 64 * i;
    const bool sel = ord[i] > sstar || (ord[i] == sstar && n <= nstar && (int)n < Np);
    const uint64_t bal = __ballot(sel);
    if (sel) {
      const int pos = base + __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32),
                                                       __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0u));
      win[w][pos] = ((uint64_t)ord[i] << 32) | (uint64_t)(0xffffffffu - n);
    }
    if (mask != nullptr && (int)n < Np) mask[((int64_t)bh * Mb + m) * Np + n] = sel ? 1 : 0;
    base += __popcll(bal);
  }
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  int32_t* row = lut + ((int64_t)bh * Mb + m) * T;
  if constexpr (CAP == 64) {
    const uint64_t key = lane < T ? win[w][lane] : 0ull;
    const int klo = (int)(uint32_t)key, khi = (int)(uint32_t)(key >> 32);
    int rank = 0;
    for (int j = 0; j < T; j += 4) {  // lanes from T on hold key 0, above no winner
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint64_t other = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane(khi, j + u) << 32) |
                               (uint32_t)__builtin_amdgcn_readlane(klo, j + u);
        rank += other > key ? 1 : 0;
      }
    }
    if (lane < T) row[rank] = (int32_t)(0xffffffffu - (uint32_t)key);
  } else {
    for (int i = lane; i < T; i += 64) {
      const uint64_t key = win[w][i];
      int rank = 0;
#pragma unroll 8
      for (int j = 0; j < T; ++j) rank += win[w][j] > key ? 1 : 0;
      row[rank] = (int32_t)(0xffffffffu - (uint32_t)key);
    }
  }
}

}  // namespace sla2h

using namespace sla2h;

// Workgroups cycling over tiles: 16 per CU of 256 (two rounds of eight
// resident ones; measured best among 1024-8192 at Config 3).
constexpr int kQuantGrid = 4096;

static int launch_quant_pool(const QuantPoolArgs& a, int ntens, int dtype, hipStream_t st) {
  const int64_t ntiles = (int64_t)a.Nb * ntens * a.BH;
  if (ntiles >= (1ll << 31) - (kQuantSets + 2) * (int64_t)kQuantGrid) return (int)hipErrorInvalidValue;
  const int grid = (int)(ntiles < kQuantGrid ? ntiles : kQuantGrid);
  if (dtype == SLA2H_DTYPE_BF16)
    quant_pool_kernel<BF16><<<grid, 256, 0, st>>>(a, (int)ntiles);
  else
    quant_pool_kernel<F16><<<grid, 256, 0, st>>>(a, (int)ntiles);
  return (int)hipGetLastError();
}

// Block means for the 1-D router (blocks of blk rows, the last one ragged):
// one block of one (b, h) per workgroup, one thread per channel, sequential
// fp32 sum over the block's real rows, then / count, then the optional
// projection out[e] = sum_d mean[d] proj[e][d] (sequential, no contraction).
template <typename TS, typename Raw>
__global__ __launch_bounds__(64) void pool_blocks_kernel(const Raw* __restrict__ x, int64_t L,
                                                        int blk, int nblk,
                                                        const float* __restrict__ proj,
                                                        int transposed, float* __restrict__ out) {
  using T16 = TS;
  __shared__ float vec[kTile];
  const int j = blockIdx.x, bh = blockIdx.y, d = threadIdx.x;
  const int64_t r0 = (int64_t)j * blk;
  const int cnt = (int)((L - r0) < blk ? (L - r0) : blk);
  const Raw* src = x + ((int64_t)bh * L + r0) * kTile + d;
  float acc = 0.f;
  int rr = 0;
  for (; rr + 16 <= cnt; rr += 16) {  // 16 loads in flight, then the adds in row order
    float xv[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) xv[u] = T16::to_f32(src[(int64_t)(rr + u) * kTile]);
#pragma unroll
    for (int u = 0; u < 16; ++u) acc = acc + xv[u];
  }
  for (; rr < cnt; ++rr) acc = acc + T16::to_f32(src[(int64_t)rr * kTile]);
  vec[d] = acc / (float)cnt;
  __syncthreads();
  float outv = vec[d];
  if (proj != nullptr) {
    const float* pr = proj + d * kTile;
    float p = 0.f;
    for (int e = 0; e < kTile; ++e) p = p + vec[e] * pr[e];
    outv = p;
  }
  if (transposed)
    out[((int64_t)bh * kTile + d) * nblk + j] = outv;
  else
    out[((int64_t)bh * nblk + j) * kTile + d] = outv;
}

// The same block means and projections for a query and a key tensor of 16-bit
// rows in one launch: half a wave per block (lane c: channels 2 c, 2 c + 1, one
// 128-byte row per load, 64 rows of loads in flight ahead of the ordered adds
// and beside the staging of the projection), eight blocks per workgroup.
// Bound by the read of x where there is enough of it: 2 x 16 heads x 29,952 fp16
// rows (123 MB) in 33.8 us (3.6 TB/s), where the quantising kernel that the
// cube router borrowed also wrote 61 MB of INT8 rows (65.4 us); small ones by
// the ordered sums' latency: 8 x 13,901 rows, 128-row query blocks 13.8 us (two
// launches of pool_blocks_kernel: 17.2 us).
struct PoolPairArgs {
  const uint16_t* x[2];
  const float* proj[2];  // (64, 64) or null
  float* out[2];         // [0] (BH, n, 64), [1] transposed (BH, 64, n)
  int blk[2], n[2];      // rows per block, blocks per head
  int BH;
  int64_t L;
  int wg0;               // workgroups of tensor 0
};

template <typename T16>
__global__ __launch_bounds__(256) void pool_pair_kernel(PoolPairArgs a) {
  __shared__ __align__(16) float pt[kTile][kTile + 4];  // the projection [d][e]
  __shared__ __align__(16) float mean[8][kTile];
  const int tid = threadIdx.x;
  const int hw = tid >> 5, c = tid & 31;
  // workgroups of tensor 0, then of tensor 1 (one projection per workgroup)
  const int t = (int)blockIdx.x >= a.wg0;
  const int64_t jj = (int64_t)((int)blockIdx.x - (t ? a.wg0 : 0)) * 8 + hw;
  const bool on = jj < (int64_t)a.BH * a.n[t];
  const int64_t bh = on ? jj / a.n[t] : 0;
  const int j = on ? (int)(jj - bh * a.n[t]) : 0;
  const int64_t r0 = (int64_t)j * a.blk[t];
  const int cnt = (int)(a.L - r0 < a.blk[t] ? a.L - r0 : a.blk[t]);
  const uint32_t* src = reinterpret_cast<const uint32_t*>(a.x[t]) + (bh * a.L + r0) * 32 + c;
  constexpr int kRows = 64;
  uint32_t v[kRows];
  auto load = [&](int rr) {  // rows past the block reload its last one
#pragma unroll
    for (int u = 0; u < kRows; ++u) {
      const int row = rr + u < cnt ? rr + u : cnt - 1;
      v[u] = src[row * 32];
    }
  };
  load(0);
  const float* proj = a.proj[t];
  if (proj != nullptr) {
    for (int i = tid; i < kTile * kTile; i += 256) pt[i & 63][i >> 6] = proj[i];
    __syncthreads();
  }
  float s0 = 0.f, s1 = 0.f;
  for (int rr = 0;;) {
    if (rr + kRows <= cnt) {
#pragma unroll
      for (int u = 0; u < kRows; ++u) {
        s0 = s0 + T16::to_f32((uint16_t)(v[u] & 0xffff));
        s1 = s1 + T16::to_f32((uint16_t)(v[u] >> 16));
      }
    } else {
#pragma unroll
      for (int u = 0; u < kRows; ++u) {
        if (rr + u < cnt) {
          s0 = s0 + T16::to_f32((uint16_t)(v[u] & 0xffff));
          s1 = s1 + T16::to_f32((uint16_t)(v[u] >> 16));
        }
      }
    }
    rr += kRows;
    if (rr >= cnt) break;
    load(rr);
  }
  s0 = s0 / (float)cnt;
  s1 = s1 / (float)cnt;
  if (proj != nullptr) {
    *reinterpret_cast<float2*>(&mean[hw][2 * c]) = make_float2(s0, s1);
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    float p0 = 0.f, p1 = 0.f;
#pragma unroll 16
    for (int d = 0; d < kTile; ++d) {
      const float m = mean[hw][d];
      const float2 w = *reinterpret_cast<const float2*>(&pt[d][2 * c]);
      p0 = p0 + m * w.x;
      p1 = p1 + m * w.y;
    }
    s0 = p0;
    s1 = p1;
  }
  if (!on) return;
  if (t) {
    float* o = a.out[1] + (bh * kTile + 2 * c) * a.n[1] + j;
    o[0] = s0;
    o[a.n[1]] = s1;
  } else {
    *reinterpret_cast<float2*>(a.out[0] + jj * kTile + 2 * c) = make_float2(s0, s1);
  }
}

extern "C" int sla2h_pool_qk(const void* q, const void* k, int dtype, int B, int H, int64_t L,
                             int D, int bq, int bk, int Nk, const float* proj_q,
                             const float* proj_k, float* qpool, float* kpool_t, void* stream) {
  SLA2H_CHECK_ARG(q && k && qpool && kpool_t);
  SLA2H_CHECK_ARG(D == kTile && bq >= 1 && bq <= 4096 && bk == kTile);
  SLA2H_CHECK_ARG(dtype == SLA2H_DTYPE_F16 || dtype == SLA2H_DTYPE_BF16);
  SLA2H_CHECK_ARG(B > 0 && H > 0 && (int64_t)B * H <= 65535 && L > 0);
  SLA2H_CHECK_ARG(((uintptr_t)q | (uintptr_t)k) % 4 == 0 && (uintptr_t)qpool % 8 == 0);
  const int64_t nq = (L + bq - 1) / bq;
  SLA2H_CHECK_ARG(nq < (1ll << 31) && Nk > 0 && (int64_t)(Nk - 1) * bk < L);
  PoolPairArgs a = {};
  a.x[0] = static_cast<const uint16_t*>(q);
  a.x[1] = static_cast<const uint16_t*>(k);
  a.proj[0] = proj_q;
  a.proj[1] = proj_k;
  a.out[0] = qpool;
  a.out[1] = kpool_t;
  a.blk[0] = bq;
  a.blk[1] = bk;
  a.n[0] = (int)nq;
  a.n[1] = Nk;
  a.BH = B * H;
  a.L = L;
  const int64_t wq = ((int64_t)a.BH * nq + 7) / 8, wk = ((int64_t)a.BH * Nk + 7) / 8;
  SLA2H_CHECK_ARG(wq + wk < (1ll << 31));
  a.wg0 = (int)wq;
  const unsigned grid = (unsigned)(wq + wk);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == SLA2H_DTYPE_BF16)
    pool_pair_kernel<BF16><<<grid, 256, 0, st>>>(a);
  else
    pool_pair_kernel<F16><<<grid, 256, 0, st>>>(a);
  return (int)hipGetLastError();
}

extern "C" int sla2h_pool_blocks(const void* x, int dtype, int64_t BH, int64_t L, int D, int blk,
                                 const float* proj, int transposed, float* out, void* stream) {
  SLA2H_CHECK_ARG(x && out);
  SLA2H_CHECK_ARG(D == kTile && blk >= 1 && blk <= 4096);
  SLA2H_CHECK_ARG(dtype == SLA2H_DTYPE_F16 || dtype == SLA2H_DTYPE_BF16 || dtype == 2);
  SLA2H_CHECK_ARG(BH > 0 && BH <= 65535 && L > 0);
  const int64_t nblk = (L + blk - 1) / blk;
  SLA2H_CHECK_ARG(nblk < (1ll << 31));
  dim3 grid((unsigned)nblk, (unsigned)BH);
  hipStream_t st = static_cast<hipStream_t>(stream);
  auto X = static_cast<const uint16_t*>(x);
  if (dtype == 2)
    pool_blocks_kernel<F32In, float><<<grid, kTile, 0, st>>>(static_cast<const float*>(x), L, blk,
                                                            (int)nblk, proj, transposed, out);
  else if (dtype == SLA2H_DTYPE_BF16)
    pool_blocks_kernel<BF16, uint16_t><<<grid, kTile, 0, st>>>(X, L, blk, (int)nblk, proj,
                                                              transposed, out);
  else
    pool_blocks_kernel<F16, uint16_t><<<grid, kTile, 0, st>>>(X, L, blk, (int)nblk, proj,
                                                             transposed, out);
  return (int)hipGetLastError();
}

extern "C" int sla2h_version(void) { return 1; }

extern "C" const char* sla2h_error_string(int code) {
  return hipGetErrorString((hipError_t)code);
}

namespace sla2h {
// x[t] (B, L, H, 64) of one dtype (2: fp32) with strides[3 t ..] of (b, l, h), 16-byte
// aligned rows.  infer = 0: the training operands (fp16 rows, all of rows[t] given or
// rows NULL, truncating law, bq = 64); infer = 1: 16-bit x as it is, half away from
// zero, q in blocks of bq rows, every key block pooled (Np = Nb).
int launch_operands(const void* const* x, const int64_t* strides, int dtype, const int64_t* idx,
                    int B, int H, int64_t L, int Np, int bq, int infer, const float* proj_q,
                    const float* proj_k, void* const* rows, int8_t* const* xq, float* const* xs,
                    float* qpool, float* kpool_t, void* stream) {
  const int64_t es = dtype == 2 ? 4 : 2;
  SLA2H_CHECK_ARG(x && strides && qpool && kpool_t && B > 0 && H > 0 && L > 0);
  SLA2H_CHECK_ARG(dtype == SLA2H_DTYPE_F16 || dtype == SLA2H_DTYPE_BF16 || (dtype == 2 && !infer));
  SLA2H_CHECK_ARG(bq == 64 || (infer && (bq == 128 || bq == 256)));
  OperandArgs a = {};
  a.B = B;
  a.H = H;
  a.L = L;
  a.Nb = (int)((L + kTile - 1) / kTile);
  a.Np = Np;
  a.Mq = (int)((L + bq - 1) / bq);
  SLA2H_CHECK_ARG(Np > 0 && (infer ? Np == a.Nb : (int64_t)Np * kTile <= L));
  a.idx = idx;
  a.pool[0] = qpool;
  a.pool[1] = kpool_t;
  a.proj[0] = proj_q;
  a.proj[1] = proj_k;
  for (int t = 0; t < 3; ++t) {
    SLA2H_CHECK_ARG(x[t] && (uintptr_t)x[t] % 16 == 0);
    for (int d = 0; d < 3; ++d) SLA2H_CHECK_ARG(strides[3 * t + d] >= 0 && strides[3 * t + d] * es % 16 == 0);
    a.x[t] = x[t];
    a.sb[t] = strides[3 * t];
    a.st[t] = strides[3 * t + 1];
    a.sh[t] = strides[3 * t + 2];
    a.rows[t] = rows == nullptr ? nullptr : static_cast<uint16_t*>(rows[t]);
    SLA2H_CHECK_ARG(rows == nullptr || (rows[t] && (uintptr_t)rows[t] % 16 == 0));
    a.xq[t] = xq[t];
    a.xs[t] = xs[t];
  }
  const int64_t nwg = (int64_t)B * H * (a.Mq + 2 * (int64_t)a.Nb);
  SLA2H_CHECK_ARG(nwg < (1ll << 31));
  hipStream_t st = static_cast<hipStream_t>(stream);
  auto run = [&](auto kernel) { kernel<<<(unsigned)nwg, 256, 0, st>>>(a); };
  auto run_infer = [&](auto ts) {
    using TS = decltype(ts);
    bq == 64 ? run(operand_kernel<TS, uint16_t, TS, true, 1>)
             : (bq == 128 ? run(operand_kernel<TS, uint16_t, TS, true, 2>)
                          : run(operand_kernel<TS, uint16_t, TS, true, 4>));
  };
  if (infer)
    dtype == SLA2H_DTYPE_BF16 ? run_infer(BF16{}) : run_infer(F16{});
  else if (dtype == 2)
    run(operand_kernel<F32In, float, F16, false, 1>);
  else if (dtype == SLA2H_DTYPE_BF16)
    run(operand_kernel<BF16, uint16_t, F16, false, 1>);
  else
    run(operand_kernel<F16, uint16_t, F16, false, 1>);
  return (int)hipGetLastError();
}
}  // namespace sla2h

extern "C" int sla2h_quant_train(const void* q, const void* k, const void* v, int dtype, int B,
                                 int H, int64_t L, int D, int E, int8_t* q8, float* qs, int8_t* k8,
                                 float* ks, int8_t* v8f, float* vs, void* stream) {
  SLA2H_CHECK_ARG(q && k && v && q8 && qs && k8 && ks && v8f && vs);
  SLA2H_CHECK_ARG(D == kTile && E == kTile);
  SLA2H_CHECK_ARG(dtype == SLA2H_DTYPE_F16 || dtype == SLA2H_DTYPE_BF16);
  SLA2H_CHECK_ARG(B > 0 && H > 0 && 3 * B * H <= 65535 && L > 0);
  QuantTrainArgs a;
  a.x[0] = static_cast<const uint16_t*>(q);
  a.x[1] = static_cast<const uint16_t*>(k);
  a.x[2] = static_cast<const uint16_t*>(v);
  a.xq[0] = q8;
  a.xq[1] = k8;
  a.xq[2] = v8f;
  a.xs[0] = qs;
  a.xs[1] = ks;
  a.xs[2] = vs;
  a.BH = B * H;
  a.L = L;
  a.Nb = (int)((L + E - 1) / E);
  a.t0 = 0;
  dim3 grid(a.Nb, 3 * a.BH);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == SLA2H_DTYPE_BF16)
    quant_train_kernel<BF16><<<grid, 256, 0, st>>>(a);
  else
    quant_train_kernel<F16><<<grid, 256, 0, st>>>(a);
  return (int)hipGetLastError();
}

// The training kernel's truncating law (sla2h_quant_train) for one tensor in
// blocks of E = 32..256 rows: Q of the 1-D SLA2 INT8 training forward, whose
// query tiles are bq rows.
extern "C" int sla2h_quantize_trunc(const void* x, int dtype, int64_t BH, int64_t L, int D,
                                    int E, int8_t* xq, float* xs, void* stream) {
  SLA2H_CHECK_ARG(x && xq && xs);
  SLA2H_CHECK_ARG(D == kTile && (E == 32 || E == 64 || E == 128 || E == 256));
  SLA2H_CHECK_ARG(dtype == SLA2H_DTYPE_F16 || dtype == SLA2H_DTYPE_BF16);
  SLA2H_CHECK_ARG(BH > 0 && BH <= 65535 && L > 0);
  const int Nb = (int)((L + E - 1) / E);
  dim3 grid(Nb, (int)BH);
  hipStream_t st = static_cast<hipStream_t>(stream);
  auto X = static_cast<const uint16_t*>(x);
  auto go = [&](auto tag) {
    using T16 = decltype(tag);
    if (E == 32)
      quant_rows_kernel<T16, 32, true><<<grid, 256, 0, st>>>(X, L, Nb, xq, xs);
    else if (E == 64)
      quant_rows_kernel<T16, 64, true><<<grid, 256, 0, st>>>(X, L, Nb, xq, xs);
    else if (E == 128)
      quant_rows_kernel<T16, 128, true><<<grid, 256, 0, st>>>(X, L, Nb, xq, xs);
    else
      quant_rows_kernel<T16, 256, true><<<grid, 256, 0, st>>>(X, L, Nb, xq, xs);
  };
  if (dtype == SLA2H_DTYPE_BF16)
    go(BF16{});
  else
    go(F16{});
  return (int)hipGetLastError();
}

// V of the inference INT8 path: quantize_qkv's law (round half away, one
// scale per 64-row block) written in the INT8 MFMA fragment order of the
// sparse kernels (the layout of sla2h_quant_train's v8f).
extern "C" int sla2h_quantize_v8f(const void* v, int dtype, int64_t BH, int64_t L, int D, int E,
                                  int8_t* v8f, float* vs, void* stream) {
  SLA2H_CHECK_ARG(v && v8f && vs);
  SLA2H_CHECK_ARG(D == kTile && E == kTile);
  SLA2H_CHECK_ARG(dtype == SLA2H_DTYPE_F16 || dtype == SLA2H_DTYPE_BF16);
  SLA2H_CHECK_ARG(BH > 0 && BH <= 65535 && L > 0);
  QuantTrainArgs a = {};
  a.x[2] = static_cast<const uint16_t*>(v);
  a.xq[2] = v8f;
  a.xs[2] = vs;
  a.BH = (int)BH;
  a.L = L;
  a.Nb = (int)((L + E - 1) / E);
  a.t0 = 2;
  dim3 grid(a.Nb, (int)BH);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == SLA2H_DTYPE_BF16)
    quant_train_kernel<BF16, true><<<grid, 256, 0, st>>>(a);
  else
    quant_train_kernel<F16, true><<<grid, 256, 0, st>>>(a);
  return (int)hipGetLastError();
}

extern "C" int sla2h_quantize(const void* x, int dtype, int64_t BH, int64_t L, int D, int E,
                              int8_t* xq, float* xs, void* stream) {
  SLA2H_CHECK_ARG(x && xq && xs);
  SLA2H_CHECK_ARG(D == kTile && (E == 32 || E == 64 || E == 128 || E == 256));
  SLA2H_CHECK_ARG(dtype == SLA2H_DTYPE_F16 || dtype == SLA2H_DTYPE_BF16);
  SLA2H_CHECK_ARG(BH > 0 && BH <= 65535 && L > 0);
  if (BH * L * D == 0) return 0;
  if (E != kTile) {
    const int Nb = (int)((L + E - 1) / E);
    dim3 grid(Nb, (int)BH);
    hipStream_t st = static_cast<hipStream_t>(stream);
    auto X = static_cast<const uint16_t*>(x);
    auto go = [&](auto tag) {
      using T16 = decltype(tag);
      if (E == 32)
        quant_rows_kernel<T16, 32><<<grid, 256, 0, st>>>(X, L, Nb, xq, xs);
      else if (E == 128)
        quant_rows_kernel<T16, 128><<<grid, 256, 0, st>>>(X, L, Nb, xq, xs);
      else
        quant_rows_kernel<T16, 256><<<grid, 256, 0, st>>>(X, L, Nb, xq, xs);
    };
    if (dtype == SLA2H_DTYPE_BF16)
      go(BF16{});
    else
      go(F16{});
    return (int)hipGetLastError();
  }
  QuantPoolArgs a = {};
  a.x[0] = static_cast<const uint16_t*>(x);
  a.xq[0] = xq;
  a.xs[0] = xs;
  a.BH = (int)BH;
  a.L = L;
  a.Nb = (int)((L + E - 1) / E);
  return launch_quant_pool(a, 1, dtype, static_cast<hipStream_t>(stream));
}

extern "C" int sla2h_quant_pool_qk(const void* q, const void* k, int dtype, int B, int H,
                                   int64_t L, int D, int E, int Np, const float* proj_q,
                                   const float* proj_k, int8_t* q8, float* qs, int8_t* k8,
                                   float* ks, float* qpool, float* kpool_t, float* kbound,
                                   void* stream) {
  SLA2H_CHECK_ARG(q && k && q8 && qs && k8 && ks && qpool && kpool_t);
  SLA2H_CHECK_ARG(D == kTile && E == kTile);
  SLA2H_CHECK_ARG(dtype == SLA2H_DTYPE_F16 || dtype == SLA2H_DTYPE_BF16);
  SLA2H_CHECK_ARG(B > 0 && H > 0 && (int64_t)B * H * 2 <= 65535);
  SLA2H_CHECK_ARG(Np > 0 && (int64_t)Np * E <= L);
  const QuantPoolArgs a = quant_pool_qk_args(q, k, B * H, L, Np, proj_q, proj_k, q8, qs, k8, ks,
                                             qpool, kpool_t, kbound);
  return launch_quant_pool(a, 2, dtype, static_cast<hipStream_t>(stream));
}

extern "C" int sla2h_route_topk(const float* qpool, const float* kpool_t, int B, int H, int Mb,
                                int Np, int D, int T, float scale, int32_t* lut, uint8_t* mask,
                                void* stream) {
  SLA2H_CHECK_ARG(qpool && kpool_t && lut);
  SLA2H_CHECK_ARG(D == kTile);
  SLA2H_CHECK_ARG(B > 0 && H > 0 && B * H <= 65535 && Mb > 0);
  SLA2H_CHECK_ARG(Np > 0 && Np <= 4096 && T >= 1 && T <= Np);
  hipStream_t st = static_cast<hipStream_t>(stream);
  // The wave-wide selection up to 512 winners per row (456 rows of 456 tiles,
  // T = 114: 95.8 -> 15.6 us against the full sort of every row).  Ranking the
  // winners takes T^2 / 64 steps per wave, so with rows that the sort holds in
  // 512 slots it stops paying at T = 448 (110 against 112 us; 512: 131 against
  // 111), with longer rows it still does at 512 (Np = 600: 162 against 229 us).
  if (T <= 448 || (T <= 512 && Np > 512)) {
    // one query block per wave: enough waves to hide the load latency
    auto go = [&](auto nk) {
      constexpr int NK = decltype(nk)::value, BIG = NK == 1 ? 64 : 512;
      dim3 grid((Mb + 3) / 4, B * H);
      auto run = [&](auto kernel) {
        kernel<<<grid, 256, 0, st>>>(qpool, kpool_t, Mb, Np, T, scale, lut, mask);
      };
      if (T <= 64)
        Np % 4 == 0 ? run(route_select_kernel<NK, 64, true>) : run(route_select_kernel<NK, 64, false>);
      else
        Np % 4 == 0 ? run(route_select_kernel<NK, BIG, true>) : run(route_select_kernel<NK, BIG, false>);
    };
    if (Np <= 64)
      go(std::integral_constant<int, 1>{});
    else if (Np <= 128)
      go(std::integral_constant<int, 2>{});
    else if (Np <= 256)
      go(std::integral_constant<int, 4>{});
    else if (Np <= 512)
      go(std::integral_constant<int, 8>{});
    else if (Np <= 1024)
      go(std::integral_constant<int, 16>{});
    else if (Np <= 2048)
      go(std::integral_constant<int, 32>{});
    else
      go(std::integral_constant<int, 64>{});
    return (int)hipGetLastError();
  }
  int P2 = 1;
  while (P2 < Np) P2 <<= 1;
  if (P2 < 2) P2 = 2;
  const int rows = P2 <= 512 ? 8 : (P2 <= 1024 ? 4 : (P2 <= 2048 ? 2 : 1));
  const size_t shmem = (size_t)rows * P2 * 8 + (size_t)rows * kTile * 4 + (size_t)rows * P2;
  dim3 grid((Mb + rows - 1) / rows, B * H);
  switch (rows) {
    case 8: route_topk_kernel<8><<<grid, 256, shmem, st>>>(qpool, kpool_t, Mb, Np, T, scale, P2, lut, mask); break;
    case 4: route_topk_kernel<4><<<grid, 256, shmem, st>>>(qpool, kpool_t, Mb, Np, T, scale, P2, lut, mask); break;
    case 2: route_topk_kernel<2><<<grid, 256, shmem, st>>>(qpool, kpool_t, Mb, Np, T, scale, P2, lut, mask); break;
    default: route_topk_kernel<1><<<grid, 256, shmem, st>>>(qpool, kpool_t, Mb, Np, T, scale, P2, lut, mask); break;
  }
  return (int)hipGetLastError();
}
