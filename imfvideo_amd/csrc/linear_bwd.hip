// Weight gradient of a linear layer, dW = dY^T X over the token rows, gfx950.
//
// Reference semantics: torch autograd of the nn.Linear layers of
// models/imf_dit_video.py:174-187, 422-467 (their fp32 weights' gradients
// under a 16-bit autocast).
//
// The product contracts over the rows (tokens, tens of thousands) and its
// output is small (a weight: 160 x 512 ... 2048 x 512), so one workgroup per
// output tile leaves most of the 256 CUs idle.  The rows are split into ranges
// as well: grid = output tiles x ranges, fp32 partial tiles, then one pass
// that adds the ranges in order (no atomics: the result does not depend on
// the dispatch order).
#include "common.h"

namespace sla2h {

namespace {

constexpr int kWT = 128;             // output tile (rows of dY columns x X columns)
constexpr int kWK = 32;              // token rows per stage: one K = 32 MFMA step
constexpr int kWStages = 4;          // LDS slots; three stages of loads in flight
constexpr int kWHalf = kWK * kWT * 2;  // bytes of one operand's stage: 32 rows x 256 B
constexpr int kWStage = 2 * kWHalf;
// s_waitcnt vmcnt(8): everything but the last two stages' loads (4 per wave each)
constexpr int kWaitVm8 = 0x0F78;

struct WgradArgs {
  const uint16_t* dy;
  const uint16_t* x;
  float* out;  // partial tiles [split][M][N] (the weight gradient itself with one range)
  int64_t ldy, ldx;
  int rows, M, N;
  int tn;        // column tiles of X
  int tiles;     // output tiles
  int per_split;  // rows of a range, a multiple of kWK
  int nwork, per_xcd;
};

// Four fragments (sub-tiles at LDS byte addresses a[t] + slot, K halves 4096
// bytes apart) read transposed, complete on return.  The compiler makes every
// LDS read that it sees wait for all copies into LDS still in flight
// (vmcnt(0)), which would undo the prefetch; reads in an asm block that waits
// for itself depend on the explicit vmcnt count of the loop alone.
__device__ inline void read_frags(const uint32_t (&a)[4], uint32_t slot, u32x4 (&f)[4]) {
  u32x2 q[8];
  asm volatile(
      "ds_read_b64_tr_b16 %0, %8\n\t"
      "ds_read_b64_tr_b16 %1, %8 offset:4096\n\t"
      "ds_read_b64_tr_b16 %2, %9\n\t"
      "ds_read_b64_tr_b16 %3, %9 offset:4096\n\t"
      "ds_read_b64_tr_b16 %4, %10\n\t"
      "ds_read_b64_tr_b16 %5, %10 offset:4096\n\t"
      "ds_read_b64_tr_b16 %6, %11\n\t"
      "ds_read_b64_tr_b16 %7, %11 offset:4096\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(q[0]), "=&v"(q[1]), "=&v"(q[2]), "=&v"(q[3]), "=&v"(q[4]), "=&v"(q[5]),
        "=&v"(q[6]), "=&v"(q[7])
      : "v"(a[0] + slot), "v"(a[1] + slot), "v"(a[2] + slot), "v"(a[3] + slot)
      : "memory");
#pragma unroll
  for (int t = 0; t < 4; ++t) f[t] = u32x4{q[2 * t].x, q[2 * t].y, q[2 * t + 1].x, q[2 * t + 1].y};
}
__device__ inline void dma16(__amdgpu_buffer_rsrc_t rs, void* dst, int voff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)dst, 16,
                                           voff, 0, 0, 0);
}

// Workgroup = one 128 x 128 tile of dW over one range of rows; wave (wm, wn)
// owns 64 x 64 of it.  Both operands are row-major in the contracted index, so
// each stage's 32 rows x 128 columns of dY and of X go to LDS as they are
// (buffer loads straight into LDS, three stages ahead, one barrier per stage)
// and the MFMA fragments come out transposed (ds_read_b64_tr_b16: a group of
// 16 lanes reads a 4 row x 16 column block per instruction).  A row's 32-byte
// column chunk c sits at chunk c ^ (row & 7), so the 16 rows of one fragment
// read cover all banks evenly.
template <typename T16>
__global__ __launch_bounds__(256, 2) void wgrad_kernel(WgradArgs a) {
  __shared__ __align__(16) unsigned char lds[kWStages * kWStage];
  const int logical = (blockIdx.x & 7) * a.per_xcd + (blockIdx.x >> 3);
  if (logical >= a.nwork) return;
  // ranges outermost: the workgroups of an XCD share a range's rows in its L2
  const int sp = __builtin_amdgcn_readfirstlane(logical / a.tiles);
  const int tile = __builtin_amdgcn_readfirstlane(logical - sp * a.tiles);
  const int m0 = (tile / a.tn) * kWT, n0 = (tile % a.tn) * kWT;
  const int k0 = sp * a.per_split;
  const int k1 = min(a.rows, k0 + a.per_split);
  const int nst = (k1 - k0 + kWK - 1) / kWK;
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l = tid & 63, r = l & 15, g = l >> 4;
  const int wm = w >> 1, wn = w & 1;

  // Rows past the last one read as zero (range check), which ends the last
  // range; a column past M or N reads the next row's (or zero) and only ever
  // feeds an output that is not stored.
  const auto ry = make_rsrc(a.dy, ((int64_t)(a.rows - 1) * a.ldy + a.M) * 2);
  const auto rx = make_rsrc(a.x, ((int64_t)(a.rows - 1) * a.ldx + a.N) * 2);
  const int ldy2 = (int)a.ldy * 2, ldx2 = (int)a.ldx * 2;
  // lane l of a load covers row 4 slot + l / 16, LDS chunk (l % 16) / 2
  const int lrow = 4 * w + (l >> 4);
  const int col = ((((l & 15) >> 1) ^ (lrow & 7)) << 5) + (l & 1) * 16;
  int oy = (k0 + lrow) * ldy2 + m0 * 2 + col;
  int ox = (k0 + lrow) * ldx2 + n0 * 2 + col;
  auto load_stage = [&](int slot) {
    unsigned char* p = lds + slot * kWStage + w * 1024;
    dma16(ry, p, oy);
    dma16(ry, p + 4096, oy + 16 * ldy2);
    dma16(rx, p + kWHalf, ox);
    dma16(rx, p + kWHalf + 4096, ox + 16 * ldx2);
    oy += kWK * ldy2;
    ox += kWK * ldx2;
  };

  // fragment reads: row 4 g + r / 4 (and + 16), chunk = 16-column sub-tile
  const int rho = 4 * g + (r >> 2);
  const uint32_t lbase = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds;
  uint32_t fy[4], fx[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    fy[t] = lbase + rho * 256 + (((4 * wm + t) ^ (rho & 7)) << 5) + (r & 3) * 8;
    fx[t] = lbase + kWHalf + rho * 256 + (((4 * wn + t) ^ (rho & 7)) << 5) + (r & 3) * 8;
  }

  f32x4 acc[4][4];  // [n sub-tile][m sub-tile]: lane holds dW[m = r][n = 4 g + i]
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Stage s lives in slot s % 4; the stages loaded past the last one hold zeros
  // or the next range's rows and are never used.
  load_stage(0);
  load_stage(1);
  load_stage(2);
  for (int s = 0; s < nst; ++s) {
    __builtin_amdgcn_s_waitcnt(kWaitVm8);  // this wave's part of stage s has landed
    __builtin_amdgcn_s_barrier();          // everyone's has, and stage s - 1 is read
    load_stage((s + 3) & 3);
    u32x4 fm[4], fn[4];
    const uint32_t slot = (s & 3) * kWStage;
    read_frags(fy, slot, fm);
    read_frags(fx, slot, fn);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = mfma_16x16x32<T16>(fn[i], fm[j], acc[i][j]);
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // no load into this workgroup's LDS outlives it

  float* out = a.out + (int64_t)sp * a.M * a.N;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int m = m0 + 64 * wm + 16 * j + r;
    if (m >= a.M) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = n0 + 64 * wn + 16 * i + 4 * g;
      if (n < a.N) *reinterpret_cast<f32x4*>(out + (int64_t)m * a.N + n) = acc[i][j];
    }
  }
}

// dW = sum over the ranges in order, four elements per thread
__global__ __launch_bounds__(256) void wgrad_sum_kernel(const f32x4* __restrict__ part, int splits,
                                                       int64_t n4, f32x4* __restrict__ dw) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  f32x4 s = part[i];
#pragma unroll 8
  for (int j = 1; j < splits; ++j) s += part[j * n4 + i];
  dw[i] = s;
}

// Ranges of rows: enough workgroups for two on each of the 256 CUs, and at
// least eight stages per range.
int wgrad_splits(int64_t rows, int M, int N) {
  const int64_t tiles = (int64_t)((M + kWT - 1) / kWT) * ((N + kWT - 1) / kWT);
  int64_t s = 512 / tiles;
  const int64_t most = rows / (8 * kWK);
  s = s < most ? s : most;
  return s < 1 ? 1 : (int)s;
}

}  // namespace

}  // namespace sla2h

using namespace sla2h;

extern "C" size_t sla2h_linear_wgrad_workspace_bytes(int64_t rows, int M, int N) {
  if (rows <= 0 || M <= 0 || N <= 0) return 0;
  const int s = wgrad_splits(rows, M, N);
  return s > 1 ? (size_t)s * M * N * 4 : 0;
}

extern "C" int sla2h_linear_wgrad(const void* dy, int64_t ldy, const void* x, int64_t ldx,
                                  int dtype, int64_t rows, int M, int N, void* workspace,
                                  float* dw, void* stream) {
  SLA2H_CHECK_ARG(dy && x && dw);
  SLA2H_CHECK_ARG(dtype == SLA2H_DTYPE_F16 || dtype == SLA2H_DTYPE_BF16);
  SLA2H_CHECK_ARG(rows > 0 && M > 0 && N > 0 && M % 8 == 0 && N % 8 == 0);
  SLA2H_CHECK_ARG(ldy >= M && ldx >= N && ldy % 8 == 0 && ldx % 8 == 0);
  SLA2H_CHECK_ARG(((uintptr_t)dy | (uintptr_t)x | (uintptr_t)dw | (uintptr_t)workspace) % 16 == 0);
  // 32-bit byte offsets, three stages and a tile of columns past the end included
  const int64_t pad = 4 * kWK + 16;
  SLA2H_CHECK_ARG((rows + pad) * ldy * 2 + 2 * kWT < ((int64_t)1 << 31) &&
                  (rows + pad) * ldx * 2 + 2 * kWT < ((int64_t)1 << 31));
  const int splits = wgrad_splits(rows, M, N);
  SLA2H_CHECK_ARG(splits == 1 || workspace);
  const int tm = (M + kWT - 1) / kWT, tn = (N + kWT - 1) / kWT;
  const int64_t per = ((rows + splits - 1) / splits + kWK - 1) / kWK * kWK;
  const int used = (int)((rows + per - 1) / per);  // ranges that hold a row
  const int64_t nwork = (int64_t)tm * tn * used;
  SLA2H_CHECK_ARG(nwork < ((int64_t)1 << 28));
  hipStream_t st = static_cast<hipStream_t>(stream);
  WgradArgs a;
  a.dy = static_cast<const uint16_t*>(dy);
  a.x = static_cast<const uint16_t*>(x);
  a.out = used > 1 ? static_cast<float*>(workspace) : dw;
  a.ldy = ldy;
  a.ldx = ldx;
  a.rows = (int)rows;
  a.M = M;
  a.N = N;
  a.tn = tn;
  a.tiles = tm * tn;
  a.per_split = (int)per;
  a.nwork = (int)nwork;
  a.per_xcd = (int)((nwork + 7) / 8);
  if (dtype == SLA2H_DTYPE_BF16)
    wgrad_kernel<BF16><<<8 * a.per_xcd, 256, 0, st>>>(a);
  else
    wgrad_kernel<F16><<<8 * a.per_xcd, 256, 0, st>>>(a);
  int err = (int)hipGetLastError();
  if (err || used == 1) return err;
  const int64_t n4 = (int64_t)M * N / 4;
  wgrad_sum_kernel<<<(unsigned)((n4 + 255) / 256), 256, 0, st>>>(
      static_cast<const f32x4*>(workspace), used, n4, reinterpret_cast<f32x4*>(dw));
  return (int)hipGetLastError();
}
