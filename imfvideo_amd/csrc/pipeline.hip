// Whole calls of the op in one host entry each: the stages' launches in order
// on one stream, with their intermediates carved out of one caller-owned
// workspace.  The stages are the entry points of include/sla2h.h; what is
// added here are the small kernels between them that torch ran as chains of
// elementwise launches (alpha from its logits, the LUT with the prefix tail,
// the per-head maximum of lse, the alpha gradient).
//
// On small shapes the op is bound by the host: per stage a Python wrapper, its
// output allocations and its launch.  One call per pass leaves the launches.
#include "common.h"
#include "quant_pool.h"
#include "train_setup.h"

namespace sla2h {

namespace {

constexpr int kT = 64;
constexpr size_t kRecBytes = 33280;

// Consecutive 256-byte aligned pieces of one buffer; with base NULL only the
// size is added up.
struct Carve {
  unsigned char* base;
  size_t used = 0;
  template <typename T>
  T* take(size_t n) {
    T* p = base == nullptr ? nullptr : reinterpret_cast<T*>(base + used);
    used += (n * sizeof(T) + 255) / 256 * 256;
    return p;
  }
};

struct Dims {
  int B, H;
  int64_t L;
  int Nb;  // 64-row blocks
  int Np;  // routable blocks
  int bq, Mq, T, J;  // query blocks of bq rows; LUT columns, with the tail J
  size_t BH, rows, elems;
  Dims(int B_, int H_, int64_t L_, int Np_, int bq_, int T_)
      : B(B_), H(H_), L(L_), Nb((int)((L_ + kT - 1) / kT)), Np(Np_), bq(bq_),
        Mq((int)((L_ + bq_ - 1) / bq_)), T(T_), J(T_ + Nb - Np_), BH((size_t)B_ * H_),
        rows(BH * L_), elems(rows * kT) {}
};

bool dims_ok(int dtype, int B, int H, int64_t L, int Np, int bq, int T) {
  return (dtype == SLA2H_DTYPE_F16 || dtype == SLA2H_DTYPE_BF16) && B > 0 && H > 0 &&
         (int64_t)B * H <= 65535 && L > 0 && L * kT * 2 < (1ll << 31) && Np > 0 &&
         (int64_t)(Np - 1) * kT < L && (bq == 64 || bq == 128 || bq == 256) && T >= 1 && T <= Np;
}

constexpr int kScoreFormCols = 4;  // LUT columns up to which the linear branch is in score form
constexpr int64_t kEarlyStates = 2560;  // tiles: 40 MB of states

__global__ __launch_bounds__(256) void train_setup_kernel(TrainSetup a) {
  train_setup(a, (int64_t)blockIdx.x * 256 + threadIdx.x);
}

// Two small jobs between bwd_prep and the backward's products.
// Blocks y < BH: the selection bits seen from the key side, a transposition of
// the forward's complement masks (cbits word (kc, mq): bit j = tile 32 kc + j not
// routed by LUT row mq): sel[n][kcq] bit i = query block 32 kcq + i routes tile n,
// and its complement over the real blocks, word (kcq, n), for the mask GEMM.
// One thread per word; the 32 words it gathers are shared by the 32 tiles of a
// kc.  (Clearing, scattering the LUT's columns with atomics and complementing
// took three launches, 27 us at 16 heads x 468 blocks of 46 tiles.)
// Blocks y == BH: d_logit[h][m] = seg a (1 - a), seg summed over the batches and
// the 64-row blocks of query block m in order.
struct SelArgs {
  const uint32_t* cbits;
  uint32_t* sel;
  uint32_t* out;
  const float* segp;
  const float* alpha;
  float* d;
  int B, H, Nb, Mq, qshift, NC, MTf, MTb;  // 16 MT words per mask row, forward / backward
};
__global__ __launch_bounds__(256) void bwd_bits_kernel(SelArgs a) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  const int BH = a.B * a.H;
  if ((int)blockIdx.y == BH) {
    const int sub = 1 << a.qshift;
    for (int e = i; e < a.H * a.Mq; e += gridDim.x * 256) {
      const int h = e / a.Mq, m = e - h * a.Mq;
      float s = 0.f;
      for (int b = 0; b < a.B; ++b)
        for (int n = m * sub; n < min(a.Nb, (m + 1) * sub); ++n)
          s += a.segp[((int64_t)b * a.H + h) * a.Nb + n];
      const float al = a.alpha[e];
      a.d[e] = s * al * (1.0f - al);
    }
    return;
  }
  const int bh = blockIdx.y;
  const int mp = 16 * a.MTb;
  if (i >= a.NC * mp) return;
  const int kcq = i / mp, n = i - kcq * mp;
  uint32_t routed = 0u, real = 0u;
  if (n < a.Nb) {
    const uint32_t* src = a.cbits + ((int64_t)bh * a.NC + (n >> 5)) * (16 * a.MTf);
    const int left = a.Nb - 32 * kcq;
    real = left >= 32 ? 0xffffffffu : ((1u << left) - 1u);
#pragma unroll
    for (int j = 0; j < 32; ++j) {
      const int m = min(32 * kcq + j, a.Nb - 1);
      routed |= ((~src[m >> a.qshift] >> (n & 31)) & 1u) << j;
    }
    routed &= real;
    a.sel[((int64_t)bh * a.Nb + n) * a.NC + kcq] = routed;
  }
  a.out[(int64_t)bh * a.NC * mp + i] = ~routed & real;
}

struct JvpWs {
  int8_t *q8, *k8;
  float *qs, *ks, *kb, *Hb, *dHb, *zb, *dzb;
  uint16_t *vt, *kt;
  unsigned char *bits, *comp;
  int32_t* lut;
  size_t bytes;
  // int8: the cube op's quantised scores; else 16-bit scores, LUT with its tail
  JvpWs(void* p, const Dims& d, bool tan, bool int8) {
    Carve c{static_cast<unsigned char*>(p)};
    const size_t nb = d.BH * d.Nb, np = d.BH * d.Np;
    if (int8) {
      q8 = c.take<int8_t>(d.elems);
      k8 = c.take<int8_t>(d.elems);
      qs = c.take<float>(nb);
      ks = c.take<float>(nb);
      kb = c.take<float>(nb);
    }
    Hb = c.take<float>(np * kT * kT);
    zb = c.take<float>(np * kT);
    dHb = tan ? c.take<float>(np * kT * kT) : nullptr;
    dzb = tan ? c.take<float>(np * kT) : nullptr;
    vt = c.take<uint16_t>(nb * kT * kT * (tan ? 2 : 1));
    kt = tan ? c.take<uint16_t>(nb * kT * kT * 2) : nullptr;
    bits = c.take<unsigned char>(sla2h_complement_workspace_bytes(d.B, d.H, d.Mq, d.Np));
    comp = c.take<unsigned char>(d.BH * d.Mq * kRecBytes);
    lut = !int8 && d.J > d.T ? c.take<int32_t>(d.BH * d.Mq * d.J) : nullptr;
    bytes = c.used;
  }
};

// What the training forward keeps for the backward
struct Saved {
  uint16_t *o_s, *o_l, *qphi;
  float *lse, *den, *Hall, *alpha;
  unsigned char *comp, *bits;
  int32_t* lut;
  size_t bytes;
  Saved(void* p, const Dims& d) {
    Carve c{static_cast<unsigned char*>(p)};
    o_s = c.take<uint16_t>(d.elems);
    o_l = c.take<uint16_t>(d.elems);
    qphi = c.take<uint16_t>(d.elems);
    lse = c.take<float>(d.rows);
    den = c.take<float>(d.rows);
    Hall = c.take<float>(d.BH * kT * kT);
    alpha = c.take<float>((size_t)d.H * d.Mq);
    comp = c.take<unsigned char>(d.BH * d.Mq * kRecBytes);
    bits = c.take<unsigned char>(sla2h_complement_workspace_bytes(d.B, d.H, d.Mq, d.Nb));
    lut = c.take<int32_t>(d.BH * d.Mq * d.J);
    bytes = c.used;
  }
};

struct FwdWs {
  int8_t *q8, *k8, *v8f;
  float *qs, *ks, *vs, *Hb, *zb, *zall, *lse_max;
  uint16_t* vt;
  size_t bytes;
  FwdWs(void* p, const Dims& d, bool int8) {
    Carve c{static_cast<unsigned char*>(p)};
    const size_t nb = d.BH * d.Nb;
    if (int8) {
      q8 = c.take<int8_t>(d.elems);
      k8 = c.take<int8_t>(d.elems);
      v8f = c.take<int8_t>(nb * kT * kT);
      qs = c.take<float>(nb);
      ks = c.take<float>(nb);
      vs = c.take<float>(nb);
    }
    vt = int8 ? nullptr : c.take<uint16_t>(nb * kT * kT);
    Hb = c.take<float>(nb * kT * kT);
    zb = c.take<float>(nb * kT);
    zall = c.take<float>(d.BH * kT);
    lse_max = c.take<float>(d.H);
    bytes = c.used;
  }
};

struct BwdWs {
  uint16_t *dos, *g16;
  float *delta, *s, *segp, *P, *Pz;
  uint32_t* sel;
  unsigned char *bits, *comp;
  size_t bytes;
  BwdWs(void* p, const Dims& d) {
    Carve c{static_cast<unsigned char*>(p)};
    const size_t nb = d.BH * d.Nb;
    dos = c.take<uint16_t>(d.elems);
    g16 = c.take<uint16_t>(d.elems);
    delta = c.take<float>(d.rows);
    s = c.take<float>(d.rows);
    segp = c.take<float>(nb);
    P = c.take<float>(nb * kT * kT);
    Pz = c.take<float>(nb * kT);
    sel = c.take<uint32_t>(nb * ((d.Nb + 31) / 32));
    bits = c.take<unsigned char>(sla2h_complement_workspace_bytes(d.B, d.H, d.Nb, d.Nb));
    comp = c.take<unsigned char>(nb * kRecBytes);
    bytes = c.used;
  }
};

int log2_of(int x) { return x == 64 ? 0 : (x == 128 ? 1 : 2); }

}  // namespace

// attn_train.hip: the sparse forwards that also raise stats[h] (may be NULL) to
// the maximum of lse over the head's rows
int sparse_fwd_qat_stats(const void* q, const int8_t* q8, const float* qs, const int8_t* k8,
                         const float* ks, const int8_t* v8f, const float* vs, const int32_t* lut,
                         int dtype, int B, int H, int64_t L, int D, int E, int Np, int T,
                         float scale, void* o_s, float* lse, void* qphi, float* stats,
                         void* stream);
int sparse_fwd_int8_stats(const void* q, const int8_t* q8, const float* qs, int qblock,
                          const int8_t* k8, const float* ks, const int8_t* v8f, const float* vs,
                          const int32_t* lut, int dtype, int B, int H, int64_t L, int D, int bq,
                          int T, float scale, void* o_s, float* lse, void* qphi, float* stats,
                          void* stream);
int sparse_fwd_1d_stats(const void* q, const void* k, const void* vt, const int32_t* lut,
                        int dtype, int B, int H, int64_t L, int D, int bq, int bk, int T,
                        float scale, void* o_s, float* lse, void* qphi, float* stats,
                        void* stream);

// quant_route.hip: layout, INT8 operands and pooled tiles of q, k, v in one pass
int launch_operands(const void* const* x, const int64_t* strides, int dtype, const int64_t* idx,
                    int B, int H, int64_t L, int Np, int bq, int infer, const float* proj_q,
                    const float* proj_k, void* const* rows, int8_t* const* xq, float* const* xs,
                    float* qpool, float* kpool_t, void* stream);

// states.hip: sla2h_linear_states_qat without the sums over the tiles and the
// setup of a training forward, in one launch; sla2h_complement with the sums
int states_and_setup(const void* k, const void* v, int dtype, int B, int H, int64_t L, float* Hb,
                     float* zb, void* vt, const TrainSetup& setup, void* stream);
int complement_sums(const float* Hb, const float* dHb, const float* zb, const float* dzb,
                    const int32_t* lut, int B, int H, int Mb, int Np, int D, int T,
                    void* workspace, void* comp, float* Hall, float* zall, const float* lse_max,
                    float* stats, void* stream);

// states.hip: INT8 operands, pooled tiles and linear states of the cube op
int quant_states(const QuantPoolArgs& a, const void* k, const void* dk, const void* v,
                 const void* dv, int dtype, int Np, float* Hb, float* dHb, float* zb, float* dzb,
                 void* vt, void* kt, void* stream);

// states.hip: the backward's complement records from given masks (word (kcq, n))
int complement_gemm_bwd(const float* P, const float* Pz, const uint32_t* cbits, int BH, int Mb,
                        void* comp, void* stream);

// attn_bwd.hip: bwd_prep with each 64-row block's alpha segment sum stored to
// segp[(b H + h) Nb + block] instead of added into seg
int bwd_prep_segp(const void* dout, const void* o_s, const void* o_l, const float* den,
                  const void* qphi, const float* alpha, int alpha_stride, int dtype, int B, int H,
                  int64_t L, int E, void* dos, float* delta, void* g16, float* s, float* segp,
                  float* P, float* Pz, void* stream);

}  // namespace sla2h

using namespace sla2h;

#define SLA2H_TRY(call)              \
  do {                               \
    const int err_ = (call);         \
    if (err_ != 0) return err_;      \
  } while (0)

extern "C" size_t sla2h_cube_jvp_workspace_bytes(int B, int H, int64_t L, int Np, int T,
                                                 int tangent) {
  if (!dims_ok(0, B, H, L, Np, kT, T)) return 0;
  return JvpWs(nullptr, Dims(B, H, L, Np, kT, T), tangent != 0, true).bytes;
}

extern "C" int sla2h_cube_jvp_quant(const void* q, const void* k, const void* v, const void* dk,
                                    const void* dv, int dtype, int B, int H, int64_t L, int Np,
                                    int T, const float* proj_q, const float* proj_k,
                                    void* workspace, float* qpool, float* kpool_t, void* stream) {
  SLA2H_CHECK_ARG(q && k && v && workspace && qpool && kpool_t && dims_ok(dtype, B, H, L, Np, kT, T));
  SLA2H_CHECK_ARG((dk == nullptr) == (dv == nullptr));
  SLA2H_CHECK_ARG((int64_t)B * H * 2 <= 65535 && (int64_t)Np * kT <= L);
  const JvpWs w(workspace, Dims(B, H, L, Np, kT, T), dk != nullptr, true);
  const QuantPoolArgs a = quant_pool_qk_args(q, k, B * H, L, Np, proj_q, proj_k, w.q8, w.qs, w.k8,
                                             w.ks, qpool, kpool_t, w.kb);
  return quant_states(a, k, dk, v, dv, dtype, Np, w.Hb, w.dHb, w.zb, w.dzb, w.vt, w.kt, stream);
}

extern "C" int sla2h_cube_jvp_attn(const void* q, const void* dq, const float* alpha,
                                   int alpha_stride, const int32_t* lut, int dtype, int B, int H,
                                   int64_t L, int Np, int T, float scale, float eps_l,
                                   void* workspace, float* o, float* d_o, void* stream) {
  SLA2H_CHECK_ARG(workspace && lut && dims_ok(dtype, B, H, L, Np, kT, T));
  const bool tan = dq != nullptr;
  SLA2H_CHECK_ARG(!tan || d_o);
  const JvpWs w(workspace, Dims(B, H, L, Np, kT, T), tan, true);
  const int Mb = (int)((L + kT - 1) / kT);
  SLA2H_TRY(sla2h_complement(w.Hb, w.dHb, w.zb, w.dzb, lut, B, H, Mb, Np, kT, T, w.bits, w.comp,
                             stream));
  return sla2h_fwd_jvp(q, dq, w.kt, w.vt, w.q8, w.k8, w.qs, w.ks, w.kb, w.comp, alpha,
                       alpha_stride, lut, dtype, B, H, L, kT, kT, Np, T, scale, eps_l, 0, o, d_o,
                       stream);
}

extern "C" size_t sla2h_jvp16_workspace_bytes(int B, int H, int64_t L, int Np, int bq, int T) {
  if (!dims_ok(0, B, H, L, Np, bq, T)) return 0;
  return JvpWs(nullptr, Dims(B, H, L, Np, bq, T), true, false).bytes;
}

extern "C" int sla2h_jvp16(const void* q, const void* k, const void* v, const void* dq,
                           const void* dk, const void* dv, const float* alpha, int alpha_stride,
                           const int32_t* lut, int dtype, int B, int H, int64_t L, int Np, int bq,
                           int T, float scale, float eps_l, void* workspace, float* o, float* d_o,
                           void* stream) {
  SLA2H_CHECK_ARG(workspace && lut && dq && dk && dv && dims_ok(dtype, B, H, L, Np, bq, T));
  const Dims d(B, H, L, Np, bq, T);
  const JvpWs w(workspace, d, true, false);
  hipStream_t st = static_cast<hipStream_t>(stream);
  SLA2H_TRY(sla2h_linear_states(k, dk, v, dv, dtype, B, H, L, kT, kT, Np, w.Hb, w.dHb, w.zb,
                                w.dzb, nullptr, nullptr, nullptr, nullptr, w.vt, w.kt, stream));
  SLA2H_TRY(sla2h_complement(w.Hb, w.dHb, w.zb, w.dzb, lut, B, H, d.Mq, Np, kT, T, w.bits, w.comp,
                             stream));
  if (d.J > T) {
    const int64_t nl = (int64_t)d.BH * d.Mq * d.J;
    train_setup_kernel<<<(unsigned)((nl + 255) / 256), 256, 0, st>>>(
        TrainSetup{nullptr, 0, nullptr, lut, nl, T, d.J, Np, w.lut, nullptr, 0});
    SLA2H_TRY((int)hipGetLastError());
    lut = w.lut;
  }
  return sla2h_fwd_jvp_1d(q, dq, w.kt, w.vt, w.comp, alpha, alpha_stride, lut, dtype, B, H, L, kT,
                          bq, kT, d.J, scale, eps_l, o, d_o, stream);
}

extern "C" size_t sla2h_train_saved_bytes(int B, int H, int64_t L, int Np, int bq, int T) {
  if (!dims_ok(0, B, H, L, Np, bq, T)) return 0;
  return Saved(nullptr, Dims(B, H, L, Np, bq, T)).bytes;
}

extern "C" size_t sla2h_train_fwd_workspace_bytes(int B, int H, int64_t L, int Np, int bq, int T,
                                                  int int8) {
  if (!dims_ok(0, B, H, L, Np, bq, T)) return 0;
  return FwdWs(nullptr, Dims(B, H, L, Np, bq, T), int8 != 0).bytes;
}

extern "C" int sla2h_train_in(const void* const* x, const int64_t* strides, int dtype,
                              const int64_t* idx, int B, int H, int64_t L, int Np,
                              const float* proj_q, const float* proj_k, void* const* rows,
                              void* workspace, float* qpool, float* kpool_t, void* stream) {
  SLA2H_CHECK_ARG(workspace && dims_ok(0, B, H, L, Np, kT, 1));
  const FwdWs w(workspace, Dims(B, H, L, Np, kT, 1), true);
  int8_t* const xq[3] = {w.q8, w.k8, w.v8f};
  float* const xs[3] = {w.qs, w.ks, w.vs};
  return launch_operands(x, strides, dtype, idx, B, H, L, Np, kT, 0, proj_q, proj_k, rows, xq, xs,
                         qpool, kpool_t, stream);
}

extern "C" int sla2h_train_fwd(const void* q, const void* k, const void* v,
                               const float* alpha_logit, const int32_t* lut, int dtype, int B,
                               int H, int64_t L, int Np, int bq, int T, int int8, int quantised,
                               float scale, float eps_l, void* saved, void* workspace, void* o, float* stats,
                               void* stream) {
  SLA2H_CHECK_ARG(q && k && v && alpha_logit && lut && saved && workspace && o);
  SLA2H_CHECK_ARG(dims_ok(dtype, B, H, L, Np, bq, T));
  const Dims d(B, H, L, Np, bq, T);
  SLA2H_CHECK_ARG(bq == kT || Np == d.Nb);  // the prefix tail goes with 64-row query blocks
  const Saved s(saved, d);
  const FwdWs w(workspace, d, int8 != 0);
  const int64_t nl = (int64_t)d.BH * d.Mq * d.J;
  const int na = H * d.Mq;
  // stats, alpha and the whole LUT rows, beside the states (w.vt: the 16-bit sparse
  // kernel's).  Large INT8 calls keep the states behind the sparse kernel, next to
  // the complement that reads them while they are still in the caches, and the
  // setup in a launch of its own.  States behind -> before the sparse kernel, us a
  // forward: 256 tiles 37.3 -> 34.9, 1040 83.8 -> 82.8, 2048 161.8 -> 159.6; 3200
  // 302.6 -> 307.3, 7488 722 -> 735.
  // The sparse kernels raise the maxima of lse in the workspace and the complement
  // copies them out when they are whole: the caller's buffer only ever receives one
  // call's values, also where calls of several streams share it.
  float* const lse_max = stats != nullptr ? w.lse_max : nullptr;
  const TrainSetup setup{alpha_logit, na, s.alpha, lut, nl, T, d.J, Np, s.lut, lse_max, H};
  const bool late = int8 && (int64_t)d.BH * d.Nb > kEarlyStates;
  if (late) {
    const int64_t n = nl > na ? nl : na;
    train_setup_kernel<<<(unsigned)((n + 255) / 256), 256, 0, static_cast<hipStream_t>(stream)>>>(
        setup);
    SLA2H_TRY((int)hipGetLastError());
  } else {
    SLA2H_TRY(states_and_setup(k, v, dtype, B, H, L, w.Hb, w.zb, int8 ? nullptr : w.vt, setup,
                               stream));
  }
  if (int8) {
    if (!quantised)
      SLA2H_TRY(sla2h_quant_train(q, k, v, dtype, B, H, L, kT, kT, w.q8, w.qs, w.k8, w.ks, w.v8f,
                                  w.vs, stream));
    if (bq == kT && (int64_t)Np * kT <= L) {
      SLA2H_TRY(sparse_fwd_qat_stats(q, w.q8, w.qs, w.k8, w.ks, w.v8f, w.vs, lut, dtype, B, H, L,
                                     kT, kT, Np, T, scale, s.o_s, s.lse, s.qphi, lse_max, stream));
    } else {  // query blocks over 64 rows, or a routable last block that is partial
      SLA2H_TRY(sla2h_quantize_trunc(q, dtype, (int64_t)d.BH, L, kT, bq, w.q8, w.qs, stream));
      SLA2H_TRY(sparse_fwd_int8_stats(q, w.q8, w.qs, bq, w.k8, w.ks, w.v8f, w.vs, lut, dtype, B,
                                      H, L, kT, bq, T, scale, s.o_s, s.lse, s.qphi, lse_max,
                                      stream));
    }
    if (late)
      SLA2H_TRY(states_and_setup(k, v, dtype, B, H, L, w.Hb, w.zb, nullptr, TrainSetup{}, stream));
  } else {
    SLA2H_TRY(sparse_fwd_1d_stats(q, k, w.vt, s.lut, dtype, B, H, L, kT, bq, kT, d.J, scale,
                                  s.o_s, s.lse, s.qphi, lse_max, stream));
  }
  // (zall: the score form's)
  SLA2H_TRY(complement_sums(w.Hb, nullptr, w.zb, nullptr, s.lut, B, H, d.Mq, d.Nb, kT, d.J, s.bits,
                            s.comp, s.Hall, d.J <= kScoreFormCols ? w.zall : nullptr, lse_max,
                            stats, stream));
  // the reference's linear branch: score form for few LUT columns, else state form
  if (d.J <= kScoreFormCols)
    SLA2H_TRY(sla2h_linear_mix_score(s.qphi, k, v, s.Hall, w.zall, s.lut, d.J, s.o_s, s.alpha,
                                     d.Mq, dtype, B, H, L, kT, bq, eps_l, o, s.o_l, s.den,
                                     stream));
  else
    SLA2H_TRY(sla2h_linear_mix_qat(s.qphi, s.comp, s.Hall, s.o_s, s.alpha, d.Mq, dtype, B, H, L,
                                   kT, bq, eps_l, o, s.o_l, s.den, stream));
  return 0;
}

extern "C" size_t sla2h_train_bwd_workspace_bytes(int B, int H, int64_t L, int Np, int bq, int T) {
  if (!dims_ok(0, B, H, L, Np, bq, T)) return 0;
  return BwdWs(nullptr, Dims(B, H, L, Np, bq, T)).bytes;
}

extern "C" int sla2h_train_bwd(const void* q, const void* k, const void* v, const void* dout,
                               const void* saved, int dtype, int B, int H, int64_t L, int Np,
                               int bq, int T, float scale, void* workspace, void* dq, void* dk,
                               void* dv, float* d_logit, void* stream) {
  SLA2H_CHECK_ARG(q && k && v && dout && saved && workspace && dq && dk && dv && d_logit);
  SLA2H_CHECK_ARG(dims_ok(dtype, B, H, L, Np, bq, T));
  const Dims d(B, H, L, Np, bq, T);
  const Saved s(const_cast<void*>(saved), d);
  const BwdWs w(workspace, d);
  hipStream_t st = static_cast<hipStream_t>(stream);
  SLA2H_TRY(bwd_prep_segp(dout, s.o_s, s.o_l, s.den, s.qphi, s.alpha, d.Mq, dtype, B, H, L, bq,
                          w.dos, w.delta, w.g16, w.s, w.segp, w.P, w.Pz, stream));
  SelArgs b;
  b.cbits = reinterpret_cast<const uint32_t*>(s.bits);
  b.sel = w.sel;
  b.out = reinterpret_cast<uint32_t*>(w.bits);
  b.segp = w.segp;
  b.alpha = s.alpha;
  b.d = d_logit;
  b.B = B;
  b.H = H;
  b.Nb = d.Nb;
  b.Mq = d.Mq;
  b.qshift = log2_of(bq);
  b.NC = (d.Nb + 31) / 32;
  b.MTf = (d.Mq + 15) / 16;
  b.MTb = (d.Nb + 15) / 16;
  bwd_bits_kernel<<<dim3((b.NC * 16 * b.MTb + 255) / 256, (unsigned)d.BH + 1), 256, 0, st>>>(b);
  SLA2H_TRY((int)hipGetLastError());
  SLA2H_TRY(complement_gemm_bwd(w.P, w.Pz, b.out, (int)d.BH, d.Nb, w.comp, stream));
  SLA2H_TRY(sla2h_bwd_dq(q, k, v, w.dos, s.lse, w.delta, w.g16, w.s, s.comp, s.Hall, s.qphi,
                         s.lut, dtype, B, H, L, kT, bq, d.J, scale, dq, stream));
  return sla2h_bwd_dkdv(q, k, v, w.dos, s.lse, w.delta, w.sel, w.comp, dtype, B, H, L, kT, kT,
                        scale, dk, dv, stream);
}

namespace sla2h {
namespace {
struct InferWs {
  int8_t *q8, *k8, *v8f;
  float *qs, *ks, *vs, *Hb, *zb, *lse;
  uint16_t *vt, *o_s, *qphi;
  unsigned char *bits, *comp;
  size_t bytes;
  InferWs(void* p, const Dims& d, bool int8) {
    Carve c{static_cast<unsigned char*>(p)};
    const size_t nb = d.BH * d.Nb;
    if (int8) {
      q8 = c.take<int8_t>(d.elems);
      k8 = c.take<int8_t>(d.elems);
      v8f = c.take<int8_t>(nb * kT * kT);
      qs = c.take<float>(nb * 2);  // scales per 32 rows or more
      ks = c.take<float>(nb);
      vs = c.take<float>(nb);
    }
    vt = int8 ? nullptr : c.take<uint16_t>(nb * kT * kT);
    Hb = c.take<float>(nb * kT * kT);
    zb = c.take<float>(nb * kT);
    lse = c.take<float>(d.rows);
    o_s = c.take<uint16_t>(d.elems);
    qphi = c.take<uint16_t>(d.elems);
    bits = c.take<unsigned char>(sla2h_complement_workspace_bytes(d.B, d.H, d.Mq, d.Nb));
    comp = c.take<unsigned char>(d.BH * d.Mq * kRecBytes);
    bytes = c.used;
  }
};
}  // namespace
}  // namespace sla2h

extern "C" size_t sla2h_sla2_infer_workspace_bytes(int B, int H, int64_t L, int bq, int T,
                                                   int int8) {
  const int Nb = (int)((L + kT - 1) / kT);
  if (!dims_ok(0, B, H, L, Nb, bq, T)) return 0;
  return InferWs(nullptr, Dims(B, H, L, Nb, bq, T), int8 != 0).bytes;
}

extern "C" int sla2h_sla2_infer_in(const void* q, const void* k, const void* v, int dtype, int B,
                                   int H, int64_t L, int bq, const float* proj_q,
                                   const float* proj_k, void* workspace, float* qpool,
                                   float* kpool_t, void* stream) {
  SLA2H_CHECK_ARG(workspace && L > 0);
  const int Nb = (int)((L + kT - 1) / kT);
  SLA2H_CHECK_ARG(dims_ok(dtype, B, H, L, Nb, bq, 1));
  const InferWs w(workspace, Dims(B, H, L, Nb, bq, 1), true);
  const void* const x[3] = {q, k, v};
  const int64_t s[3] = {H * L * kT, kT, L * kT};
  const int64_t strides[9] = {s[0], s[1], s[2], s[0], s[1], s[2], s[0], s[1], s[2]};
  int8_t* const xq[3] = {w.q8, w.k8, w.v8f};
  float* const xs[3] = {w.qs, w.ks, w.vs};
  return launch_operands(x, strides, dtype, nullptr, B, H, L, Nb, bq, 1, proj_q, proj_k, nullptr,
                         xq, xs, qpool, kpool_t, stream);
}

extern "C" int sla2h_sla2_infer(const void* q, const void* k, const void* v, const float* alpha,
                                int alpha_stride, const int32_t* lut, int dtype, int B, int H,
                                int64_t L, int bq, int T, int int8, int qblock, int quantised,
                                float scale, float eps_l, void* workspace, void* o, void* stream) {
  SLA2H_CHECK_ARG(q && k && v && alpha && lut && workspace && o && L > 0);
  const int Nb = (int)((L + kT - 1) / kT);
  SLA2H_CHECK_ARG(dims_ok(dtype, B, H, L, Nb, bq, T) && (!quantised || (int8 && qblock == bq)));
  const Dims d(B, H, L, Nb, bq, T);
  const InferWs w(workspace, d, int8 != 0);
  SLA2H_TRY(sla2h_hblocks_states(k, v, dtype, B, H, L, kT, kT, w.Hb, w.zb, nullptr, nullptr, w.vt,
                                 stream));
  if (int8) {
    const int64_t bh = (int64_t)d.BH;
    if (!quantised) {
      SLA2H_TRY(sla2h_quantize(q, dtype, bh, L, kT, qblock, w.q8, w.qs, stream));
      SLA2H_TRY(sla2h_quantize(k, dtype, bh, L, kT, kT, w.k8, w.ks, stream));
      SLA2H_TRY(sla2h_quantize_v8f(v, dtype, bh, L, kT, kT, w.v8f, w.vs, stream));
    }
    SLA2H_TRY(sla2h_sparse_fwd_int8(q, w.q8, w.qs, qblock, w.k8, w.ks, w.v8f, w.vs, lut, dtype, B,
                                    H, L, kT, bq, T, scale, w.o_s, w.lse, w.qphi, stream));
  } else {
    SLA2H_TRY(sla2h_sparse_fwd_1d(q, k, w.vt, lut, dtype, B, H, L, kT, bq, kT, T, scale, w.o_s,
                                  w.lse, w.qphi, stream));
  }
  SLA2H_TRY(sla2h_complement(w.Hb, nullptr, w.zb, nullptr, lut, B, H, d.Mq, Nb, kT, T, w.bits,
                             w.comp, stream));
  return sla2h_lin_fwd3(w.qphi, w.comp, w.o_s, alpha, alpha_stride, dtype, B, H, L, kT, bq, eps_l,
                        o, stream);
}
