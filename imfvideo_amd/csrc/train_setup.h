// The small per-call values of a training forward: alpha = sigmoid(logit); LUT rows
// with the tail blocks Np .. Nb - 1 appended; stats = -inf.  Each part may be
// absent (n = 0 or NULL).
#pragma once

#include "common.h"

namespace sla2h {

struct TrainSetup {
  const float* logit;
  int na;
  float* alpha;
  const int32_t* lut;
  int64_t nl;  // entries of lut_aug
  int T, J, Np;
  int32_t* lut_aug;
  float* stats;
  int H;
};

__device__ inline void train_setup(const TrainSetup& a, int64_t i) {
  if (i < a.na) a.alpha[i] = 1.0f / (1.0f + expf(-a.logit[i]));
  if (a.stats != nullptr && i < a.H) a.stats[i] = -INFINITY;
  if (i < a.nl) {
    const int64_t row = i / a.J;
    const int j = (int)(i - row * a.J);
    a.lut_aug[i] = j < a.T ? a.lut[row * a.T + j] : a.Np + (j - a.T);
  }
}

}  // namespace sla2h
