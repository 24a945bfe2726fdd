// Library-internal entries of the small-matrix Muon path (muon_small.hip), used by
// the phases of muon.hip.
#pragma once

#include <stdint.h>

#include "common.h"

namespace morph {

constexpr int kSmallMaxMats = 64;

// Whether an operand [m, n] (m <= n) takes the small path: X, padded to 32, and A
// fit one CU's LDS, and m is at most kSmallMaxRows.
constexpr int kSmallMaxRows = 128;
constexpr int kSmallLds = 160 * 1024;
inline bool small_fits(int64_t m, int64_t n) {
  if (m > kSmallMaxRows) return false;
  const int64_t mp = (m + 31) / 32 * 32, np = (n + 31) / 32 * 32;
  return mp * (np + 8) + mp * (mp + 8) <= kSmallLds / 2;
}

// The matrices of a batch, stored [m, n], or [n, m] when `tall` (the operand X [m, n]
// is then the transpose).  X0 of matrix i: bf16, in the stored layout, rows of ld
// elements (the stored row length rounded up to 8), at x0 + i * stride.  prepare leaves
// the orientations in `form` (the chain may run without the matrices' descriptors).
struct SmallBatch {
  const float* grad[kSmallMaxMats];
  const float* mom[kSmallMaxMats];
  float* mom_out[kSmallMaxMats];
  float* param[kSmallMaxMats];
  uint64_t tall;    // bit i; prepare only
  uint32_t* form;   // [count]: 1 when tall
  uint16_t* x0;
  float* scale;  // [3][count]: 1 / den, 1 / den^2, den
  int64_t stride;
  int32_t m, n, count;
};

// Momentum, Nesterov blend, X0, the norm and the non-finite flag in one launch.
__attribute__((visibility("hidden"))) int small_prepare(const SmallBatch& b, bool orth_only,
                                                        float mom_w, float nest_w,
                                                        uint32_t* found_inf, hipStream_t s);

enum class SmallOut { kStore, kApply, kExtract };

struct SmallChain {
  float a, b, c;
  int32_t steps;
  // kStore: X of matrix i, [m, n] in rows of ldx at x + i * stride
  uint16_t* x;
  int64_t ldx;
  // kApply: the parameter update (as muon_update_element), scale by matrix
  float decay, neg_lr;
  float scale[kSmallMaxMats];
};

// The whole Newton-Schulz chain of every matrix, and what follows it, in one launch.
__attribute__((visibility("hidden"))) int small_chain(const SmallBatch& b, const SmallChain& c,
                                                      SmallOut out, hipStream_t s);

}  // namespace morph
