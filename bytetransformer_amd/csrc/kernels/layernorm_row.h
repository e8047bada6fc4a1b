// One LayerNorm row in the registers of a wave: what the LayerNorm launches and the launch that goes straight on to
// FFN1 share.
#pragma once
#include "common.h"

namespace bt {

// V consecutive halfs of a row: what a lane loads, adds and stores at a time.
template <int V>
struct LnVec;
template <>
struct LnVec<8> {
  typedef half8_t halfs;
  typedef uint4_t bits;
};
template <>
struct LnVec<4> {
  typedef half4_t halfs;
  typedef uint2_t bits;
};

// x = (a + r) + bias, two fp16-rounded adds; leaves x - mean in v and returns 1 / sqrt(variance + eps).
template <int NC, int V, typename H = typename LnVec<V>::halfs>
__device__ __forceinline__ float ln_statistics(const H (&av)[NC], const H (&rv)[NC], const H (&bias_v)[NC],
                                               const bool (&live)[NC], float inv_n, float eps, float (&v)[NC][V]) {
  // (four sums side by side: a quarter of the chain)
  float part[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const H x = (av[i] + rv[i]) + bias_v[i];  // two fp16-rounded adds
#pragma unroll
    for (int j = 0; j < V; ++j) {
      v[i][j] = live[i] ? (float)x[j] : 0.f;
      part[j & 3] += v[i][j];
    }
  }
  const float mean = wave_sum((part[0] + part[1]) + (part[2] + part[3])) * inv_n;
  float sq[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < NC; ++i) {
#pragma unroll
    for (int j = 0; j < V; ++j) {
      v[i][j] = live[i] ? v[i][j] - mean : 0.f;
      sq[j & 3] += v[i][j] * v[i][j];
    }
  }
  return rsqrtf(wave_sum((sq[0] + sq[1]) + (sq[2] + sq[3])) * inv_n + eps);
}

}  // namespace bt
