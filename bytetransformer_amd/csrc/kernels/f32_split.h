// Floats as scaled pairs of fp16 numbers (fp32_split.hip says what they are): shared by the launches that make them.
#pragma once
#include "common.h"

namespace bt {

constexpr int kSplitChunk = 256;   // values of a weight's column that share a scale
constexpr float kSplitLow = 1.0f / 2048.0f;   // what a pair's second number is worth

struct SplitPair {
  half_t h, l;
  float off;   // what the pair leaves out
  __device__ __forceinline__ bool held(float x) const {   // the value to 2^-22 of itself (what is not finite counts as held)
    return !(__builtin_fabsf(off) > __builtin_fabsf(x) * 0x1p-22f);
  }
};
// of a scaled value: the second number is zero where the first is not finite
__device__ __forceinline__ SplitPair split_pair(float x) {
  const half_t h = (half_t)x;
  const float rest = (x - (float)h) * 2048.0f;
  const half_t l = __builtin_fabsf((float)h) < __builtin_inff() ? (half_t)rest : (half_t)0.f;
  return SplitPair{h, l, (rest - (float)l) * kSplitLow};
}
// The exponent that brings a largest value m >= 0 to [2^14, 2^15) (0 for no value at all), held where 2^e is a float.
__device__ __forceinline__ int split_exponent(float m) {
  const int e = 14 + 127 - (int)(__builtin_bit_cast(unsigned, m) >> 23);
  return m == 0.f ? 0 : min(e, 126);   // (at least -113: m is finite)
}
__device__ __forceinline__ float split_power(int e) { return __builtin_bit_cast(float, (unsigned)(e + 127) << 23); }

// What a value v says of its row (or chunk of a column): how far off its pair is, relative to the value and squared, less what
// it may be.  Where the sum is positive the pairs are off by more than 2^-22.5 of their values in the root mean square - the
// error of products that all weigh the same, whatever the scales of their operands - and the row is marked.  (Ordinary rows
// are at 2^-24.6; a value that does this alone lies below 2^-31 of the largest, in one chunk of ten million and one row of
// five.)
__device__ __forceinline__ float split_score(float v, float scale) {
  const float x = v * scale;
  const SplitPair p = split_pair(x);
  const float off = p.off * __builtin_amdgcn_rcpf(x);
  const float mine = x == 0.f ? 1.f : fminf(off * off, 1.f);   // (NaN: 1; only finite values count)
  return v == 0.f || !(__builtin_fabsf(v) < __builtin_inff()) ? 0.f : mine - 0x1p-45f;
}
__device__ __forceinline__ float split_score(float4_t v, float scale) {
  return (split_score(v[0], scale) + split_score(v[1], scale)) + (split_score(v[2], scale) + split_score(v[3], scale));
}
// No scaled value from here on is lost (what its pair leaves out is 2^-36 at most, 2^-22 of the value).
constexpr float kSplitHeldFrom = 1.0f / (1 << 14);
// An exponent that carries this mark is that of a row whose sums are formed from its floats.
constexpr int kSplitMark = 1 << 12;
__device__ __forceinline__ bool split_marked(int e) { return e >= kSplitMark / 2; }
__device__ __forceinline__ int split_unmarked(int e) { return split_marked(e) ? e - kSplitMark : e; }

// Four scaled values (float4 c of a row) into the row's pairs; true if one may be lost.
__device__ __forceinline__ bool split_store(half_t *row, int c, float4_t x) {
  half4_t h, l;
  bool small = false;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const SplitPair p = split_pair(x[e]);
    h[e] = p.h, l[e] = p.l, small = small || __builtin_fabsf(x[e]) < kSplitHeldFrom;
  }
  half_t *to = row + (c >> 3) * 64 + (c & 7) * 4;
  store_through(to, __builtin_bit_cast(uint2_t, h));
  store_through(to + 32, __builtin_bit_cast(uint2_t, l));
  return small;
}

// Where a row of pairs holds floats instead: a word that is not zero if it does at all, and a bit for every 32 columns.
__host__ __device__ constexpr int split_raw_words(int columns) { return 1 + (columns + 1023) / 1024; }

// 0.5 x (1 + tanh(u)) == x / (1 + exp(-2u)),  u = 0.79788456 (x + 0.044715 x^3), the exponent folded into one polynomial
__device__ __forceinline__ float f32_gelu(float x) {
  constexpr float c1 = -2.0f * 0.7978845608028654f * 1.4426950408889634f;
  constexpr float c3 = c1 * 0.044715f;
  const float e = __builtin_amdgcn_exp2f(x * (c1 + c3 * x * x));
  return x * __builtin_amdgcn_rcpf(1.0f + e);
}

}  // namespace bt
