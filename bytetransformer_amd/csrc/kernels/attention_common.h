// Device helpers shared by the fp16 attention kernels.
#pragma once
#include "common.h"

namespace bt {

constexpr float kNegBig = -1.0e30f;
constexpr float kLog2e = 1.4426950408889634f;
#ifndef BT_LAZY_MAX
#define BT_LAZY_MAX 8.0f
#endif
constexpr float kLazyMax = BT_LAZY_MAX;   // see the running maximum in the tile loops

typedef float float2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Reductions over the four 16-lane rows of a wave (lanes l, l^16, l^32, l^48) with the
// row-swap VALU instructions: after a swap of two copies of x, the pair holds x of
// rows {0,0,2,2} / {1,1,3,3} (16-lane swap) or {0,1,0,1} / {2,3,2,3} (32-lane swap),
// so one max / add per step folds the partner row in - no LDS round trip.  The empty
// asm keeps the optimiser from treating the two results of a swap of equal inputs as
// equal (it then drops the max / add).
__device__ __forceinline__ void swap_rows16(float x, float &lo, float &hi) {
  const unsigned u = __builtin_bit_cast(unsigned, x);
  auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  unsigned r0 = r[0], r1 = r[1];
  asm volatile("" : "+v"(r0), "+v"(r1));
  lo = __builtin_bit_cast(float, r0);
  hi = __builtin_bit_cast(float, r1);
}
__device__ __forceinline__ void swap_rows32(float x, float &lo, float &hi) {
  const unsigned u = __builtin_bit_cast(unsigned, x);
  auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  unsigned r0 = r[0], r1 = r[1];
  asm volatile("" : "+v"(r0), "+v"(r1));
  lo = __builtin_bit_cast(float, r0);
  hi = __builtin_bit_cast(float, r1);
}
__device__ __forceinline__ float rows_max(float x) {
  float a, b;
  swap_rows16(x, a, b);
  swap_rows32(fmaxf(a, b), a, b);
  return fmaxf(a, b);
}
__device__ __forceinline__ float rows_sum(float x) {
  float a, b;
  swap_rows16(x, a, b);
  swap_rows32(a + b, a, b);
  return a + b;
}

template <int N>
__device__ __forceinline__ void att_wait_vmcnt() {
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0F70);
}

__device__ __forceinline__ void lds_dma16(const half_t *src, half_t *dst) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src,
                                   (__attribute__((address_space(3))) void *)dst, 16, 0, 0);
}

// LDS transpose read of 4 rows x 16 columns per 16 lanes, and the wait for what is tied to it, as
// assembly: in front of the compiler's own transpose read it waits for every direct-to-LDS load in
// flight, that is, for the tile that was requested moments ago, and a ring of tiles then hides nothing
// (batch 16 x 512: 30.4 us of attention over full sequences with those waits, 29.8 without; 12 x 380 under a mask 24.4 and 23.2).
template <int OFFSET>
__device__ __forceinline__ uint2_t lds_read_tr(unsigned address) {
  static_assert(OFFSET >= 0 && OFFSET < 65536, "offset field of an LDS instruction");
  uint2_t v;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v) : "v"(address), "n"(OFFSET));
  return v;
}
template <int LEFT>   // all but the LEFT youngest LDS operations have returned, these eight among them
__device__ __forceinline__ void lds_wait_tied(uint2_t (&a)[4], uint2_t (&b)[4]) {
  asm volatile("s_waitcnt lgkmcnt(%8)"
               : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3])
               : "n"(LEFT));
}
__device__ __forceinline__ unsigned lds_address(const half_t *p) {
  return (unsigned)(unsigned long long)(__attribute__((address_space(3))) const half_t *)p;
}

// Additive terms of the logits in the exp2 domain: the mask shift (mask - 1) * 10000 (the reference's
// non-remove-padding kernels, attention_fused.cu:234-237) plus the attention bias (softmax.h:41-46 adds
// it to the scaled logits before the mask term).  One row [S] of such a tensor, read four
// consecutive keys at a time as they lie (the memory path takes 8-byte loads at any even address);
// keys at or past S get what follows in memory and are excluded by the caller, by index.  At the very
// end of the tensor the load moves back to the last four elements and is shifted.  (Launches of S = 1,
// whose tensors can be smaller than that, come without terms: see drop_terms_of_one_key.)
struct TermRow {
  const half_t *at;   // the row
  int last;           // offset from `at` of the tensor's last four elements
  __device__ __forceinline__ TermRow(const half_t *tensor, size_t row, int S, size_t rows) {
    at = tensor + row * S;
    const size_t left = (rows - row) * S;   // elements from here to the end
    last = (left < 0x40000000 ? (int)left : 0x40000000) - 4;
  }
  // Request (INSIDE: all four keys lie in the row) and, once it is used, the elements in order.
  template <bool INSIDE>
  __device__ __forceinline__ uint2_t fetch(int key) const {
    uint2_t v;
    __builtin_memcpy(&v, at + (INSIDE ? key : min(key, last)), sizeof(v));
    return v;
  }
  __device__ __forceinline__ uint2_t in_order(uint2_t v, int key) const {
    const int by = 16 * min(key - min(key, last), 3);
    return __builtin_bit_cast(uint2_t, __builtin_bit_cast(unsigned long long, v) >> by);
  }
};
// Which additive terms a kernel applies (a template parameter: decided at run time, the choice is a branch
// per four keys, and a tile of them takes twice as long).
enum AddKind { kAddNone = 0, kAddMask = 1, kAddBias = 2, kAddBoth = 3, kAddZero = 4 };
// Without terms (kAddNone) the logits stay unscaled until they are in the exponent: the maximum is taken
// over them as they are, and keys that do not exist are -1e30 among them.  That needs a positive scale, and
// one that keeps -1e30 far below every logit; under any other the launch scales them first, as the ones
// with terms do (kAddZero: a kernel of its own, because a flag in the loop cost every small launch 0.2 us).
inline int add_kind(const half_t *mask, const half_t *bias, float scale) {
  const int kind = (mask ? kAddMask : 0) | (bias ? kAddBias : 0);
  return kind == kAddNone && !(scale >= 1e-20f) ? kAddZero : kind;
}
// A single key's probability does not depend on its term; what is left of a mask tensor is that
// every one of the S keys takes part.  Returns that for launches of S = 1.
inline bool drop_terms_of_one_key(int S, const half_t *&mask, const half_t *&bias) {
  const bool every_key = S == 1 && mask;
  if (S == 1) mask = bias = nullptr;
  return every_key;
}
// x = s * scale + term for four keys, from the raw elements of the mask row and the bias row.
template <int KIND>
__device__ __forceinline__ float4_t add_terms(float4_t s, float scale, uint2_t mask, uint2_t bias) {
  constexpr float kShift = 10000.0f * kLog2e;
  const half4_t m = __builtin_bit_cast(half4_t, mask), a = __builtin_bit_cast(half4_t, bias);
  float4_t v;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float t = 0.f;
    if (KIND & kAddMask) t = __builtin_fmaf((float)m[r], kShift, -kShift);
    if (KIND & kAddBias) t = __builtin_fmaf((float)a[r], kLog2e, t);
    v[r] = __builtin_fmaf(s[r], scale, t);
  }
  return v;
}

// ---- cache warm-up on behalf of later kernels ------------------------------------------------
// Ranges that the launches after this one will read (the layer's remaining weights): some workgroups
// touch one dword per 128-byte line of their slice, so that the products find them in the memory-side
// cache.  Range r holds the lines [end[r - 1], end[r]) of the concatenation (end[3] = 0: none).
constexpr int kWarmRanges = 4;
struct WarmDuty {
  const char *base[kWarmRanges];
  unsigned end[kWarmRanges];
  unsigned first;       // the workgroups from here on take part
  unsigned per;         // lines of each
  unsigned grid_work;   // workgroups of the attention itself: later ones do nothing else
};
template <int THREADS>
__device__ __forceinline__ void warm_slice(const WarmDuty &w) {
  const unsigned lines = w.end[kWarmRanges - 1];
  if (!lines || workgroup_id() < w.first) return;
  const unsigned first = (workgroup_id() - w.first) * w.per;
  touch_lines(w.base, w.end, first + thread_id(), min(first + w.per, lines), THREADS);
}
// Who takes part, for a launch of `grid` workgroups (grown here by the ones that only warm).
//   Two workgroups per CU and more (option prefetch_min_grid): the last quarter of the issue order -
//   short sequences and dead tiles, which retire early - at four lines a thread (batch 16 at 512 tokens: -4
//   to -6 % per forward; half of the grid measured 0.7 % slower).
//   Fewer: the launch leaves CUs idle, and 96 to 208 workgroups of their own, about what fills the chip
//   up, touch the weights meanwhile.  Left to the attention's own workgroups the touches lengthened
//   it (+3 to +8 % per forward); with workgroups of their own 12 layers take 454 -> 412 us at batch
//   1 x 32, 545 -> 490 at 1 x 256, 520 -> 477 at 4 x 96, 800 -> 762 at 7 x 217, 929 -> 875 at 6 x 250.
//   More than 12 MB (BERT-large has 25 with the next layer's QKV weight) takes longer than the
//   attention itself: 24 layers of hidden 1024 at 3 x 28, encoder entry 924 us with 12 MB, 935 with all.
inline int plan_warm_duty(const char *who, WarmDuty &w, unsigned &grid, const void *const *ranges,
                          const unsigned long long *bytes, int count) {
  for (int r = 0; r < kWarmRanges; ++r) {
    w.base[r] = nullptr;
    w.end[r] = 0;
  }
  w.first = w.grid_work = grid;
  w.per = 0;
  BT_REQUIRE(count >= 0 && count <= kWarmRanges, BT_ERR_INVALID_ARGUMENT,
             "%s: prefetch_count=%d outside [0, %d]", who, count, kWarmRanges);
  BT_REQUIRE(count == 0 || (ranges && bytes), BT_ERR_INVALID_ARGUMENT,
             "%s: prefetch ranges need their pointers and sizes", who);
  if (!count || !option_prefetch()) return BT_OK;
  unsigned long long left;   // lines that the duty workgroups take on
  if (grid < (unsigned)option_prefetch_min_grid()) {
    const unsigned idle = grid < 256 ? 256 - grid : 0, extra = idle < 96 ? 96 : idle > 208 ? 208 : idle;
    grid += extra;
    left = 98304;   // 12 MB: what fits beside an attention of 4 to 6 us
  } else {
    w.first = (unsigned)((unsigned long long)grid * 3 / 4);
    left = (unsigned long long)(grid - w.first) * 4 * 256;
  }
  unsigned end = 0;
  for (int r = 0; r < kWarmRanges; ++r) {
    if (r < count && ranges[r] && left) {
      // one dword at the start of each 128-byte line; a last line of fewer than four bytes
      // is left alone, so no byte outside the range is read
      unsigned long long lines = (bytes[r] + 124) / 128;
      if (lines > left) lines = left;
      left -= lines;
      w.base[r] = (const char *)ranges[r];
      end += (unsigned)lines;
    }
    w.end[r] = end;
  }
  if (end) w.per = (end + (grid - w.first) - 1) / (grid - w.first);
  return BT_OK;
}

}  // namespace bt
