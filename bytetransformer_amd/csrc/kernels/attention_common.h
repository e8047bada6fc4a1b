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
// Ranges that the launches after this one will read (the layer's remaining weights): some workgroups touch one
// dword per 128-byte line of them.  A range is rows of `pitch` bytes, and the workgroups of XCD x touch one eighth of
// it: 2^-cols of the bytes of 2^(cols - 3) of the rows.  For a weight that is the eighth whose tiles the XCD will
// work on (tile_at: products of few rows go column by column), so they are found in its own L2 and not just in the
// memory-side cache: 96 KB come to a CU in 1.2 us from the one and in 1.6 to 2.5 from the other.
// 12 layers with the lines as they lie dealt out to all XCDs, and so, us: as stored 1 x 32 341 -> 331, 1 x 64 342 -> 339,
// pre-packed (rows of 128 bytes) 1 x 32 318 -> 315.  With more rows than that order has (prefetch_weight) nothing is
// gained, and the shorter runs cost: a wave's lines 1 KB apart 7 x 217 +4 %, eighths 16 x 512 +1 %.
constexpr int kWarmRanges = 4;
struct WarmDuty {
  const char *base[kWarmRanges];
  unsigned shape[kWarmRanges];   // pitch / 64 | rows << 16, or how many lines
  unsigned ends;                 // byte r: of an XCD's workgroups that take part, those below it take ranges 0 .. r
  unsigned forms_turns;          // per range 4 bits, cols | rows first << 2; from bit 16: the most lines of a thread
  unsigned first;                // the workgroups from here on take part, a multiple of 8
  unsigned grid_work;            // workgroups of the attention itself: later ones do nothing else
};
constexpr unsigned kWarmRowsFirst = 4;   // form: the eighths are counted along the rows first
constexpr unsigned kWarmLines = 8;       // form: no eighths, lines as they lie, dealt out to all XCDs
__host__ __device__ constexpr unsigned warm_rows(unsigned shape, unsigned cols) {   // of an eighth
  return ((shape >> 16) + (8u >> cols) - 1) >> (3 - cols);
}
__host__ __device__ constexpr unsigned warm_row_lines(unsigned shape, unsigned cols) {
  return (((shape & 0xffffu) * 64u >> cols) + 127) / 128;
}
template <int THREADS>
__device__ __forceinline__ void warm_slice(const WarmDuty &w) {
  if (workgroup_id() < w.first) return;
  const unsigned x = workgroup_id() & 7, mine = (workgroup_id() - w.first) >> 3;
  // (a workgroup has one range: with the lines of all dealt out one after the other, every thread found its range by
  // itself, and the attention of 1 x 256 took 8.1 us, of 8 x 64 4.75)
  unsigned begin = 0, end = w.ends & 0xff, shape = w.shape[0], form = w.forms_turns & 15;
  const char *from = w.base[0];
#pragma unroll
  for (int r = 1; r < kWarmRanges; ++r) {
    const bool here = mine >= end;
    begin = here ? end : begin, shape = here ? w.shape[r] : shape, form = here ? w.forms_turns >> 4 * r & 15 : form;
    from = here ? w.base[r] : from, end = here ? w.ends >> 8 * r & 0xff : end;
  }
  if (mine >= end) return;
  const unsigned turns = w.forms_turns >> 16;
  if (form & kWarmLines) {
    const unsigned parts = (end - begin) * 8;
    touch_lines<THREADS>(min(shape, parts * THREADS * turns), (mine - begin) * 8 + x, parts,
                         [&](unsigned l) { return (unsigned long long)from + l * 128ull; });
    return;
  }
  const unsigned cols = form & 3, pitch = (shape & 0xffffu) * 64, rows = warm_rows(shape, cols), row_lines = warm_row_lines(shape, cols);
  const unsigned at_row = (form & kWarmRowsFirst ? x & ((8u >> cols) - 1) : x >> cols) * rows;
  const unsigned at_col = form & kWarmRowsFirst ? x >> (3 - cols) : x & ((1u << cols) - 1);
  from += (unsigned long long)at_row * pitch + (at_col * (pitch >> cols) & ~63u);
  const int last = (int)(shape >> 16) - 1 - (int)at_row;   // row of the share that is the range's last
  const float inverse = __builtin_amdgcn_rcpf((float)row_lines);
  touch_lines<THREADS>(min(rows * row_lines, (end - begin) * THREADS * turns), mine - begin, end - begin, [&](unsigned l) {
    const int row = (int)(((float)l + 0.5f) * inverse);   // l / row_lines, exact below 2^21
    return (unsigned long long)from + ((long long)min(row, last) * pitch + (l - row * row_lines) * 128);
  });
}
// Who takes part, for a launch of `grid` workgroups (grown here by the ones that only warm).
//   Two workgroups per CU and more (option prefetch_min_grid): the last quarter of the issue order -
//   short sequences and dead tiles, which retire early - at four lines a thread (batch 16 at 512 tokens: -4
//   to -6 % per forward; half of the grid measured 0.7 % slower).
//   Fewer: the launch leaves CUs idle, and 96 to 208 workgroups of their own, about what fills the chip
//   up, touch the weights meanwhile.  Left to the attention's own workgroups the touches lengthened
//   it (+3 to +8 % per forward); with workgroups of their own 12 layers take 454 -> 412 us at batch
//   1 x 32, 545 -> 490 at 1 x 256, 520 -> 477 at 4 x 96, 800 -> 762 at 7 x 217, 929 -> 875 at 6 x 250.
//   More than 15 MB (BERT-large has 25 with the next layer's QKV weight) takes longer than the
//   attention itself and is cut to 12: 24 layers of hidden 1024, encoder entry, 3 x 28 924 us with 12 MB, 935 with all;
//   10 x 100 1398 with 12, 1430 with 14.  Hidden 768 has 14.2 with the next QKV weight: 12 layers, all and with 12 (the
//   QKV weight's end left out), us: 4 x 96 372 / 383, 8 x 64 417 / 424, 7 x 217 579 / 596.
inline int plan_warm_duty(const char *who, WarmDuty &w, unsigned &grid, const void *const *ranges,
                          const unsigned long long *bytes, int count) {
  for (int r = 0; r < kWarmRanges; ++r) {
    w.base[r] = nullptr;
    w.shape[r] = 0;
  }
  w.first = w.grid_work = grid;
  w.ends = w.forms_turns = 0;
  BT_REQUIRE(count >= 0 && count <= kWarmRanges, BT_ERR_INVALID_ARGUMENT,
             "%s: prefetch_count=%d outside [0, %d]", who, count, kWarmRanges);
  BT_REQUIRE(count == 0 || (ranges && bytes), BT_ERR_INVALID_ARGUMENT,
             "%s: prefetch ranges need their pointers and sizes", who);
  if (!count || !option_prefetch()) return BT_OK;
  unsigned per, most;   // workgroups of an XCD, and lines that they take on
  if (grid < (unsigned)option_prefetch_min_grid()) {
    const unsigned idle = grid < 256 ? 256 - grid : 0, extra = idle < 96 ? 96 : idle > 208 ? 208 : idle;
    w.first = (grid + 7) / 8 * 8;
    per = extra / 8;
    grid = w.first + per * 8;
    unsigned long long all = 0;
    for (int r = 0; r < count; ++r) all += ranges[r] ? bytes[r] & ((1ull << 40) - 1) : 0;
    most = all <= (15ull << 20) ? 15360 : 12288;   // of 128 bytes and eight XCDs: 15 and 12 MB
  } else {
    w.first = (unsigned)(((unsigned long long)grid * 3 / 4 + 7) / 8 * 8);
    per = grid > w.first ? (grid - w.first) / 8 : 0;
    if (per > 0xff) per = 0xff;
    most = per * 4 * 256;
  }
  unsigned lines = 0, upto[kWarmRanges];
  int at = 0;
  for (int r = 0; r < count; ++r) {
    const unsigned long long size = bytes[r] & ((1ull << 40) - 1);
    unsigned pitch = (unsigned)(bytes[r] >> 40 & 0xffff) * 64, cols = (unsigned)(bytes[r] >> 56 & 3);
    unsigned form = cols | (bytes[r] >> 58 & 1 ? kWarmRowsFirst : 0);
    unsigned long long rows = pitch ? size / pitch : 0;
    if (!rows || rows > 0xffff || rows * pitch != size || rows % (8u >> cols) || (pitch >> cols) % 64) {
      // (of the last line at least four bytes lie inside the range, so no byte outside it is read)
      rows = (size + 124) / 128;
      if (rows > 0xffffff) rows = 0xffffff;
      form = kWarmLines;
    }
    if (!ranges[r] || !rows || lines >= most) continue;
    w.base[at] = (const char *)ranges[r];
    w.shape[at] = form == kWarmLines ? (unsigned)rows : pitch / 64 | (unsigned)rows << 16;
    w.forms_turns |= form << 4 * at;
    lines += form == kWarmLines ? (unsigned)(rows + 7) / 8 : warm_rows(w.shape[at], cols) * warm_row_lines(w.shape[at], cols);
    upto[at++] = lines = lines < most ? lines : most;   // (what is beyond is the last range's end)
  }
  if (!at || !per) return BT_OK;
  // workgroups by lines, one for a range at least, and turns enough for every line: a product that finds nine lines in ten
  // takes nearly as long as one that finds none (7 x 217 with a tenth left out: FFN2 10.2 -> 12.9 us)
  unsigned turns = 1;
  for (int r = 0; r < at; ++r) {
    unsigned end = (unsigned)(((unsigned long long)upto[r] * per + lines / 2) / lines);
    const unsigned before = r ? w.ends >> 8 * (r - 1) & 0xff : 0, threads = 256;
    if (end <= before) end = before + 1;
    if (end > per) end = per;
    for (int q = r; q < kWarmRanges; ++q) w.ends = (w.ends & ~(0xffu << 8 * q)) | end << 8 * q;
    const unsigned mine = upto[r] - (r ? upto[r - 1] : 0), at_once = (end - before) * threads;
    if (at_once && (mine + at_once - 1) / at_once > turns) turns = (mine + at_once - 1) / at_once;
  }
  w.forms_turns |= turns << 16;
  return BT_OK;
}

}  // namespace bt
