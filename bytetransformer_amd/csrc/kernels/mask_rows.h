// Offsets counted from the mask by a launch that needs them: what the products and the launch that splits float operands share.
// Args has mask, mask_B, mask_S and out_batch_idx, out_word_idx, out_seq_order.
#pragma once
#include "common.h"

namespace bt {

constexpr int kMaskNone = 0, kMaskF16 = 1, kMaskF32 = 2;

// ---- rows from the mask ---------------------------------------------------------
constexpr int kMaskRowsMaxBatch = 64;   // one wave scans the lengths

// Per-lane view of the offsets, the same in every wave: lane l < B holds sequence l.
struct MaskRows {
  int len;     // its length
  int excl;    // its first packed row (lanes >= B: M)
  int delta;   // l * S - excl: padded row = packed row + delta
  int M;       // live rows
};

// All `nwaves` waves of the workgroup take part (one barrier inside).  `s_len`: 64 ints of
// LDS that nothing else writes until every wave has left this function.
template <int MASK, typename Args>
__device__ __forceinline__ MaskRows mask_rows_setup(const Args &p, int wave, int nwaves, int lane, int *s_len) {
  using T = std::conditional_t<MASK == kMaskF32, float, half_t>;
  const int B = p.mask_B, S = p.mask_S;
  const size_t plane = (size_t)S * S;
  // R rows per wave in flight at a time: two for up to 2 * nwaves sequences (their 16-byte
  // loads cover rows of up to 1024 halfs in one round trip), four beyond
  auto count_rows = [&](auto r_tag) {
    constexpr int R = decltype(r_tag)::value;
    const T *m = (const T *)p.mask;
    for (int b0 = wave; b0 < B; b0 += R * nwaves) {
      const T *rows[R];
      int count[R];
#pragma unroll
      for (int r = 0; r < R; ++r)
        rows[r] = b0 + r * nwaves < B ? m + (b0 + r * nwaves) * plane : nullptr;
      wave_row_lengths<T, R>(rows, S, lane, count);
      if (lane == 0) {
#pragma unroll
        for (int r = 0; r < R; ++r)
          if (b0 + r * nwaves < B) s_len[b0 + r * nwaves] = count[r];
      }
    }
  };
  using two = std::integral_constant<int, 2>;
  using four = std::integral_constant<int, 4>;
  if (B <= 2 * nwaves) count_rows(two{}); else count_rows(four{});
  __syncthreads();
  MaskRows mr;
  mr.len = lane < B ? s_len[lane] : 0;
  const int incl = wave_inclusive_sum(mr.len);
  mr.excl = incl - mr.len;
  mr.delta = lane * S - mr.excl;
  mr.M = __builtin_amdgcn_readlane(incl, 63);
  return mr;
}

// Which sequences the packed rows [r0, r1] (0 <= r0 <= r1 < M, wave-uniform) belong to: the
// first one and how many more.  The first packed rows rise with the lane, so the lanes whose
// sequence starts at or before a row form a prefix; the last of them holds the row (empty
// sequences in between start at the same row and lose to it).
struct MaskRowSpan {
  int first, more;
};
__device__ __forceinline__ MaskRowSpan mask_rows_span(const MaskRows &mr, int B, int lane, int r0,
                                                      int r1) {
  const int lo = __popcll(__ballot(lane < B && mr.excl <= r0)) - 1;
  const int hi = __popcll(__ballot(lane < B && mr.excl <= r1)) - 1;
  return MaskRowSpan{lo, hi - lo};
}

// Padded row of packed row r inside such a span.  Every lane of the wave must call it (the
// look-ups read the other lanes' registers).
__device__ __forceinline__ int mask_rows_map(const MaskRows &mr, const MaskRowSpan &sp, int r) {
  int b = sp.first;
  for (int k = 1; k <= sp.more; ++k) b += r >= __builtin_amdgcn_readlane(mr.excl, sp.first + k);
  return r + __shfl(mr.delta, b, 64);
}

// The offsets as the stand-alone launch writes them (padding.hip), by `nthreads` threads
// (whole waves, t = thread index among them) of one workgroup.
template <typename Args>
__device__ __forceinline__ void mask_rows_write(const Args &p, const MaskRows &mr, int t, int nthreads, int lane) {
  const int B = p.mask_B, S = p.mask_S;
  if (t < 64) {   // the first of the writing waves
    if (p.out_batch_idx) {
      if (lane < B) p.out_batch_idx[lane] = mr.excl;
      if (lane == 0) p.out_batch_idx[B] = mr.M;
    }
    if (p.out_seq_order) {
      // sequences by descending length (ties by index): rank by counting
      int rank = 0;
      for (int o = 0; o < B; ++o) {
        const int lo = __shfl(mr.len, o, 64);
        rank += (lo > mr.len) || (lo == mr.len && o < lane);
      }
      if (lane < B) p.out_seq_order[rank] = lane;
    }
  }
  if (p.out_word_idx) {
    for (int b = 0; b < B; ++b) {
      const int off = __shfl(mr.excl, b, 64), len = __shfl(mr.len, b, 64);
      const int pad_at = mr.M + b * S - off;   // the padded positions fill the tail from M on
      for (int i = t; i < S; i += nthreads)
        p.out_word_idx[i < len ? off + i : pad_at + i - len] = b * S + i;
    }
  }
}

}  // namespace bt
