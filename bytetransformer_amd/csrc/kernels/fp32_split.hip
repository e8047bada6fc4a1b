// The products of the float layer on fp16 matrix instructions, for batches whose operands are worth splitting
// once: every operand is stored as pairs of fp16 numbers by the launch that makes it, and the products are the
// tiled fp16 products' twins with three matrix instructions where those have one.
//
//   split_f32_kernel       weights [K, N] and gathered rows of the input -> their pairs, k-contiguous
//   f32_split_gemm_kernel  c = a . w (+ bias), or the pairs of GELU(a . w + bias)
//   f32_layernorm_split    (fp32_path.hip) writes the pairs of its rows beside the rows
//
// The pair.  A row (or 256 consecutive values of a weight's column) is scaled by a power of two that brings its largest value to [2^14, 2^15);
// of x so scaled, h = fp16(x) and l = fp16((x - h) 2^11), round to nearest.  x - h is exact and at most 2^-11 |x|,
// so h + l / 2^11 is x to 2^-23 of its own (three floats in four exactly), and since l has the exponent range of h
// that holds down to 2^-27 of the largest value; what is smaller still is off by 2^-50 of that value at most
// (h and l are subnormal there: off by 2^-25 in l, 2^-36 of a value scaled to 2^14 or more).
// a . w is then the sum of ah wh and of (ah wl + al wh) / 2^11, each in float accumulators of its own; al wl, 2^-22
// of a product, is left out.  Against the exact bfloat16 triples of bt_gemm_f32 (six matrix instructions, one
// accumulator) the operands are rounded, but the sums are half to a sixth as many roundings: see
// bt_gemm_f32_split in bt_hip.h for both errors.
// Infinities and NaN keep their places in h (the scale comes from the finite values of a row); a row with a sum that is
// not finite is formed again, from the floats.
//
// Rows and chunks of columns of which the pairs hold less, because some values are out of all proportion to the rest, are
// marked (split_score), and what they enter is summed from the floats: the large value may meet a zero, the small one a large.
//
// The scale of FFN1's results has to be known before them, so it comes from a bound.  One large column makes that bound
// and with it what 2^-50 is worth to the results of all others, be it 10^12 times as large as any of them.  So where
// the pairs of a result's row do not hold what they should in the columns of a wave, these stay floats in the
// place of their pairs (as many bytes), with a bit that says so, and the product that reads that row forms its sums again.
//
// In memory a row of K floats is K / 32 blocks of 128 bytes: 32 h, then 32 l.  A block is one k-step's row of an
// LDS tile, so loads, swizzle and LDS reads are those of an fp16 product of 2 K halfs.
#include "f32_split.h"
#include "gemm_common.h"
#include "mask_rows.h"

#include <cmath>

namespace bt {
namespace {

typedef int int4_t __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// operands -> pairs
// ---------------------------------------------------------------------------
// A unit of a weight: 32 columns x 256 rows, which it reads once and scales by their own largest values.  (With one scale
// for a whole column every unit had to see all of its rows first: 28.6 us for the weights of a layer of hidden 768 out of
// HBM.)  What bounds it is the memory: 28 MB in and out.
constexpr int kSplitThreads = 512, kSplitCols = 32;
constexpr int kSplitPitch = 2 * kSplitChunk + 8;   // halfs of a column's rows in LDS

struct SplitWeight {
  const float *w;     // [K, N]
  half_t *pairs;      // [N][K / 32][64]
  int *exps;          // [ceil(K / 256)][N]
  int K, N, strips, unit_end;
};
struct SplitArgs {
  SplitWeight weight[4];
  int count, units;
  int bounded;              // the weight that `bounds` speaks of, -1: none
  int layer;                // bounds of GELU(. W + bias): what a bias adds to the largest |result| (else |bias|); marks
  const float *bias;        // [N] its bias
  float *bounds;            // [units of that weight][2]: largest finite |w| and |bias| of its columns
  const float *rows;        // rows to split as well, or null
  half_t *row_pairs;        // [rows_cap][K / 32][64]
  int *row_exps;
  const int *row_index, *valid_rows;
  int rows_cap, hidden;
  int row_blocks;           // workgroups for the rows
  // a launch that counts the rows from the mask, and leaves the offsets for the launches behind it
  const void *mask;
  int mask_B, mask_S;
  int *out_batch_idx, *out_word_idx, *out_seq_order;
};

__device__ __forceinline__ float finite_or_zero(float x) {
  return (__builtin_bit_cast(unsigned, x) & 0x7f800000u) == 0x7f800000u ? 0.f : __builtin_fabsf(x);
}

__device__ __forceinline__ void split_weight_unit(const SplitArgs &a, int unit) {
  constexpr int kPasses = kSplitChunk / (kSplitThreads / 8);   // 64 rows each
  __shared__ float4_t s_most[kSplitThreads / 64][8];
  __shared__ float s_scale[kSplitCols];
  __shared__ float4_t s_score[kSplitThreads / 64][8];
  __shared__ int s_small[kSplitThreads / 64];
  __shared__ __attribute__((aligned(16))) half_t s_tile[kSplitCols * kSplitPitch];
  int j = 0, first = 0;
#pragma unroll
  for (int i = 1; i < 4; ++i)
    if (i < a.count && unit >= a.weight[i - 1].unit_end) j = i, first = a.weight[i - 1].unit_end;
  const SplitWeight jb = a.weight[j];
  const int u = unit - first, chunk = u / jb.strips, strip = u - chunk * jb.strips;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int cq = t & 7, r0 = t >> 3, n0 = strip * kSplitCols, k0 = chunk * kSplitChunk;
  const float4_t *src = (const float4_t *)(jb.w + n0) + cq;

  // thread: four columns of rows r0, r0 + 64, ... (K is a multiple of 64)
  float4_t v[kPasses];
#pragma unroll
  for (int i = 0; i < kPasses; ++i) {
    v[i] = float4_t{0.f, 0.f, 0.f, 0.f};
    if (k0 + 64 * i < jb.K) v[i] = src[(size_t)(k0 + 64 * i + r0) * (jb.N / 4)];
  }
  float4_t most = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < kPasses; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) most[e] = fmaxf(most[e], finite_or_zero(v[i][e]));
#pragma unroll
  for (int o = 8; o < 64; o <<= 1)
#pragma unroll
    for (int e = 0; e < 4; ++e) most[e] = fmaxf(most[e], __shfl_xor(most[e], o, 64));
  if (lane < 8) s_most[wave][lane] = most;
  __syncthreads();
  int column_e = 0;
  if (t < kSplitCols) {
    float m = 0.f;
#pragma unroll
    for (int w = 0; w < kSplitThreads / 64; ++w) m = fmaxf(m, s_most[w][t >> 2][t & 3]);
    const int e = split_exponent(m);
    s_scale[t] = split_power(e);
    column_e = e;
    if (j == a.bounded) {
      // (|GELU(x)| <= x above zero, 0.17 and |x| below)
      const float of = a.bias[n0 + t];
      float b = finite_or_zero(of);
      if (a.layer && of < 0.f) b = fminf(b, 0.1701f);
#pragma unroll
      for (int o = 1; o < 32; o <<= 1) m = fmaxf(m, __shfl_xor(m, o, 64)), b = fmaxf(b, __shfl_xor(b, o, 64));
      if (t == 0) a.bounds[2 * u] = m, a.bounds[2 * u + 1] = b;
    }
  }
  __syncthreads();
  float scale[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) scale[e] = s_scale[4 * cq + e];
  bool small = false;
#pragma unroll
  for (int i = 0; i < kPasses; ++i) {
    half_t *to = s_tile + (64 * i + (r0 & 32)) * 2 + (r0 & 31);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float x = v[i][e] * scale[e];
      const SplitPair p = split_pair(x);
      to[(4 * cq + e) * kSplitPitch] = p.h;
      to[(4 * cq + e) * kSplitPitch + 32] = p.l;
      small = small || (__builtin_fabsf(x) < kSplitHeldFrom && v[i][e] != 0.f);
    }
  }
  const bool wave_small = a.layer && __builtin_amdgcn_ballot_w64(small) != 0;
  if (lane == 0) s_small[wave] = wave_small;
  __syncthreads();
  int any_small = 0;
#pragma unroll
  for (int w = 0; w < kSplitThreads / 64; ++w) any_small |= s_small[w];
  bool marked = false;
  if (__builtin_amdgcn_readfirstlane(any_small)) {   // (of the units of ordinary weights perhaps one)
    float4_t score = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    // (read once more: with the values in registers from before, half as many waves fit)
    for (int k = k0 + r0; k < min(k0 + kSplitChunk, jb.K); k += 64) {
      const float4_t again = src[(size_t)k * (jb.N / 4)];
#pragma unroll
      for (int e = 0; e < 4; ++e) score[e] += split_score(again[e], scale[e]);
    }
#pragma unroll
    for (int o = 8; o < 64; o <<= 1)
#pragma unroll
      for (int e = 0; e < 4; ++e) score[e] += __shfl_xor(score[e], o, 64);
    if (lane < 8) s_score[wave][lane] = score;
    __syncthreads();
    if (t < kSplitCols) {
      float all = 0.f;
#pragma unroll
      for (int w = 0; w < kSplitThreads / 64; ++w) all += s_score[w][t >> 2][t & 3];
      marked = all > 0.f;
    }
  }
  if (t < kSplitCols) jb.exps[(size_t)chunk * jb.N + n0 + t] = column_e + (marked ? kSplitMark : 0);
  const int rows = min(kSplitChunk, jb.K - k0), chunks16 = rows / 4;   // 16-byte pieces of a column
  for (int at = t; at < kSplitCols * (kSplitChunk / 4); at += kSplitThreads) {
    const int n = at / (kSplitChunk / 4), c = at % (kSplitChunk / 4);
    if (c < chunks16)
      store_through(jb.pairs + (size_t)(n0 + n) * 2 * jb.K + 2 * k0 + c * 8, *(const uint4_t *)(s_tile + n * kSplitPitch + c * 8));
  }
}

// The rows' workgroups come first: theirs is the longer chain, above all where they count the mask rows, and the weights'
// move in behind them.
template <int MASK>
__global__ __launch_bounds__(kSplitThreads) void split_f32_kernel(SplitArgs a) {
  if ((int)blockIdx.x >= a.row_blocks) return split_weight_unit(a, (int)blockIdx.x - a.row_blocks);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = (int)blockIdx.x * (kSplitThreads / 64) + wave;
  const int lane = threadIdx.x & 63;
  size_t from;
  if constexpr (MASK != kMaskNone) {
    __shared__ int s_len[kMaskRowsMaxBatch];
    const MaskRows mr = mask_rows_setup<MASK>(a, wave, kSplitThreads / 64, lane, s_len);
    if (blockIdx.x == 0) mask_rows_write(a, mr, (int)threadIdx.x, kSplitThreads, lane);
    if (r >= min(mr.M, a.rows_cap)) return;
    from = (size_t)__builtin_amdgcn_readfirstlane(mask_rows_map(mr, mask_rows_span(mr, a.mask_B, lane, r, r), r));
  } else {
    const int M = a.valid_rows ? min(scalar_load(a.valid_rows), a.rows_cap) : a.rows_cap;
    if (r >= M) return;
    from = a.row_index ? (size_t)scalar_load(a.row_index + r) : (size_t)r;
  }
  const float4_t *src = (const float4_t *)(a.rows + from * a.hidden);
  // up to 1024 values stay in registers, all asked for at once; of longer rows the rest is read again
  constexpr int kKept = 4;
  float4_t kept[kKept];
#pragma unroll
  for (int i = 0; i < kKept; ++i) {
    kept[i] = float4_t{0.f, 0.f, 0.f, 0.f};
    if (lane + 64 * i < a.hidden / 4) kept[i] = src[lane + 64 * i];
  }
  float most = 0.f;
  const auto look = [&](float4_t v) {
#pragma unroll
    for (int e = 0; e < 4; ++e) most = fmaxf(most, finite_or_zero(v[e]));
  };
#pragma unroll
  for (int i = 0; i < kKept; ++i) look(kept[i]);
  for (int c = lane + 64 * kKept; c < a.hidden / 4; c += 64) look(src[c]);
  const int e = split_exponent(wave_max(most));
  const float scale = split_power(e);
  bool small = false;
  half_t *to = a.row_pairs + (size_t)r * 2 * a.hidden;
#pragma unroll
  for (int i = 0; i < kKept; ++i)
    if (lane + 64 * i < a.hidden / 4) small = split_store(to, lane + 64 * i, kept[i] * scale) || small;
  for (int c = lane + 64 * kKept; c < a.hidden / 4; c += 64) small = split_store(to, c, src[c] * scale) || small;
  bool marked = false;
  if (a.layer && __builtin_amdgcn_ballot_w64(small) != 0) {
    float score = 0.f;
    for (int c = lane; c < a.hidden / 4; c += 64) score += split_score(src[c], scale);
    marked = wave_sum(score) > 0.f;
  }
  if (lane == 0) a.row_exps[r] = e + (marked ? kSplitMark : 0);
}

// ---------------------------------------------------------------------------
// products
// ---------------------------------------------------------------------------
struct F32SplitTail {
  const float *bias;   // [N] or null
  const int *gelu_exps;   // GELU: exponent that a row of the result is scaled by
  unsigned *raw;          // GELU: where a row of the result holds floats, [rows][split_raw_words(N)], or null
  const unsigned *a_raw;  // the same of the rows of a, or null
  const float *w;         // [K, N] the weight itself, or null
  const float *a_rows;    // row a_row_index[r] (r without an index) is what row r of a was made of, or null
  const int *a_row_index;
};
#define BT_F32_SPLIT_FIRST                                                                                  \
  const half_t *a, const half_t *w, const int *valid_rows, const int *a_exps, const int *w_exps, void *out, \
      int rows_cap, int N, int K, unsigned per_n
constexpr int kF32SplitFirstBytes = 64;   // the tail's place among the arguments

#if defined(__HIP_DEVICE_COMPILE__)
constexpr float kGeluFloor = 1.0f / (1 << 20);   // results below it may go: what they add is a rounding of what made the scale

// Sums of 16 rows and 16 TN columns on float matrix instructions, from the floats where there are any: those that the pairs
// do not give.  Lane (fr, lg): columns 16 i + 4 lg .. + 3 of row fr, as the products of pairs leave them; it brings row fr
// and columns 16 i + fr, values 4 lg .. 4 lg + 3 of every 16 of k, four loads of a column being one step's operands.
// Summed 64 values at a time (256: 2.9e-7 from float64 at k = 768, where bt_gemm_f32 has 2.1e-7; 64: 1.6e-7).  It waits for
// its own loads at every step: a layer of 16 x 256, hidden 768, whose FFN2 comes from here takes 853 us in place of 211, one
// whose QKV product does 652 in place of 296 (alone, launches included; by float multiply-adds, four rows a lane, 1860 and
// 2550).
template <int TN>
__device__ __forceinline__ void split_sums_of_floats(const half_t *a, const half_t *w, const int *a_exps, const int *w_exps,
                                                     const F32SplitTail &tail, int N, int K, int m, int n_first, int fr, int lg,
                                                     float4_t (&sum)[TN]) {
  const float4_t zero4 = {0.f, 0.f, 0.f, 0.f};
  float4_t part[TN];
#pragma unroll
  for (int i = 0; i < TN; ++i) sum[i] = part[i] = zero4;
  const int ea = split_unmarked(a_exps[m]);
  const unsigned *raw = tail.a_raw ? tail.a_raw + (size_t)m * split_raw_words(K) : nullptr;
  const float *row = tail.a_rows ? tail.a_rows + (size_t)(tail.a_row_index ? tail.a_row_index[m] : m) * K : nullptr;
#pragma unroll 1
  for (int k0 = 0; k0 < K; k0 += 16) {
    const int b = k0 >> 5, k = (k0 & 16) + 4 * lg;   // in its block
    float4_t x, y[TN];
    if (row) {
      x = *(const float4_t *)(row + k0 + 4 * lg);
    } else {
      const half_t *block = a + (size_t)m * 2 * K + b * 64;
      const half4_t h = *(const half4_t *)(block + k), l = *(const half4_t *)(block + 32 + k);
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = __builtin_amdgcn_ldexpf((float)h[e] + (float)l[e] * kSplitLow, -ea);
      if (raw && (raw[1 + (b >> 5)] >> (b & 31) & 1)) x = *(const float4_t *)((const float *)block + k);
    }
#pragma unroll
    for (int i = 0; i < TN; ++i) {
      const int n = min(n_first + 16 * i + fr, N - 1);
      if (tail.w) {
        const float *from = tail.w + (size_t)k0 * N;
#pragma unroll
        for (int e = 0; e < 4; ++e) y[i][e] = from[(unsigned)((4 * lg + e) * N + n)];
      } else {
        const half_t *block = w + (size_t)n * 2 * K + b * 64;
        const half4_t h = *(const half4_t *)(block + k), l = *(const half4_t *)(block + 32 + k);
        const int ew = split_unmarked(w_exps[(size_t)(k0 / kSplitChunk) * N + n]);
#pragma unroll
        for (int e = 0; e < 4; ++e) y[i][e] = __builtin_amdgcn_ldexpf((float)h[e] + (float)l[e] * kSplitLow, -ew);
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < TN; ++i) part[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(y[i][e], x[e], part[i], 0, 0, 0);
    if ((k0 + 16) % 64 == 0)
#pragma unroll
      for (int i = 0; i < TN; ++i) sum[i] += part[i], part[i] = zero4;
  }
}

// BM x BN tile, WM x WN waves that load and multiply, a ring of STAGES k-steps of 32 floats.  A wave's step is
// 3 TM TN matrix instructions on 2 (TM + TN) LDS reads: the matrix pipe is what it waits for, from 64 x 64 a wave on.
template <int BM, int BN, int WM, int WN, int KG, int STAGES, bool GELU>
__device__ __forceinline__ void f32_split_tile(BT_F32_SPLIT_FIRST, const F32SplitTail &tail) {
  constexpr int NG = WM * WN, NW = NG * KG, WTM = BM / WM, WTN = BN / WN, TM = WTM / 16, TN = WTN / 16;
  constexpr int NI = (BM + BN) / 8 / NG, NIA = BM / 8 / NG;   // every group loads its own k-steps
  constexpr int STEP_HALFS = (BM + BN) * kBK, STAGE_HALFS = KG * STEP_HALFS;
  static_assert(BM % (8 * NG) == 0 && BN % (8 * NG) == 0, "tile rows must split evenly over the waves");
  static_assert(WTN % 32 == 0, "whole blocks of pairs");
  extern __shared__ __attribute__((aligned(1024))) half_t split_smem[];
  const int lane = threadIdx.x & 63;
  const int wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int group = KG > 1 ? wave_all / NG : 0, wave = wave_all % NG;
  const int M = valid_rows ? min(scalar_load(valid_rows), rows_cap) : rows_cap;
  int tile_m, tile_n;
  {
    // XCD x works on a contiguous range of the live tiles
    const int tiles_n = (N + BN - 1) / BN, live = (M + BM - 1) / BM * tiles_n, per = (live + 7) >> 3;
    const int bid = (int)blockIdx.x, L = (bid & 7) * per + (bid >> 3);
    if (bid >= per * 8 || L >= live) return;
    tile_m = (int)divide((unsigned)L, (unsigned)tiles_n, per_n);
    tile_n = L - tile_m * tiles_n;
  }
  const int m0 = tile_m * BM, n0 = tile_n * BN, nk = K / 32 / KG;   // k-steps of a group: group, group + KG, ...
  const size_t pitch = 2 * (size_t)K;   // halfs
  // (dead rows read as zero: the ones of the last tile would come from HBM, where nothing of this call is)
  const rsrc_t rs_a = make_rsrc(a + m0 * pitch, (M - m0) * pitch * sizeof(half_t));
  const rsrc_t rs_w = make_rsrc(w + n0 * pitch, (N - n0) * pitch * sizeof(half_t));
  int voff[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    // (BM rows further on the swizzle is the same, and so the offsets of the two operands)
    const int r = ((i < NIA ? i : i - NIA) * NG + wave) * 8 + (lane >> 3);
    voff[i] = (r * 2 * K + (((lane & 7) ^ swz(r)) << 3)) * (int)sizeof(half_t);
  }
  auto issue = [&](int kt, int stage) {
#pragma unroll
    for (int i = 0; i < NI; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          i < NIA ? rs_a : rs_w,
          (__attribute__((address_space(3))) void *)(split_smem + stage * STAGE_HALFS + group * STEP_HALFS + (i * NG + wave) * 8 * kBK),
          16, voff[i], (kt * KG + group) * kBK * (int)sizeof(half_t), 0, 0);
  };
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < nk) issue(s, s);

  const int wm = wave / WN, wn = wave % WN, fr = lane & 15, lg = lane >> 4;
  // hh, cross: the products of one chunk of the weight's column, then scaled and added to `sum`.  (In one chain over all of k
  // the largest error of a result was up to 1.8 times that of the bfloat16 triples, whose waves share k.)
  float4_t sum[TN][TM], hh[TN][TM], cross[TN][TM];
  const float4_t zero4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) sum[i][j] = hh[i][j] = cross[i][j] = zero4;
  // The weight's scales: behind the ring, factor[c][n] = 2^(e - exponent of chunk c of column n), e[n] the smallest of the
  // column's, so that no factor is above 1.  (They are on their way beside the first k-steps.)
  const int chunks = (K + kSplitChunk - 1) / kSplitChunk;
  float *factor = (float *)(split_smem + STAGES * STAGE_HALFS);
  int *column_e = (int *)factor + chunks * BN;
  // ... the columns' bias, the rows' exponents and whether they hold floats: looked at behind the last k-step (in registers
  // from before it on, the 256 x 128 tile spilled)
  int *row_e = column_e + BN;
  float *column_bias = (float *)(row_e + 2 * BM);
  static_assert(BM <= NW * 64 && BN <= NW * 64, "a thread each");
  int e_of_row = 0, raw_of_row = 0;
  if ((int)threadIdx.x < BM) {
    const size_t m = min(m0 + (int)threadIdx.x, M - 1);
    e_of_row = a_exps[m], raw_of_row = tail.a_raw ? (int)tail.a_raw[m * split_raw_words(K)] : 0;
  }
  if (const int n = threadIdx.x; n < BN) {
    const int *from = w_exps + min(n0 + n, N - 1);
    int least = 1 << 20, mark = 0;
    for (int c = 0; c < chunks; ++c) {
      const int e = split_unmarked(from[(size_t)c * N]);
      mark |= split_marked(from[(size_t)c * N]) ? kSplitMark : 0;
      least = min(least, e);
      ((int *)factor)[c * BN + n] = e;
    }
    for (int c = 0; c < chunks; ++c) factor[c * BN + n] = __builtin_amdgcn_ldexpf(1.f, least - ((int *)factor)[c * BN + n]);
    column_e[n] = least + mark;
    column_bias[n] = tail.bias ? tail.bias[min(n0 + n, N - 1)] : 0.f;
  }
  if ((int)threadIdx.x < BM) row_e[threadIdx.x] = e_of_row, row_e[BM + threadIdx.x] = raw_of_row;
  __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): there, behind the first barrier of the loop
  constexpr int kFold = kSplitChunk / 32 / KG;   // k-steps of a group in a chunk
  const float *my_factor = factor + wn * WTN + 4 * lg;
  auto fold = [&](int chunk) {
#pragma unroll
    for (int i = 0; i < TN; ++i) {
      const float4_t f = *(const float4_t *)(my_factor + chunk * BN + 16 * i);
#pragma unroll
      for (int j = 0; j < TM; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          sum[i][j][e] = __builtin_fmaf(__builtin_fmaf(cross[i][j][e], kSplitLow, hh[i][j][e]), f[e], sum[i][j][e]);
    }
  };
  // (swz does not depend on the 16-row block, so a fragment's address is this plus a constant)
  const int at_h = fr * kBK + ((lg ^ swz(fr)) << 3), at_l = fr * kBK + (((4 + lg) ^ swz(fr)) << 3);

  int stage = 0;
  for (int kt = 0; kt < nk; ++kt) {
    if (kt % kFold == 0 && kt > 0) {
      fold(kt / kFold - 1);
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) hh[i][j] = cross[i][j] = zero4;
    }
    wait_stages<NI, STAGES - 2>(nk - 1 - kt);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();   // k-step kt is in LDS; the stage of the step before is free
    asm volatile("" ::: "memory");
    if (kt + STAGES - 1 < nk) {
      int ps = stage + STAGES - 1;
      if (ps >= STAGES) ps -= STAGES;
      issue(kt + STAGES - 1, ps);
    }
    const half_t *sA = split_smem + stage * STAGE_HALFS + group * STEP_HALFS + wm * WTM * kBK;
    const half_t *sW = split_smem + stage * STAGE_HALFS + group * STEP_HALFS + (BM + wn * WTN) * kBK;
    half8_t ah[TM], al[TM], wh[2], wl[2];
    auto read_w = [&](int i) {
      wh[i & 1] = *(const half8_t *)(sW + i * 16 * kBK + at_h);
      wl[i & 1] = *(const half8_t *)(sW + i * 16 * kBK + at_l);
    };
    auto read_a = [&](int j) {
      ah[j] = *(const half8_t *)(sA + j * 16 * kBK + at_h);
      al[j] = *(const half8_t *)(sA + j * 16 * kBK + at_l);
    };
    auto times = [&](int i, int j, int part) {   // hh, wh al, wl ah
      float4_t &to = part ? cross[i][j] : hh[i][j];
      to = __builtin_amdgcn_mfma_f32_16x16x32_f16(part == 2 ? wl[i & 1] : wh[i & 1], part == 1 ? al[j] : ah[j], to, 0, 0, 0);
    };
    // The waves of a workgroup come from their barrier together, so reads that all products wait for would leave the
    // matrix pipe idle for as long as the LDS takes to serve them: the first column block starts on the first row block's
    // reads, those of the others come between its products.
    read_w(0), read_a(0);
    times(0, 0, 0), times(0, 0, 1);
#pragma unroll
    for (int j = 1; j < TM; ++j) {
      read_a(j);
      times(0, j - 1, 2), times(0, j, 0), times(0, j, 1);
    }
    if (TN > 1) read_w(1);
    times(0, TM - 1, 2);
#pragma unroll
    for (int i = 1; i < TN; ++i) {
      if (i + 1 < TN) read_w(i + 1);
#pragma unroll
      for (int part = 0; part < 3; ++part)
#pragma unroll
        for (int j = 0; j < TM; ++j) times(i, j, part);
    }
    __builtin_amdgcn_sched_group_barrier(kSchedLdsRead, 6, 0);   // (one row block ahead)
    __builtin_amdgcn_sched_group_barrier(kSchedMfma, 2, 0);
    __builtin_amdgcn_sched_group_barrier(kSchedLdsRead, 2, 0);   // (of row block 2, or of column block 1)
#pragma unroll
    for (int j = 2; j < TM; ++j) {
      __builtin_amdgcn_sched_group_barrier(kSchedMfma, 3, 0);
      __builtin_amdgcn_sched_group_barrier(kSchedLdsRead, 2, 0);
    }
    __builtin_amdgcn_sched_group_barrier(kSchedMfma, 4, 0);
#pragma unroll
    for (int i = 1; i < TN; ++i) {
      if (i + 1 < TN) {
        __builtin_amdgcn_sched_group_barrier(kSchedMfma, 1, 0);
        __builtin_amdgcn_sched_group_barrier(kSchedLdsRead, 1, 0);
        __builtin_amdgcn_sched_group_barrier(kSchedMfma, 1, 0);
        __builtin_amdgcn_sched_group_barrier(kSchedLdsRead, 1, 0);
        __builtin_amdgcn_sched_group_barrier(kSchedMfma, 3 * TM - 2, 0);
      } else {
        __builtin_amdgcn_sched_group_barrier(kSchedMfma, 3 * TM, 0);
      }
    }
    if (++stage == STAGES) stage = 0;
  }
  fold((nk - 1) / kFold);

  // Two groups share the rows of their sums: each hands over the blocks that are the other's and adds what it gets.
  constexpr int kFirstRows = KG > 1 ? (TM + 1) / 2 : TM;   // row blocks of group 0
  static_assert(KG <= 2, "two groups at most");
  if (KG > 1) {
    static_assert(KG == 1 || (size_t)NG * TN * TM * 256 * sizeof(float) <= (size_t)STAGES * STAGE_HALFS * sizeof(half_t), "sums fit the ring");
    float4_t *shared = (float4_t *)split_smem + wave * (TN * TM * 64) + lane;
    __builtin_amdgcn_s_barrier();   // everyone is done with the ring
#pragma unroll
    for (int j = 0; j < TM; ++j)
      if ((j < kFirstRows) != (group == 0))
#pragma unroll
        for (int i = 0; i < TN; ++i) shared[(i * TM + j) * 64] = sum[i][j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < TM; ++j)
      if ((j < kFirstRows) == (group == 0))
#pragma unroll
        for (int i = 0; i < TN; ++i) sum[i][j] += shared[(i * TM + j) * 64];
  }

  // lane: columns n .. n + 3 of block i, row m of block j
  int ea[TM];
  unsigned holds_floats[TM];
#pragma unroll
  for (int j = 0; j < TM; ++j) {
    const int r = wm * WTM + 16 * j + fr;
    ea[j] = row_e[r], holds_floats[j] = (unsigned)row_e[BM + r];
  }
  bool column = false;   // one of the wave's columns is marked
#pragma unroll
  for (int i = 0; i < TN; ++i) {
    const int4_t marks = *(const int4_t *)(column_e + wn * WTN + 16 * i + 4 * lg);
#pragma unroll
    for (int e = 0; e < 4; ++e) column = column || (split_marked(marks[e]) && n0 + wn * WTN + 16 * i + 4 * lg < N);
  }
  constexpr int EP = 2 * WTN + 8;   // halfs of a staged row of pairs
  static_assert(!GELU || (size_t)NW * 16 * EP <= (size_t)STAGES * STAGE_HALFS, "staging fits the ring");
  half_t *staged = split_smem + wave_all * 16 * EP;
  column = __builtin_amdgcn_ballot_w64(column) != 0;
  // Rows that the pairs do not give: marked ones, those under a marked column, and those with a sum that is not finite.
  // (Dead rows hold what the scratch held before, and do not count.)
  unsigned again[TM], any = 0;
#pragma unroll
  for (int j = 0; j < TM; ++j) {
    again[j] = 0;
    if (KG > 1 && (j < kFirstRows) != (group == 0)) continue;
    const int m = m0 + wm * WTM + 16 * j + fr;
    float none[2] = {0.f, 0.f};   // (0 . x is NaN where x is not finite)
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) none[e & 1] = __builtin_fmaf(sum[i][j][e], 0.f, none[e & 1]);
    const bool wrong = column || split_marked(ea[j]) || holds_floats[j] != 0 || none[0] + none[1] != 0.f;
    const unsigned long long rows = __builtin_amdgcn_ballot_w64(wrong && m < M);
    again[j] = (unsigned)(rows | rows >> 16 | rows >> 32 | rows >> 48) & 0xffffu;
    any |= again[j];
  }
  if (__builtin_expect(any != 0, 0)) {
    // (What only this needs is read from the arguments here: held in registers from the start, it pushed others of the loop out.)
    typedef const __attribute__((address_space(4))) char *arguments_t;
    arguments_t late = (arguments_t)__builtin_amdgcn_kernarg_segment_ptr() + kF32SplitFirstBytes;
    asm volatile("" : "+s"(late));
    const F32SplitTail rare = *(const __attribute__((address_space(4))) F32SplitTail *)late;
    // (one copy of the code, a column block or two at a time, in the registers that the ring's loop leaves: whose sums they
    // are is picked behind it)
    constexpr int CN = TN > 2 ? 2 : 1;
#pragma unroll 1
    for (int at = 0; at < TM * (TN / CN); ++at) {
      const int j = at / (TN / CN), c = at % (TN / CN);
      unsigned rows = again[0];
#pragma unroll
      for (int q = 1; q < TM; ++q) rows = q == j ? again[q] : rows;
      if (rows == 0) continue;
      float4_t formed[CN];
      split_sums_of_floats<CN>(a, w, a_exps, w_exps, rare, N, K, min(m0 + wm * WTM + 16 * j + fr, M - 1),
                               n0 + wn * WTN + 16 * CN * c, fr, lg, formed);
#pragma unroll
      for (int q = 0; q < TM; ++q)
#pragma unroll
        for (int i = 0; i < TN; ++i)
          if (q == j && i / CN == c && (rows >> fr & 1)) sum[i][q] = formed[i % CN];
    }
  }
  asm volatile("" ::: "memory");   // (read once more: kept from before, sixteen registers that the sums of floats want)
  int4_t ew[TN];
  float4_t bias[TN];
#pragma unroll
  for (int i = 0; i < TN; ++i) {
    bias[i] = *(const float4_t *)(column_bias + wn * WTN + 16 * i + 4 * lg);
    ew[i] = *(const int4_t *)(column_e + wn * WTN + 16 * i + 4 * lg);
#pragma unroll
    for (int e = 0; e < 4; ++e) ew[i][e] = split_unmarked(ew[i][e]);
  }
  if (GELU) __builtin_amdgcn_s_barrier();   // everyone is done with the ring
#pragma unroll
  for (int j = 0; j < TM; ++j) {
    if (KG > 1 && (j < kFirstRows) != (group == 0)) continue;
    const int m_first = m0 + wm * WTM + 16 * j, m = m_first + fr, m_in = min(m, M - 1);
    const bool formed = again[j] >> fr & 1;   // (not scaled)
    const int e_row = split_unmarked(ea[j]);
    float to_pair = 1.f;
    if (GELU) to_pair = split_power(tail.gelu_exps[m_in]);
#pragma unroll
    for (int i = 0; i < TN; ++i) {
      const int n = n0 + wn * WTN + 16 * i + 4 * lg;
      float4_t v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = __builtin_amdgcn_ldexpf(sum[i][j][e], formed ? 0 : -(e_row + ew[i][e]));
      v += bias[i];
      if (!GELU) {
        if (m < M && n < N) store_through((float *)out + (size_t)m * N + n, __builtin_bit_cast(uint4_t, v));
        continue;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = f32_gelu(v[e]);
      sum[i][j] = v;
    }
    if (GELU) {
      // Floats stay where the pairs hold three results from kGeluFloor on no longer, or one where all are small.  Rows
      // whose bound is below 2^9, as ordinary ones are, lose none of those and are through with a comparison.
      bool raw = false, some_raw = false;
      if (tail.raw && __builtin_amdgcn_ballot_w64(to_pair * kGeluFloor < kSplitHeldFrom && m < M) != 0) {
        int lost = 0;
        float most = 0.f;
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float v = n0 + wn * WTN + 16 * i + 4 * lg < N ? sum[i][j][e] : 0.f, scaled = v * to_pair;
            lost += !split_pair(scaled).held(scaled) && __builtin_fabsf(v) >= kGeluFloor ? 1 : 0;
            most = fmaxf(most, __builtin_fabsf(scaled));
          }
#pragma unroll
        for (int o = 16; o < 64; o <<= 1) lost += __shfl_xor(lost, o, 64), most = fmaxf(most, __shfl_xor(most, o, 64));
        raw = m < M && (lost >= 3 || (lost > 0 && most < 1.0f / 256));
        some_raw = __builtin_amdgcn_ballot_w64(raw) != 0;
        const int n_first = n0 + wn * WTN;
        if (raw && lg == 0) {
          unsigned *words = tail.raw + (size_t)m * split_raw_words(N);
          words[0] = 1;
#pragma unroll
          for (int n = n_first; n < n_first + WTN; n += 32)
            if (n < N) atomicOr(words + 1 + (n >> 10), 1u << (n >> 5 & 31));
        }
      }
#pragma unroll
      for (int i = 0; i < TN; ++i) {
        half_t *to = staged + fr * EP + (i >> 1) * 64;
        const int at = (i & 1) * 16 + 4 * lg;
        half4_t h, l;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const SplitPair p = split_pair(sum[i][j][e] * to_pair);
          h[e] = p.h, l[e] = p.l;
        }
        *(half4_t *)(to + at) = h;
        *(half4_t *)(to + 32 + at) = l;
      }
      if (some_raw) {
        asm volatile("" ::: "memory");   // (over the pairs, of which all are there before)
        if (raw)
#pragma unroll
          for (int i = 0; i < TN; ++i)
            *(float4_t *)((float *)(staged + fr * EP + (i >> 1) * 64) + (i & 1) * 16 + 4 * lg) = sum[i][j];
      }
      constexpr int CPR = WTN / 4, RPS = 64 / CPR;   // 16-byte chunks of a row; rows per store instruction
      static_assert(64 % CPR == 0 && 16 % RPS == 0, "whole rows");
#pragma unroll
      for (int r = lane / CPR; r < 16; r += RPS) {
        const int c = lane % CPR, n = n0 + wn * WTN + (c >> 3) * 32;
        const uint4_t v = *(const uint4_t *)(staged + r * EP + c * 8);
        if (m_first + r < M && n < N)
          store_through((half_t *)out + (size_t)(m_first + r) * 2 * N + (n0 + wn * WTN) * 2 + c * 8, v);
      }
    }
  }
}
#endif  // __HIP_DEVICE_COMPILE__

template <int BM, int BN, int WM, int WN, int KG, int STAGES, bool GELU>
__global__ __launch_bounds__(WM *WN *KG * 64, WM *WN *KG == 8 && BN == 64 ? 4 : 2)
void f32_split_gemm_kernel(BT_F32_SPLIT_FIRST, F32SplitTail tail) {
#if defined(__HIP_DEVICE_COMPILE__)
  f32_split_tile<BM, BN, WM, WN, KG, STAGES, GELU>(a, w, valid_rows, a_exps, w_exps, out, rows_cap, N, K, per_n, tail);
#endif
}

struct F32SplitArgs {
  const half_t *a, *w;
  const int *valid_rows, *a_exps, *w_exps;
  void *out;
  int rows_cap, N, K;
  F32SplitTail tail;
};
template <int BM, int BN, int KG, int STAGES>
size_t f32_split_lds(int k) {
  return (size_t)KG * STAGES * (BM + BN) * kBK * sizeof(half_t) + (size_t)((k + kSplitChunk - 1) / kSplitChunk + 2) * BN * 4 + 2 * BM * 4;
}
template <int BM, int BN, int WM, int WN, int KG, int STAGES>
int launch_f32_split(const F32SplitArgs &p, hipStream_t s) {
  const size_t smem = f32_split_lds<BM, BN, KG, STAGES>(p.K);
  const int tiles_n = (p.N + BN - 1) / BN;
  const unsigned grid = (unsigned)(((long long)((p.rows_cap + BM - 1) / BM) * tiles_n + 7) / 8 * 8);
  const auto with = [&](auto gelu) {
    return Launch<f32_split_gemm_kernel<BM, BN, WM, WN, KG, STAGES, gelu()>>::on(
        s, "f32_split_gemm_kernel", grid, WM * WN * KG * 64, smem, p.a, p.w, p.valid_rows, p.a_exps, p.w_exps, p.out, p.rows_cap, p.N,
        p.K, inverse_of((unsigned)tiles_n), p.tail);
  };
  return p.tail.gelu_exps ? with(std::true_type{}) : with(std::false_type{});
}

}  // namespace
}  // namespace bt

using namespace bt;

extern "C" int bt_split_f32(int weight_count, const void *const *w, void *const *w_pairs, int *const *w_exps, const int *k,
                            const int *n, int bounded, const void *bounded_bias, float *bounds, const void *rows,
                            void *row_pairs, int *row_exps, const int *row_index, const int *valid_rows, int rows_cap,
                            int hidden_dim, void *stream) {
  return bt_split_f32_layer(weight_count, w, w_pairs, w_exps, k, n, bounded, bounded_bias, bounds, rows, row_pairs, row_exps,
                            row_index, valid_rows, rows_cap, hidden_dim, 0, stream);
}

static int split_f32(SplitArgs a, int weight_count, const void *const *w, void *const *w_pairs, int *const *w_exps, const int *k,
                     const int *n, int bounded, const void *bounded_bias, float *bounds, const void *rows, void *row_pairs,
                     int *row_exps, const int *row_index, const int *valid_rows, int rows_cap, int hidden_dim, int layer,
                     void *stream) {
  const char *who = "bt_split_f32";
  BT_REQUIRE(weight_count >= 0 && weight_count <= 4, BT_ERR_INVALID_ARGUMENT, "%s: weight_count=%d outside [0, 4]", who, weight_count);
  BT_REQUIRE(weight_count == 0 || (w && w_pairs && w_exps && k && n), BT_ERR_INVALID_ARGUMENT, "%s: null pointer argument", who);
  BT_REQUIRE(bounded < weight_count && (bounded < 0 || (bounded_bias && bounds)), BT_ERR_INVALID_ARGUMENT,
             "%s: bounded=%d needs a weight, its bias and an array of bounds", who, bounded);
  int units = 0;
  for (int i = 0; i < weight_count; ++i) {
    BT_REQUIRE(w[i] && w_pairs[i] && w_exps[i], BT_ERR_INVALID_ARGUMENT, "%s: null pointer of matrix %d", who, i);
    BT_REQUIRE(aligned16({w[i], w_pairs[i], w_exps[i]}), BT_ERR_INVALID_ARGUMENT, "%s: pointers must be 16-byte aligned", who);
    BT_REQUIRE(k[i] > 0 && n[i] > 0 && k[i] % 64 == 0 && n[i] % kSplitCols == 0, BT_ERR_UNSUPPORTED,
               "%s: k=%d must be a multiple of 64 and n=%d of 32", who, k[i], n[i]);
    const int strips = n[i] / kSplitCols;
    units += strips * ((k[i] + kSplitChunk - 1) / kSplitChunk);
    a.weight[i] = SplitWeight{(const float *)w[i], (half_t *)w_pairs[i], w_exps[i], k[i], n[i], strips, units};
  }
  a.count = weight_count, a.units = units;
  a.bounded = bounded < 0 ? -1 : bounded, a.bias = (const float *)bounded_bias, a.bounds = bounds;
  a.layer = layer;
  int row_blocks = 0;
  if (rows) {
    BT_REQUIRE(row_pairs && row_exps && row_pairs != rows, BT_ERR_INVALID_ARGUMENT, "%s: rows need an area of their own for the pairs", who);
    BT_REQUIRE(aligned16({rows, row_pairs}), BT_ERR_INVALID_ARGUMENT, "%s: pointers must be 16-byte aligned", who);
    BT_REQUIRE(rows_cap >= 0 && hidden_dim > 0 && hidden_dim % 32 == 0, BT_ERR_UNSUPPORTED,
               "%s: hidden_dim=%d must be a multiple of 32", who, hidden_dim);
    BT_REQUIRE(!row_index || valid_rows, BT_ERR_INVALID_ARGUMENT, "%s: row_index needs valid_rows", who);
    a.rows = (const float *)rows, a.row_pairs = (half_t *)row_pairs, a.row_exps = row_exps;
    a.row_index = row_index, a.valid_rows = valid_rows, a.rows_cap = rows_cap, a.hidden = hidden_dim;
    row_blocks = (rows_cap + kSplitThreads / 64 - 1) / (kSplitThreads / 64);
  }
  a.row_blocks = row_blocks;
  if (units + row_blocks == 0) return BT_OK;
  if (a.mask) return Launch<split_f32_kernel<kMaskF32>>::on(as_stream(stream), who, units + row_blocks, kSplitThreads, 0, a);
  return Launch<split_f32_kernel<kMaskNone>>::on(as_stream(stream), who, units + row_blocks, kSplitThreads, 0, a);
}

extern "C" int bt_split_f32_layer(int weight_count, const void *const *w, void *const *w_pairs, int *const *w_exps,
                                  const int *k, const int *n, int bounded, const void *bounded_bias, float *bounds,
                                  const void *rows, void *row_pairs, int *row_exps, const int *row_index,
                                  const int *valid_rows, int rows_cap, int hidden_dim, int layer, void *stream) {
  return split_f32(SplitArgs{}, weight_count, w, w_pairs, w_exps, k, n, bounded, bounded_bias, bounds, rows, row_pairs, row_exps,
                   row_index, valid_rows, rows_cap, hidden_dim, layer, stream);
}

extern "C" int bt_split_f32_layer_mask_rows(int weight_count, const void *const *w, void *const *w_pairs, int *const *w_exps,
                                            const int *k, const int *n, int bounded, const void *bounded_bias, float *bounds,
                                            const void *rows, void *row_pairs, int *row_exps, const void *atten_mask,
                                            int batch_size, int seq_len, int *batch_idx, int *word_idx, int *seq_order,
                                            int hidden_dim, void *stream) {
  const char *who = "bt_split_f32_layer_mask_rows";
  BT_REQUIRE(rows && atten_mask && batch_idx, BT_ERR_INVALID_ARGUMENT, "%s: null pointer argument", who);
  BT_REQUIRE(bt_gemm_qkv_mask_rows_supported(batch_size, seq_len, BT_F32), BT_ERR_UNSUPPORTED,
             "%s: batch_size=%d seq_len=%d is outside what bt_gemm_qkv_mask_rows_supported allows", who, batch_size, seq_len);
  BT_REQUIRE(aligned16({atten_mask}), BT_ERR_INVALID_ARGUMENT, "%s: tensor pointers must be 16-byte aligned", who);
  SplitArgs a{};
  a.mask = atten_mask, a.mask_B = batch_size, a.mask_S = seq_len;
  a.out_batch_idx = batch_idx, a.out_word_idx = word_idx, a.out_seq_order = seq_order;
  return split_f32(a, weight_count, w, w_pairs, w_exps, k, n, bounded, bounded_bias, bounds, rows, row_pairs, row_exps, nullptr,
                   nullptr, batch_size * seq_len, hidden_dim, 1, stream);
}

extern "C" int bt_gemm_f32_split(const void *a_pairs, const int *a_exps, const void *w_pairs, const int *w_exps, const void *bias,
                                 void *c, const int *gelu_exps, const int *valid_rows, int rows_cap, int n, int k,
                                 void *stream) {
  return bt_gemm_f32_split_with(a_pairs, a_exps, w_pairs, w_exps, bias, c, gelu_exps, valid_rows, rows_cap, n, k, nullptr, stream);
}

extern "C" int bt_gemm_f32_split_with(const void *a_pairs, const int *a_exps, const void *w_pairs, const int *w_exps,
                                      const void *bias, void *c, const int *gelu_exps, const int *valid_rows, int rows_cap,
                                      int n, int k, const bt_f32_split_more *more, void *stream) {
  const char *who = "bt_gemm_f32_split";
  BT_REQUIRE(a_pairs && a_exps && w_pairs && w_exps && c, BT_ERR_INVALID_ARGUMENT, "%s: null pointer argument", who);
  BT_REQUIRE(aligned16({a_pairs, w_pairs, w_exps, c}), BT_ERR_INVALID_ARGUMENT, "%s: pointers must be 16-byte aligned", who);
  BT_REQUIRE(rows_cap >= 0 && n > 0 && k > 0 && n % 32 == 0 && k % 64 == 0, BT_ERR_UNSUPPORTED,
             "%s: n=%d must be a multiple of 32 and k=%d of 64", who, n, k);
  BT_REQUIRE(k <= (1 << 14), BT_ERR_UNSUPPORTED, "%s: k=%d is beyond 2^14", who, k);   // (the scales of its chunks lie in LDS)
  BT_REQUIRE(!gelu_exps || bias, BT_ERR_INVALID_ARGUMENT, "%s: gelu needs a bias", who);
  if (rows_cap == 0) return BT_OK;
  const bt_f32_split_more none{}, &m = more ? *more : none;
  BT_REQUIRE(!m.raw || gelu_exps, BT_ERR_INVALID_ARGUMENT, "%s: floats among the pairs of a result that is not pairs", who);
  BT_REQUIRE(aligned16({m.a, m.w}), BT_ERR_INVALID_ARGUMENT, "%s: pointers must be 16-byte aligned", who);
  const F32SplitArgs p{(const half_t *)a_pairs, (const half_t *)w_pairs, valid_rows, a_exps, w_exps, c, rows_cap, n, k,
                       {(const float *)bias, gelu_exps, m.raw, m.a_raw, (const float *)m.w, (const float *)m.a, m.a_row_index}};
  hipStream_t s = as_stream(stream);
  // Tiles: 0: 64x64, two groups of waves over k, two workgroups a CU | 1: 64x128 likewise, one | 2: 96x128, one group, two.
  // What a step waits for is its operands: a CU takes in about 40 bytes a clock from the L2 and reads 128 from the LDS, and
  // the larger the tile the fewer it needs, as long as no CU goes without.  us at 2458 rows of hidden 768, bt_gemm_f32 and
  // tiles 0 / 1 / 2: QKV 57 and 41 / 46 / 28, projection 21 and 13.1 / 12.6 / 17.4, FFN1 77 and 61 / 69 / 49, FFN2 68 and 40 /
  // 45 / 62.  (256x128, eight waves: 38 / 33 / 40 / 103, but 71 for FFN1 from 2561 rows on, a second round: below;
  // 128x128, eight waves: 44 / 21 / 46 / 63.)  A launch is priced by its rounds of the chip, a last one
  // that is partly full where two workgroups share a CU at half of one and half of its share: 5 us less than these
  // and those of 600 and 4915 rows, give or take 15 %.  The groups add up in another order, so the choice follows from sizes
  // alone, never from a row hint, and where the count is known in some calls only, from the capacity of all (tile_rows);
  // a padded batch counts as 60 % full, give or take a fifth.
  int tile = option_f32_gemm_tile();
  if (tile < 0 || tile > 2) {
    struct Candidate { int bm, bn, per_cu; float step, fixed; };   // of a round: us per 64 of k, and besides
    static const Candidate candidates[3] = {{64, 64, 2, 0.66f, 7.f}, {64, 128, 1, 0.74f, 6.8f}, {96, 128, 2, 1.8f, 5.4f}};
    const long long capacity = m.tile_rows > 0 ? m.tile_rows : rows_cap;
    const long long rows = valid_rows ? (capacity * 3LL + 4) / 5 : capacity;
    float best = 0.f;
    for (int t = 0; t < 3; ++t) {
      const Candidate &c = candidates[t];
      float us = 0.f;
      for (int i = valid_rows ? 8 : 10; i <= (valid_rows ? 12 : 10); ++i) {
        const float load = (float)(((rows * i / 10 + c.bm - 1) / c.bm) * ((n + c.bn - 1) / c.bn)) / (float)(cu_count() * c.per_cu);
        const float full = floorf(load), part = load - full;
        us += (full + (part == 0.f ? 0.f : c.per_cu == 1 ? 1.f : 0.5f + 0.5f * part)) * (c.step * (float)(k / 64) + c.fixed);
      }
      if (t == 0 || us < best) best = us, tile = t;
    }
  }
  if (tile == 0) return launch_f32_split<64, 64, 2, 2, 2, 2>(p, s);
  if (tile == 1) return launch_f32_split<64, 128, 2, 2, 2, 2>(p, s);
  // 256x128 with eight waves, a workgroup a CU, gives the bits of 96x128 (the same order of a sum, the same columns a wave),
  // so what the caller knows of the live rows may decide: where one round of it takes the place of more than one of those
  // (FFN1 of 2458 rows, alone 51 -> 40 us, in a layer 51 -> 39; QKV there, one round either way, keeps the 96x128).
  const long long known = valid_rows ? m.rows_hint : rows_cap, tiles_n = (n + 127) / 128;
  if (known > 0 && (known + 255) / 256 * tiles_n <= cu_count() && (known + 95) / 96 * tiles_n > 2 * cu_count() &&
      option_f32_gemm_tile() < 0)
    return launch_f32_split<256, 128, 4, 2, 1, 2>(p, s);
  return launch_f32_split<96, 128, 2, 2, 1, 2>(p, s);
}
