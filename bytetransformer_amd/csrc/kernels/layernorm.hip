// add-bias + residual + LayerNorm, packed in place and packed -> padded with
// zero fill.  Memory-bound: one wave64 per row, 16-byte lanes, the row lives in
// registers between the two statistics passes, reductions are wave shuffles
// (no LDS, no block barrier).
//
// Numerics follow bytetransformer/include/layernorm.h:114-159,273-296,334-373:
// x = (out + residual) + bias with both adds rounded to fp16, mean and biased
// variance in fp32 (two-pass), y = (x - mean) * rsqrt(var + eps) * gamma + beta.
#include "layernorm_row.h"

namespace bt {

constexpr int kLnRowsPerBlock = 4;   // 2, 8 and 16 rows per workgroup measured 0-20 % slower

// Statistics and store of one row held in registers (x = (a + r) + bias, two fp16-rounded adds).
template <int NC, int V, bool GB32, bool kAffineEarly, int NG, typename H = typename LnVec<V>::halfs>
__device__ __forceinline__ void ln_finish(const H (&av)[NC], const H (&rv)[NC], const H (&bias_v)[NC],
                                          const H (&gh)[NC], const H (&bh)[NC],
                                          const float4_t (&g32)[NG][V / 4], const float4_t (&b32)[NG][V / 4],
                                          const void *gamma, const void *beta, const int (&cc)[NC],
                                          const bool (&live)[NC], half_t *o, float inv_n, float eps) {
  float v[NC][V];
  const float rstd = ln_statistics<NC, V>(av, rv, bias_v, live, inv_n, eps, v);

#pragma unroll
  for (int i = 0; i < NC; ++i) {
    float g[V], bt_[V];
    if (GB32) {
#pragma unroll
      for (int h = 0; h < V / 4; ++h) {
        const float4_t gv = kAffineEarly ? g32[kAffineEarly ? i : 0][h] : ((const float4_t *)gamma)[V / 4 * cc[i] + h];
        const float4_t bv = kAffineEarly ? b32[kAffineEarly ? i : 0][h] : ((const float4_t *)beta)[V / 4 * cc[i] + h];
#pragma unroll
        for (int j = 0; j < 4; ++j) g[4 * h + j] = gv[j], bt_[4 * h + j] = bv[j];
      }
    } else {
#pragma unroll
      for (int j = 0; j < V; ++j) {
        g[j] = (float)gh[i][j];
        bt_[j] = (float)bh[i][j];
      }
    }
    H y;
#pragma unroll
    for (int j = 0; j < V; ++j) y[j] = (half_t)(v[i][j] * rstd * g[j] + bt_[j]);
    if (live[i]) store_through(o + cc[i] * V, __builtin_bit_cast(typename LnVec<V>::bits, y));
  }
}

// SPLITS > 0: `src` holds SPLITS fp32 partial sums of the row ([SPLITS][split_rows][H], the
// output of a split-k GEMM); their sum, rounded to fp16 once, takes the place of `out`.
//
// A launch of a few thousand rows is one round of waves, each living for the length of its
// chain of dependent memory accesses, so the kernel is written to keep that chain short:
// everything whose address does not depend on loaded data (bias, gamma, beta, the row
// index or the sequence offsets, and on packed rows the row of `src` itself) is requested
// at the top in one batch, a lane past the end of the row loads the last chunk again
// instead of branching, and the only dependent step left is the row(s) behind an index.
// The row is a wave's, so what finds it (count, offsets, index, addresses) is scalar.
//
// FULL: the row is exactly NC chunks of V halfs for each of the 64 lanes (hidden 768 as three of 4, 512 and 1024 as
// one and two of 8), so no lane holds a chunk that does not count: 12 elements a lane at hidden 768 instead of 16
// behind selects.  A launch of a few rows is the length of one wave.
template <int NC, int V, bool FULL, bool RESTORE, bool GB32, int SPLITS>
__device__ __forceinline__ void layernorm_block(
    int block, const half_t *src, const half_t *__restrict__ residual,
    const half_t *__restrict__ bias, const void *__restrict__ gamma,
    const void *__restrict__ beta, half_t *dst, const int *__restrict__ idx,
    const int *__restrict__ residual_row_index, int B, int S, int rows_cap, int split_rows,
    int hidden, float inv_n, float eps, unsigned per_s) {
  typedef typename LnVec<V>::halfs vec_t;
  typedef typename LnVec<V>::bits bits_t;
  const int r = block * kLnRowsPerBlock + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (r >= rows_cap) return;
  const int H = FULL ? NC * V * kWave : hidden, chunks = H / V;
  // fp32 gamma / beta of wide rows would not fit the registers next to the row: those
  // instantiations fetch them after the statistics, as before
  constexpr bool kAffineEarly = !GB32 || NC * V <= 16;

  int cc[NC];        // this lane's chunks, clamped into the row
  bool live[NC];
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int c = lane + i * kWave;
    live[i] = FULL || c < chunks;
    cc[i] = live[i] ? c : chunks - 1;
  }

  // ---- first batch: nothing here depends on loaded data ----
  vec_t bias_v[NC];
  vec_t gh[NC], bh[NC];
  float4_t g32[kAffineEarly && GB32 ? NC : 1][V / 4], b32[kAffineEarly && GB32 ? NC : 1][V / 4];
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    bias_v[i] = ((const vec_t *)bias)[cc[i]];
    if (kAffineEarly) {
      if (GB32) {
#pragma unroll
        for (int h = 0; h < V / 4; ++h) {
          g32[i][h] = ((const float4_t *)gamma)[V / 4 * cc[i] + h];
          b32[i][h] = ((const float4_t *)beta)[V / 4 * cc[i] + h];
        }
      } else {
        gh[i] = ((const vec_t *)gamma)[cc[i]];
        bh[i] = ((const vec_t *)beta)[cc[i]];
      }
    }
  }
  auto row_of = [&](const half_t *tensor, size_t row, int i) { return ((const vec_t *)(tensor + row * H))[cc[i]]; };
  auto zero_row = [&](size_t row) {
    const vec_t z = {};
#pragma unroll
    for (int i = 0; i < NC; ++i)
      if (live[i]) store_through(dst + row * H + cc[i] * V, __builtin_bit_cast(bits_t, z));
  };

  size_t src_row = r, dst_row = r;
  vec_t av[NC], rv[NC];
  if (RESTORE && residual_row_index && SPLITS == 0) {
    // restore through the row map (word_idx of the offsets: entry r < M is the padded
    // position of packed row r, the entries from M on are the padded positions that stay
    // empty): only the store address depends on a loaded value, so the rows are requested
    // together with it.  idx = batch_idx, M = idx[B].
#pragma unroll
    for (int i = 0; i < NC; ++i) av[i] = row_of(src, src_row, i);
#pragma unroll
    for (int i = 0; i < NC; ++i) rv[i] = row_of(residual, src_row, i);
    dst_row = (size_t)scalar_load(residual_row_index + r);
    const int M = scalar_load(idx + B);
    if (r >= M) return zero_row(dst_row);
    ln_finish<NC, V, GB32, kAffineEarly>(av, rv, bias_v, gh, bh, g32, b32, gamma, beta, cc, live,
                                         dst + dst_row * H, inv_n, eps);
    return;
  }
  size_t res_row;
  if (RESTORE) {
    // r walks the padded [B, S] grid; idx = batch_idx
    const int b = (int)divide((unsigned)r, (unsigned)S, per_s), s = r - b * S;
    const int start = scalar_load(idx + b), len = scalar_load(idx + b + 1) - start;
    if (s >= len) return zero_row(dst_row);
    res_row = src_row = (size_t)start + s;
  } else {
    // idx = pointer to the live-row count (or null: all rows live): one scalar load, the same
    // address for every wave of the launch, and the one thing a wave waits for before it asks
    // for its rows - the waves of the rows past the count (40 % of a launch sized for the
    // padded batch) would otherwise read 1.5 KB each for nothing.
    const int M = idx ? scalar_load(idx) : rows_cap;
    if (r >= M) return;
    res_row = residual_row_index ? (size_t)scalar_load(residual_row_index + src_row) : src_row;
  }
  if (SPLITS == 0) {
#pragma unroll
    for (int i = 0; i < NC; ++i) av[i] = row_of(src, src_row, i);
  }
#pragma unroll
  for (int i = 0; i < NC; ++i) rv[i] = row_of(residual, res_row, i);
  if (SPLITS > 0) {
#pragma unroll
    for (int i = 0; i < NC; ++i)
#pragma unroll
      for (int h = 0; h < V / 4; ++h) {
        const float4_t *pp = (const float4_t *)((const float *)src + src_row * H) + V / 4 * cc[i] + h;
        float4_t part = pp[0];
#pragma unroll
        for (int sp = 1; sp < SPLITS; ++sp) part += pp[(size_t)sp * split_rows * (H / 4)];
#pragma unroll
        for (int j = 0; j < 4; ++j) av[i][4 * h + j] = (half_t)part[j];
      }
  }

  ln_finish<NC, V, GB32, kAffineEarly>(av, rv, bias_v, gh, bh, g32, b32, gamma, beta, cc, live,
                                       dst + dst_row * H, inv_n, eps);
}

template <int NC, int V, bool FULL, bool RESTORE, bool GB32, int SPLITS>
__global__ __launch_bounds__(kLnRowsPerBlock *kWave) void layernorm_kernel(
    const half_t *src, const half_t *__restrict__ residual,
    const half_t *__restrict__ bias, const void *__restrict__ gamma,
    const void *__restrict__ beta, half_t *dst, const int *__restrict__ idx,
    const int *__restrict__ residual_row_index, int B, int S, int rows_cap, int split_rows,
    int hidden, float inv_n, float eps, unsigned per_s) {
  layernorm_block<NC, V, FULL, RESTORE, GB32, SPLITS>(blockIdx.x, src, residual, bias, gamma, beta, dst, idx,
                                                      residual_row_index, B, S, rows_cap, split_rows, hidden,
                                                      inv_n, eps, per_s);
}

// Calls `with` with the way that rows of H halfs are dealt to a wave as compile-time constants.
template <typename Then>
static int by_row_shape(int H, Then with) {
  using std::integral_constant;
  if (H == 768) return with(integral_constant<int, 3>{}, integral_constant<int, 4>{}, std::true_type{});
  if (H == 512) return with(integral_constant<int, 1>{}, integral_constant<int, 8>{}, std::true_type{});
  if (H == 1024) return with(integral_constant<int, 2>{}, integral_constant<int, 8>{}, std::true_type{});
  const int nc = (H / 8 + kWave - 1) / kWave;
  if (nc <= 1) return with(integral_constant<int, 1>{}, integral_constant<int, 8>{}, std::false_type{});
  if (nc <= 2) return with(integral_constant<int, 2>{}, integral_constant<int, 8>{}, std::false_type{});
  if (nc <= 4) return with(integral_constant<int, 4>{}, integral_constant<int, 8>{}, std::false_type{});
  return with(integral_constant<int, 8>{}, integral_constant<int, 8>{}, std::false_type{});
}

// The packed LayerNorm with k-contiguous weight copies riding along: the first `copy_blocks`
// workgroups of the grid move 64 x 64 tiles of the [K, N] matrices of `jobs` into their [N, K]
// copies (through LDS, as the layer's prologue launch does), the others are the LayerNorm's.
// A launch of a few thousand rows moves its 20 MB at half of what the memory system
// sustains, so the copy of a few MB costs this launch less than a launch of its own would,
// and the product behind it (FFN1) reads its weight k-contiguous.
template <int NC, int V, bool FULL, bool GB32>
__global__ __launch_bounds__(kLnRowsPerBlock *kWave) void layernorm_copy_kernel(
    const half_t *src, const half_t *__restrict__ residual,
    const half_t *__restrict__ bias, const void *__restrict__ gamma,
    const void *__restrict__ beta, half_t *dst, const int *__restrict__ idx,
    const int *__restrict__ residual_row_index, int rows_cap, int hidden, float inv_n, float eps,
    WeightJobs jobs, int copy_blocks) {
  static_assert(kLnRowsPerBlock * kWave == 256, "a tile is moved by 256 threads");
  if ((int)blockIdx.x < copy_blocks) {
    __shared__ half_t tiles[64][kTransposePitch];
    const int t_end = jobs.tile_end[jobs.count - 1];
    for (int t0 = blockIdx.x; t0 < t_end; t0 += copy_blocks)
      transpose_tiles_64<1>(jobs, t0, tiles, threadIdx.x);
    return;
  }
  layernorm_block<NC, V, FULL, false, GB32, 0>((int)blockIdx.x - copy_blocks, src, residual, bias, gamma,
                                               beta, dst, idx, residual_row_index, 0, 1, rows_cap, rows_cap,
                                               hidden, inv_n, eps, 0);
}

template <bool RESTORE, int SPLITS = 0>
static int launch_ln(const void *src, const void *residual, const void *bias, const void *gamma,
                     const void *beta, int gb32, void *dst, const int *idx,
                     const int *residual_row_index, int B, int S, int rows_cap, int H, float eps,
                     hipStream_t s, const char *who, int split_rows = 0) {
  BT_REQUIRE(H > 0 && H % 8 == 0, BT_ERR_UNSUPPORTED, "%s: hidden_dim %d must be a multiple of 8",
             who, H);
  BT_REQUIRE(aligned16({src, residual, bias, gamma, beta, dst}), BT_ERR_INVALID_ARGUMENT,
             "%s: tensor pointers must be 16-byte aligned", who);
  BT_REQUIRE(H <= 8 * 8 * kWave, BT_ERR_UNSUPPORTED, "%s: hidden_dim %d exceeds 4096", who, H);
  if (rows_cap == 0) return BT_OK;
  const int grid = (rows_cap + kLnRowsPerBlock - 1) / kLnRowsPerBlock;
  const float inv_n = 1.0f / (float)H;
  return by_row_shape(H, [&](auto nc, auto v, auto full) {
    const auto with = [&](auto affine32) {
      return Launch<layernorm_kernel<nc(), v(), full(), RESTORE, affine32(), SPLITS>>::on(
          s, who, grid, kLnRowsPerBlock * kWave, 0, (const half_t *)src, (const half_t *)residual, (const half_t *)bias,
          gamma, beta, (half_t *)dst, idx, residual_row_index, B, S, rows_cap, split_rows ? split_rows : rows_cap, H,
          inv_n, eps, inverse_of((unsigned)S));
    };
    return gb32 ? with(std::true_type{}) : with(std::false_type{});
  });
}

}  // namespace bt

using namespace bt;

extern "C" int bt_add_bias_residual_layernorm(void *out, const void *residual,
                                              const int *residual_row_index, const void *bias,
                                              const void *gamma, const void *beta,
                                              int gamma_beta_fp32, const int *valid_rows,
                                              int rows_cap, int hidden_dim, float eps,
                                              void *stream) {
  BT_REQUIRE(out && residual && bias && gamma && beta, BT_ERR_INVALID_ARGUMENT,
             "bt_add_bias_residual_layernorm: null pointer argument");
  BT_REQUIRE(rows_cap >= 0, BT_ERR_INVALID_ARGUMENT,
             "bt_add_bias_residual_layernorm: negative rows_cap");
  BT_REQUIRE(!residual_row_index || valid_rows, BT_ERR_INVALID_ARGUMENT,
             "bt_add_bias_residual_layernorm: residual_row_index needs valid_rows");
  return launch_ln<false>(out, residual, bias, gamma, beta, gamma_beta_fp32, out, valid_rows,
                          residual_row_index, 0, 1, rows_cap, hidden_dim, eps, as_stream(stream),
                          "bt_add_bias_residual_layernorm");
}

extern "C" int bt_add_bias_residual_layernorm_copy(
    void *out, const void *residual, const int *residual_row_index, const void *bias,
    const void *gamma, const void *beta, int gamma_beta_fp32, const int *valid_rows, int rows_cap,
    int hidden_dim, float eps, int weight_count, const void *const *w, void *const *wt,
    const int *k, const int *n, void *stream) {
  const char *who = "bt_add_bias_residual_layernorm_copy";
  BT_REQUIRE(out && residual && bias && gamma && beta, BT_ERR_INVALID_ARGUMENT,
             "%s: null pointer argument", who);
  BT_REQUIRE(rows_cap >= 0, BT_ERR_INVALID_ARGUMENT, "%s: negative rows_cap", who);
  BT_REQUIRE(!residual_row_index || valid_rows, BT_ERR_INVALID_ARGUMENT,
             "%s: residual_row_index needs valid_rows", who);
  WeightJobs jobs;
  const int rc = make_weight_jobs(who, &jobs, weight_count, w, wt, k, n, 0, nullptr, nullptr);
  if (rc != BT_OK) return rc;
  if (jobs.count == 0)
    return launch_ln<false>(out, residual, bias, gamma, beta, gamma_beta_fp32, out, valid_rows,
                            residual_row_index, 0, 1, rows_cap, hidden_dim, eps, as_stream(stream),
                            who);
  const int H = hidden_dim;
  BT_REQUIRE(H > 0 && H % 8 == 0, BT_ERR_UNSUPPORTED, "%s: hidden_dim %d must be a multiple of 8",
             who, H);
  BT_REQUIRE(aligned16({out, residual, bias, gamma, beta}), BT_ERR_INVALID_ARGUMENT,
             "%s: tensor pointers must be 16-byte aligned", who);
  BT_REQUIRE(H <= 8 * 8 * kWave, BT_ERR_UNSUPPORTED, "%s: hidden_dim %d exceeds 4096", who, H);
  // one tile per copying workgroup up to 1024 of them (a BERT-large FFN weight has 1024 tiles)
  const int tiles = jobs.tile_end[jobs.count - 1];
  const int copy_blocks = tiles < 1024 ? tiles : 1024;
  const int grid = copy_blocks + (rows_cap + kLnRowsPerBlock - 1) / kLnRowsPerBlock;
  const float inv_n = 1.0f / (float)H;
  hipStream_t s = as_stream(stream);
  return by_row_shape(H, [&](auto nc, auto v, auto full) {
    const auto with = [&](auto affine32) {
      return Launch<layernorm_copy_kernel<nc(), v(), full(), affine32()>>::on(
          s, who, grid, kLnRowsPerBlock * kWave, 0, (const half_t *)out, (const half_t *)residual, (const half_t *)bias,
          gamma, beta, (half_t *)out, valid_rows, residual_row_index, rows_cap, H, inv_n, eps, jobs, copy_blocks);
    };
    return gamma_beta_fp32 ? with(std::true_type{}) : with(std::false_type{});
  });
}

extern "C" int bt_add_bias_residual_layernorm_restore(
    const void *out, const void *residual, const void *bias, const void *gamma, const void *beta,
    int gamma_beta_fp32, void *out_padded, const int *batch_idx, const int *word_idx,
    int batch_size, int seq_len, int hidden_dim, float eps, void *stream) {
  BT_REQUIRE(out && residual && bias && gamma && beta && out_padded && batch_idx,
             BT_ERR_INVALID_ARGUMENT,
             "bt_add_bias_residual_layernorm_restore: null pointer argument");
  BT_REQUIRE(batch_size > 0 && seq_len > 0, BT_ERR_INVALID_ARGUMENT,
             "bt_add_bias_residual_layernorm_restore: sizes must be positive");
  BT_REQUIRE((long long)batch_size * seq_len < (1ll << 31), BT_ERR_UNSUPPORTED,
             "bt_add_bias_residual_layernorm_restore: too many rows");
  return launch_ln<true>(out, residual, bias, gamma, beta, gamma_beta_fp32, out_padded, batch_idx,
                         word_idx, batch_size, seq_len, batch_size * seq_len, hidden_dim, eps,
                         as_stream(stream), "bt_add_bias_residual_layernorm_restore");
}

extern "C" int bt_splitk_layernorm(const void *partials, int splits, const void *residual,
                                   const int *residual_row_index, const void *bias,
                                   const void *gamma, const void *beta, int gamma_beta_fp32,
                                   void *dst, const int *batch_idx, const int *valid_rows,
                                   int batch_size, int seq_len, int rows_cap, int hidden_dim,
                                   float eps, void *stream) {
  BT_REQUIRE(partials && residual && bias && gamma && beta && dst, BT_ERR_INVALID_ARGUMENT,
             "bt_splitk_layernorm: null pointer argument");
  BT_REQUIRE(splits >= 2 && splits <= 4, BT_ERR_UNSUPPORTED,
             "bt_splitk_layernorm: splits=%d (supported: 2, 3, 4)", splits);
  BT_REQUIRE(rows_cap >= 0, BT_ERR_INVALID_ARGUMENT, "bt_splitk_layernorm: negative rows_cap");
  hipStream_t s = as_stream(stream);
  if (batch_idx) {
    // restore mode: dst is the padded [batch_size, seq_len, hidden] output
    // rows_cap is the row count of one partial-sum slice (what bt_gemm_splitk was given)
    BT_REQUIRE(batch_size > 0 && seq_len > 0 && (long long)batch_size * seq_len < (1ll << 31) &&
                   rows_cap > 0 && rows_cap <= batch_size * seq_len,
               BT_ERR_INVALID_ARGUMENT,
               "bt_splitk_layernorm: restore needs 0 < rows_cap <= batch_size * seq_len");
    BT_REQUIRE(!residual_row_index, BT_ERR_INVALID_ARGUMENT,
               "bt_splitk_layernorm: no residual gather in restore mode");
    const int padded = batch_size * seq_len;
    const auto launch = splits == 2 ? launch_ln<true, 2> : splits == 3 ? launch_ln<true, 3> : launch_ln<true, 4>;
    return launch(partials, residual, bias, gamma, beta, gamma_beta_fp32, dst, batch_idx, nullptr, batch_size,
                  seq_len, padded, hidden_dim, eps, s, "bt_splitk_layernorm", rows_cap);
  }
  BT_REQUIRE(!residual_row_index || valid_rows, BT_ERR_INVALID_ARGUMENT,
             "bt_splitk_layernorm: residual_row_index needs valid_rows");
  const auto launch = splits == 2 ? launch_ln<false, 2> : splits == 3 ? launch_ln<false, 3> : launch_ln<false, 4>;
  return launch(partials, residual, bias, gamma, beta, gamma_beta_fp32, dst, valid_rows, residual_row_index, 0, 1,
                rows_cap, hidden_dim, eps, s, "bt_splitk_layernorm", 0);
}
