// add-bias + residual + LayerNorm and FFN1 with its bias and GELU in one launch, for a few dozen rows.
#include "gemm_common.h"
#include "layernorm_row.h"

namespace bt {

constexpr int kLgRows = 16, kLgWaves = 8;

// A workgroup normalises 16 rows (two a wave, in registers as the LayerNorm launch has them), keeps them in LDS as one
// operand and multiplies them by COLS columns of the weight.  Every column tile of a row tile repeats the rows' work:
// what it costs is less than a launch and its gap, and the weight, whose fetch is most of FFN1's time here, is on its way
// meanwhile: it goes straight to registers, all of it requested at the head of the kernel behind the rows.
// (12 layers, operator, 1 x 32, one box: 329 -> 311 us; the two launches and this one at other sizes: lg_cols.)
//
// The waves share k; lane l of a wave has the W columns from W (l & 15) on at eight k, from 8 (l >> 4) on, of every 32: of
// a [K, N] weight W neighbouring halfs of eight k-rows, which make W operands of a 16x16x32 instruction in lane, of an
// [N, K] weight 16 bytes of each column.  Either way instruction j of the W has columns j, W + j, 2 W + j, ..., a lane's
// sums are 4 W neighbouring columns of a row, and the bits are the same.
template <int HIDDEN, int COLS>
struct LgShape {
  static constexpr int W = COLS / 16, KS = kLgWaves;   // columns a lane; slices of k
  static constexpr int KB = HIDDEN / KS / 32;          // 32 k at a time, of a wave's share
  static constexpr int PITCH = HIDDEN + 8;             // rows 16 bytes further on: 16 of them lie in different banks
  static constexpr size_t kRowBytes = (size_t)kLgRows * PITCH * sizeof(half_t);
  static constexpr size_t kLds = kRowBytes + (size_t)kLgRows * COLS * KS * sizeof(float);
  static_assert(HIDDEN % (32 * KS) == 0 && kRowBytes % 16 == 0 && kLds <= 160 * 1024, "whole shares of k");
};

#if defined(__HIP_DEVICE_COMPILE__)
// sizeof(T) bytes at `lane_bytes + scalar_bytes` of the descriptor.
template <typename T>
__device__ __forceinline__ T lg_load(rsrc_t rs, int lane_bytes, int scalar_bytes) {
  if constexpr (sizeof(T) == 16)
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b128(rs, lane_bytes, scalar_bytes, 0));
  else if constexpr (sizeof(T) == 8)
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(rs, lane_bytes, scalar_bytes, 0));
  else
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(rs, lane_bytes, scalar_bytes, 0));
}
#endif

template <int HIDDEN, int COLS, bool WKN>
__global__ __launch_bounds__(kLgWaves *kWave) void layernorm_gelu_kernel(
    const half_t *src, const half_t *residual, const int *residual_row_index, const int *valid_rows, const half_t *w,
    const half_t *bias, const half_t *gamma, const half_t *beta, half_t *dst, const half_t *ffn_bias, half_t *out,
    int rows_cap, int N, float eps, int unused) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef LgShape<HIDDEN, COLS> Sh;
  constexpr int W = Sh::W, KB = Sh::KB, KS = Sh::KS, PITCH = Sh::PITCH;
  constexpr int V = HIDDEN % 512 == 0 ? 8 : 4, NC = HIDDEN / kWave / V;
  constexpr int kWaveRows = kLgRows / kLgWaves;
  typedef typename LnVec<V>::halfs vec_t;
  typedef _Float16 cols_t __attribute__((ext_vector_type(W)));
  static_assert(NC * V * kWave == HIDDEN, "a row fills the lanes");
  extern __shared__ __attribute__((aligned(1024))) half_t lg_smem[];

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int M = valid_rows ? min(scalar_load(valid_rows), rows_cap) : rows_cap;
  if (M <= 0) return;
  // XCD x (workgroups x, x + 8, ...) has the same eighth of the columns whatever the row count, as warm_slice deals it
  const int tiles_m = (M + kLgRows - 1) / kLgRows, tiles_n = N / COLS, per = tiles_n / 8, at = (int)blockIdx.x >> 3;
  const int column = divide_small(at, tiles_m);
  if (column >= per) return;
  const int tile_n = ((int)blockIdx.x & 7) * per + column, m0 = (at - column * tiles_m) * kLgRows, n0 = tile_n * COLS;

  // the rows (past the last live one, that one again: its results are not stored)
  vec_t av[kWaveRows][NC], rv[kWaveRows][NC], bias_v[NC], gamma_v[NC], beta_v[NC];
  int row[kWaveRows], from[kWaveRows];
#pragma unroll
  for (int i = 0; i < kWaveRows; ++i) from[i] = row[i] = min(m0 + wave * kWaveRows + i, M - 1);
  if (residual_row_index) {
#pragma unroll
    for (int i = 0; i < kWaveRows; ++i) from[i] = scalar_load(residual_row_index + row[i]);
  }
  const auto load_row = [&](const half_t *tensor, int r, vec_t (&to)[NC]) {
    const rsrc_t rs = make_rsrc(tensor + (size_t)r * HIDDEN, HIDDEN * sizeof(half_t));
#pragma unroll
    for (int c = 0; c < NC; ++c)
      to[c] = lg_load<vec_t>(rs, lane * (int)sizeof(vec_t), c * kWave * (int)sizeof(vec_t));
  };
#pragma unroll
  for (int i = 0; i < kWaveRows; ++i) load_row(src, row[i], av[i]);
#pragma unroll
  for (int i = 0; i < kWaveRows; ++i) load_row(residual, from[i], rv[i]);
  load_row(bias, 0, bias_v);
  load_row(gamma, 0, gamma_v);
  load_row(beta, 0, beta_v);
  // the sums that wave q < W folds and stores
  const int fold_n = n0 + 4 * W * (lane >> 4) + 4 * min(wave, W - 1), fold_r = lane & 15;
  const half4_t ffn_bias_v = *(const half4_t *)(ffn_bias + fold_n);

  // the weight
  const int slice_k = wave * KB * 32, lane_n = W * (lane & 15), lane_k = 8 * (lane >> 4);
  // (one lane offset, the rest in scalars: with an address for every load this took 1.3 us of instructions)
  const size_t first = WKN ? (size_t)slice_k * N + n0 : (size_t)n0 * HIDDEN + slice_k;
  const rsrc_t rs_w = make_rsrc(w + first, ((size_t)HIDDEN * N - first) * sizeof(half_t));
  const int lane_at = (WKN ? lane_k * N + lane_n : lane_n * HIDDEN + lane_k) * (int)sizeof(half_t);
  cols_t rows_w[WKN ? KB : 1][8];
  half8_t cols_w[WKN ? 1 : KB][W];
#pragma unroll
  for (int b = 0; b < KB; ++b) {
    if constexpr (WKN) {
#pragma unroll
      for (int e = 0; e < 8; ++e) rows_w[b][e] = lg_load<cols_t>(rs_w, lane_at, (b * 32 + e) * N * (int)sizeof(half_t));
    } else {
#pragma unroll
      for (int j = 0; j < W; ++j) cols_w[b][j] = lg_load<half8_t>(rs_w, lane_at, (j * HIDDEN + b * 32) * (int)sizeof(half_t));
    }
  }
  __builtin_amdgcn_sched_barrier(0);   // (all requested before the first row is waited for)

  constexpr float kInverse = 1.0f / (float)HIDDEN;
  bool live[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) live[c] = true;
#pragma unroll
  for (int i = 0; i < kWaveRows; ++i) {
    float v[NC][V];
    const float rstd = ln_statistics<NC, V>(av[i], rv[i], bias_v, live, kInverse, eps, v);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      vec_t y;
#pragma unroll
      for (int j = 0; j < V; ++j) y[j] = (half_t)(v[c][j] * rstd * (float)gamma_v[c][j] + (float)beta_v[c][j]);
      *(vec_t *)(lg_smem + (wave * kWaveRows + i) * PITCH + (lane + c * kWave) * V) = y;
    }
  }
  __syncthreads();

  float4_t acc[W] = {};
#pragma unroll
  for (int b = 0; b < KB; ++b) {
    const half8_t fa = *(const half8_t *)(lg_smem + (lane & 15) * PITCH + slice_k + lane_k + b * 32);
#pragma unroll
    for (int j = 0; j < W; ++j) {
      half8_t fw;
      if constexpr (WKN) {
#pragma unroll
        for (int e = 0; e < 8; ++e) fw[e] = rows_w[b][e][j];
      } else {
        fw = cols_w[b][j];
      }
      acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fw, fa, acc[j], 0, 0, 0);
    }
  }

  // fold: acc[j][v] is column 4 W (lane >> 4) + W v + j of row lane & 15; four neighbouring columns of a lane are quad h,
  // which wave h adds up over the slices
  float4_t *sums = (float4_t *)((char *)lg_smem + Sh::kRowBytes);
#pragma unroll
  for (int h = 0; h < W; ++h) {
    float4_t four;
#pragma unroll
    for (int t = 0; t < 4; ++t) four[t] = acc[(4 * h + t) % W][(4 * h + t) / W];
    sums[(wave * W + h) * kWave + lane] = four;
  }
  __syncthreads();
  if (wave < W && m0 + fold_r < M) {
    float4_t v = sums[wave * kWave + lane];
#pragma unroll
    for (int s = 1; s < KS; ++s) v += sums[(s * W + wave) * kWave + lane];
    half4_t y;
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = (half_t)gelu_tanh_f32(v[e] + (float)ffn_bias_v[e]);
    store_through(out + (size_t)(m0 + fold_r) * N + fold_n, __builtin_bit_cast(uint2_t, y));
  }
  // the normalised rows, for the last LayerNorm: row r by column tile r, r + tiles_n, ...
  for (int r = tile_n; r < kLgRows && m0 + r < M; r += tiles_n)
    if ((int)threadIdx.x < HIDDEN / 8)
      store_through(dst + (size_t)(m0 + r) * HIDDEN + threadIdx.x * 8, *(const uint4_t *)(lg_smem + r * PITCH + threadIdx.x * 8));
#endif
}

// Columns of a tile, 0 where the two launches are the faster way: a workgroup repeats its rows' work, which pays while it
// has little of the weight to fetch (some 30 bytes a clock come to a CU) and its tiles fit one round of the chip with the
// rows that may be live (all of them, or 120 % of the expected share of a padded batch).  LayerNorm and FFN1, us as two
// launches / one with 32 columns / with 64: hidden 768, [K, N] weight, 32 rows 7.01 / 5.18 / 5.95, 48 rows 6.99 / 6.89 (two
// rounds) / 5.96, 80 rows 7.19 / - / 6.03, 96 rows 7.22 / - / 8.47 (two rounds); hidden 1024 32 rows 7.58 / 5.60 / 6.24, 64
// rows 7.60 / - / 6.34.  [N, K] weight, whose 64-byte pieces arrive more slowly: hidden 768 32 rows 6.12 / 5.03 / 6.44, 64
// rows 6.36 / 7.71 / 6.61; hidden 1024 32 rows 6.49 / 5.13 / 7.29.  Wider tiles for more rows: 128 columns 160 rows 8.19 / 7.67,
// 7.65 / 10.55 for [N, K]; 32 rows by 128 columns 256 rows 8.51 / 9.42, 8.26 / 11.34.
static int lg_cols(int rows_cap, int all_live, int n, int k, int weight_kn) {
  if ((k != 768 && k != 1024) || option_gemm_tile() >= 0) return 0;
  const long long rows = all_live ? rows_cap : (rows_cap * 18LL + 24) / 25;
  for (int cols = 32; cols <= (weight_kn ? 64 : 32); cols *= 2)
    if (n % (8 * cols) == 0 && n >= kLgRows * cols && (rows + kLgRows - 1) / kLgRows * (n / cols) <= cu_count()) return cols;
  return 0;
}

}  // namespace bt

using namespace bt;

extern "C" int bt_layernorm_gemm_bias_gelu_pays(int rows_cap, int all_live, int n, int k, int weight_kn) {
  static const bool have_gpu = [] {
    int devices = 0;
    return hipGetDeviceCount(&devices) == hipSuccess && devices > 0;
  }();
  if (rows_cap <= 0 || n <= 0 || !have_gpu) return 0;
  return lg_cols(rows_cap, all_live, n, k, weight_kn) != 0;
}

extern "C" int bt_layernorm_gemm_bias_gelu(const void *src, const void *residual, const int *residual_row_index,
                                           const void *bias, const void *gamma, const void *beta, void *dst, const void *w,
                                           const void *ffn_bias, void *out, const int *valid_rows, int rows_cap, int all_live,
                                           int n, int hidden_dim, int weight_kn, float eps, void *stream) {
  const char *who = "bt_layernorm_gemm_bias_gelu";
  BT_REQUIRE(src && residual && bias && gamma && beta && dst && w && ffn_bias && out, BT_ERR_INVALID_ARGUMENT,
             "%s: null pointer argument", who);
  BT_REQUIRE(dst != src && dst != residual, BT_ERR_INVALID_ARGUMENT,
             "%s: many workgroups read src and residual, dst must be another tensor", who);
  BT_REQUIRE(rows_cap >= 0 && n > 0, BT_ERR_INVALID_ARGUMENT, "%s: rows_cap=%d n=%d", who, rows_cap, n);
  BT_REQUIRE(!residual_row_index || valid_rows, BT_ERR_INVALID_ARGUMENT, "%s: residual_row_index needs valid_rows", who);
  BT_REQUIRE(aligned16({src, residual, bias, gamma, beta, dst, w, ffn_bias, out}), BT_ERR_INVALID_ARGUMENT,
             "%s: tensor pointers must be 16-byte aligned", who);
  if (rows_cap == 0) return BT_OK;
  const int cols = lg_cols(rows_cap, all_live, n, hidden_dim, weight_kn);
  BT_REQUIRE(cols, BT_ERR_UNSUPPORTED, "%s: %d rows of hidden_dim %d times %d columns are outside what "
             "bt_layernorm_gemm_bias_gelu_pays allows", who, rows_cap, hidden_dim, n);
  const unsigned grid = (unsigned)((rows_cap + kLgRows - 1) / kLgRows * (n / cols));
  const auto launch = [&](auto hidden, auto width, auto kn) {
    return Launch<layernorm_gelu_kernel<hidden(), width(), kn()>>::on(
        as_stream(stream), who, grid, kLgWaves * kWave, LgShape<hidden(), width()>::kLds, (const half_t *)src,
        (const half_t *)residual, residual_row_index, valid_rows, (const half_t *)w, (const half_t *)bias, (const half_t *)gamma,
        (const half_t *)beta, (half_t *)dst, (const half_t *)ffn_bias, (half_t *)out, rows_cap, n, eps, 0);
  };
  using std::integral_constant;
  const auto by_tile = [&](auto hidden) {
    if (cols == 64) return launch(hidden, integral_constant<int, 64>{}, std::true_type{});
    return weight_kn ? launch(hidden, integral_constant<int, 32>{}, std::true_type{})
                     : launch(hidden, integral_constant<int, 32>{}, std::false_type{});
  };
  return hidden_dim == 768 ? by_tile(integral_constant<int, 768>{}) : by_tile(integral_constant<int, 1024>{});
}
