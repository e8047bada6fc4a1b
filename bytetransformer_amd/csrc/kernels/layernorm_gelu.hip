// add-bias + residual + LayerNorm and FFN1 with its bias and GELU in one launch, for a few dozen rows.
#include "gemm_common.h"
#include "layernorm_row.h"

namespace bt {

constexpr int kLgRows = 16, kLgWaves = 8;

// A workgroup normalises 16 rows (two a wave, in registers as the LayerNorm launch has them), keeps them in LDS as one
// operand and multiplies them by COLS columns of the weight.  Every column tile of a row tile repeats the rows' work:
// what it costs is less than a launch and its gap, and the weight, whose fetch is most of FFN1's time here, is on its way
// meanwhile: all of it is requested, straight into LDS, at the head of the kernel behind the rows.
// (12 layers, operator, 1 x 32, one box: 330 -> 310 us.  With the weight in registers, each wave an eighth of k, the launch took
// 0.2 to 0.4 us longer, hidden 768, 32 rows 5.28 / 5.04 for a [K, N] weight and 5.01 / 4.68 for [N, K], and added up in an
// order of its own.)
//
// The results are, bit for bit, those of the two launches: a sum is formed in the order of the product that these sizes
// would get (product_takes_wave_k).  SLICED: tile 14's, four slices of k, every fourth step of 64 each, added up in the end
// and the bias behind them; a wave has a slice of half the columns.  Else that of all other tiles, one chain over k from the
// bias on; four waves have 16 columns each.  (A 16x16x32 instruction gives the bits of two 32x32x16 ones.)
template <int HIDDEN, int COLS>
struct LgShape {
  static constexpr int ROW_HALFS = kLgRows * HIDDEN, WEIGHT_HALFS = HIDDEN * COLS;
  static constexpr size_t kOperands = (size_t)(ROW_HALFS + WEIGHT_HALFS) * sizeof(half_t);
  static constexpr size_t kSums = (size_t)4 * kLgRows * COLS * sizeof(float);   // of the slices
  static constexpr bool kSumsApart = kOperands + kSums <= 160 * 1024;           // else in the weight's place
  static constexpr size_t kLds = kOperands + (kSumsApart ? kSums : 0);
  static constexpr int LOADS = WEIGHT_HALFS / 512 / kLgWaves;   // 1 KB a wave's instruction
  static_assert(HIDDEN % 256 == 0 && (COLS == 32 || COLS == 64) && kLds <= 160 * 1024, "whole rounds of the waves, LDS budget");
  static_assert(kSums <= (size_t)WEIGHT_HALFS * sizeof(half_t), "sums fit the weight's place");
};

// Where chunk c (16 bytes) of row r of the normalised rows lies: 16 rows of one chunk, what a pass of the operand's reads
// takes, are in 16 places of the 256 bytes that the banks hold.
__device__ __forceinline__ int lg_chunk(int r, int c) { return c ^ r; }

template <int HIDDEN, int COLS, bool WKN, bool SLICED>
__global__ __launch_bounds__(kLgWaves *kWave) void layernorm_gelu_kernel(
    const half_t *src, const half_t *residual, const int *residual_row_index, const int *valid_rows, const half_t *w,
    const half_t *bias, const half_t *gamma, const half_t *beta, half_t *dst, const half_t *ffn_bias, half_t *out,
    int rows_cap, int N, float eps, int unused) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef LgShape<HIDDEN, COLS> Sh;
  constexpr int V = HIDDEN % 512 == 0 ? 8 : 4, NC = HIDDEN / kWave / V;
  constexpr int kWaveRows = kLgRows / kLgWaves;
  typedef typename LnVec<V>::halfs vec_t;
  static_assert(NC * V * kWave == HIDDEN, "a row fills the lanes");
  static_assert(WKN || COLS == 32, "an [N, K] image is laid out for 32 columns");
  extern __shared__ __attribute__((aligned(1024))) half_t lg_smem[];
  half_t *rows = lg_smem, *weight = lg_smem + Sh::ROW_HALFS;

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
    for (int c = 0; c < NC; ++c) {
      if constexpr (V == 8)
        to[c] = __builtin_bit_cast(vec_t, __builtin_amdgcn_raw_buffer_load_b128(rs, lane * 16, c * kWave * 16, 0));
      else
        to[c] = __builtin_bit_cast(vec_t, __builtin_amdgcn_raw_buffer_load_b64(rs, lane * 8, c * kWave * 8, 0));
    }
  };
#pragma unroll
  for (int i = 0; i < kWaveRows; ++i) load_row(src, row[i], av[i]);
#pragma unroll
  for (int i = 0; i < kWaveRows; ++i) load_row(residual, from[i], rv[i]);
  load_row(bias, 0, bias_v);
  load_row(gamma, 0, gamma_v);
  load_row(beta, 0, beta_v);
  // wave t < COLS / 16 stores columns 16 t + 4 (lane >> 4) .. + 3 of row lane & 15
  const int out_r = lane & 15, out_n = n0 + 16 * min(wave, COLS / 16 - 1) + 4 * (lane >> 4);
  const half4_t ffn_bias_v = *(const half4_t *)(ffn_bias + out_n);

  // the weight: instruction i of wave v lands KB 8 i + v of the image, a lane offset and the rest in scalars.  [K, N]: its k-rows
  // of COLS columns (swz_kn); [N, K]: for every 64 k a tile of 32 columns (swz)
  {
    const rsrc_t rs = WKN ? make_rsrc(w + n0, ((size_t)HIDDEN * N - n0) * sizeof(half_t))
                          : make_rsrc(w + (size_t)n0 * HIDDEN, (size_t)(N - n0) * HIDDEN * sizeof(half_t));
    int lane_at, step;   // bytes; from one instruction to the next
    if constexpr (WKN) {
      lane_at = kn_load_offset<COLS>(wave, lane, N, COLS);
      step = 4096 / COLS * N * (int)sizeof(half_t);
    } else {
      const int col = (wave & 3) * 8 + (lane >> 3);
      lane_at = (col * HIDDEN + (wave >> 2) * 64 + (((lane & 7) ^ swz(col)) << 3)) * (int)sizeof(half_t);
      step = 128 * (int)sizeof(half_t);
    }
#pragma unroll
    for (int i = 0; i < Sh::LOADS; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void *)(weight + (8 * i + wave) * 512), 16,
                                               lane_at, i * step, 0, 0);
  }
  __builtin_amdgcn_sched_barrier(0);   // (all requested before the first row is waited for)

  constexpr float kInverse = 1.0f / (float)HIDDEN;
  bool live[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) live[c] = true;
#pragma unroll
  for (int i = 0; i < kWaveRows; ++i) {
    const int r = wave * kWaveRows + i;
    float v[NC][V];
    const float rstd = ln_statistics<NC, V>(av[i], rv[i], bias_v, live, kInverse, eps, v);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      vec_t y;
#pragma unroll
      for (int j = 0; j < V; ++j) {
        float f = v[c][j] * rstd * (float)gamma_v[c][j] + (float)beta_v[c][j];
        asm("" : "+v"(f));   // a float, then a half, as in the LayerNorm launch: not v_fma_mixlo_f16, which rounds once
        y[j] = (half_t)f;
      }
      const int k = (lane + c * kWave) * V;
      *(vec_t *)(rows + r * HIDDEN + lg_chunk(r, k >> 3) * 8 + (k & 7)) = y;
    }
  }
  wait_vmcnt<0>();   // (the weight of this wave)
  __syncthreads();

  // 32 k from k0 on: 16 columns from column n of the tile, and the rows
  const auto columns = [&](int n, int k0) {
    if constexpr (WKN) return load_kn_frag<COLS>(weight, n, k0, lane);
    const int col = n + (lane & 15), chunk = (k0 & 63) / 8 + (lane >> 4);
    return *(const half8_t *)(weight + (k0 >> 6) * (32 * 64) + col * 64 + ((chunk ^ swz(col)) << 3));
  };
  const auto operand = [&](int k0) {
    return *(const half8_t *)(rows + (lane & 15) * HIDDEN + lg_chunk(lane & 15, k0 / 8 + (lane >> 4)) * 8);
  };
  float4_t v;
  if constexpr (SLICED) {
    constexpr int G = COLS / 32;   // 16 columns each, of a wave
    const int slice = wave & 3, half = wave >> 2;
    float4_t acc[G] = {};
#pragma unroll
    for (int u = 0; u < HIDDEN / 128; ++u) {
      const int k0 = (u >> 1) * 256 + slice * 64 + (u & 1) * 32;
      const half8_t fa = operand(k0);
#pragma unroll
      for (int g = 0; g < G; ++g)
        acc[g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(columns((half * G + g) * 16, k0), fa, acc[g], 0, 0, 0);
    }
    if (!Sh::kSumsApart) __syncthreads();   // everyone is done with the weight
    float4_t *sums = (float4_t *)(Sh::kSumsApart ? weight + Sh::WEIGHT_HALFS : weight);
#pragma unroll
    for (int g = 0; g < G; ++g) sums[(slice * 2 * G + half * G + g) * kWave + lane] = acc[g];
    __syncthreads();
    if (wave < 2 * G) {
      v = sums[wave * kWave + lane];
#pragma unroll
      for (int s = 1; s < 4; ++s) v += sums[(s * 2 * G + wave) * kWave + lane];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += (float)ffn_bias_v[e];
    }
  } else if (wave < COLS / 16) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = (float)ffn_bias_v[e];
#pragma unroll
    for (int k0 = 0; k0 < HIDDEN; k0 += 32)
      v = __builtin_amdgcn_mfma_f32_16x16x32_f16(columns(wave * 16, k0), operand(k0), v, 0, 0, 0);
  }
  if (wave < COLS / 16 && m0 + out_r < M) {
    half4_t y;
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = (half_t)gelu_tanh_f32(v[e]);
    store_through(out + (size_t)(m0 + out_r) * N + out_n, __builtin_bit_cast(uint2_t, y));
  }
  // the normalised rows, for the last LayerNorm: row r by column tile r, r + tiles_n, ...
  for (int r = tile_n; r < kLgRows && m0 + r < M; r += tiles_n)
    if ((int)threadIdx.x < HIDDEN / 8)
      store_through(dst + (size_t)(m0 + r) * HIDDEN + threadIdx.x * 8,
                    *(const uint4_t *)(rows + r * HIDDEN + lg_chunk(r, threadIdx.x) * 8));
#endif
}

// Columns of a tile, 0 where the two launches are the faster way: a workgroup repeats its rows' work, which pays while it
// has little of the weight to fetch (some 30 bytes a clock come to a CU) and its tiles fit one round of the chip with the
// rows that may be live (all of them, or 120 % of the expected share of a padded batch).  LayerNorm and FFN1, us as two
// launches / one with 32 columns / with 64, from the rows on where 32 and 64 columns take a second round: hidden 768, [K, N]
// weight, 32 rows 7.06 / 5.08 / 5.64, 33 rows 6.74 / 6.79 / 5.67, 80 rows 7.20 / - / 5.77, 96 rows 7.21 / - / 9.27; hidden 1024
// 32 rows 7.55 / 5.48 / 6.17, 33 rows 7.23 / 8.41 / 6.19, 64 rows 7.57 / 9.00 / 6.22, 65 rows 7.80 / - / 10.36.  [N, K] weight: hidden
// 768 32 rows 6.21 / 4.69, 33 rows 6.26 / 6.25; hidden 1024 32 rows 6.42 / 4.79, 33 rows 6.76 / 7.95; 64 columns, whose 64-byte
// pieces came more slowly while the weight went to registers, were slower there than the two launches (32 rows 6.44 and 7.29)
// and have no image here.  Nor have other hidden sizes: these two are what has been measured.
static int lg_cols(int rows_cap, int all_live, int n, int k, int weight_kn) {
  if ((k != 768 && k != 1024) || option_gemm_tile() >= 0) return 0;
  const long long rows = all_live ? rows_cap : (rows_cap * 18LL + 24) / 25;
  for (int cols = 32; cols <= (weight_kn ? 64 : 32); cols *= 2) {
    // (32 columns of rows that fit one round here always fit one of tile 14, so one chain over k is built for 64 only)
    if (cols == 32 && !product_takes_wave_k(rows_cap, n, k)) continue;
    if (n % (8 * cols) == 0 && n >= kLgRows * cols && (rows + kLgRows - 1) / kLgRows * (n / cols) <= cu_count()) return cols;
  }
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
  // (what the two launches ask for: FFN1's bias is read a few halfs at a time)
  BT_REQUIRE(aligned16({src, residual, bias, gamma, beta, dst, w, out}), BT_ERR_INVALID_ARGUMENT,
             "%s: tensor pointers must be 16-byte aligned", who);
  if (rows_cap == 0) return BT_OK;
  const int cols = lg_cols(rows_cap, all_live, n, hidden_dim, weight_kn);
  BT_REQUIRE(cols, BT_ERR_UNSUPPORTED, "%s: %d rows of hidden_dim %d times %d columns are outside what "
             "bt_layernorm_gemm_bias_gelu_pays allows", who, rows_cap, hidden_dim, n);
  const unsigned grid = (unsigned)((rows_cap + kLgRows - 1) / kLgRows * (n / cols));
  const bool sliced = product_takes_wave_k(rows_cap, n, hidden_dim);
  const auto launch = [&](auto hidden, auto width, auto kn, auto slices) {
    return Launch<layernorm_gelu_kernel<hidden(), width(), kn(), slices()>>::on(
        as_stream(stream), who, grid, kLgWaves * kWave, LgShape<hidden(), width()>::kLds, (const half_t *)src,
        (const half_t *)residual, residual_row_index, valid_rows, (const half_t *)w, (const half_t *)bias, (const half_t *)gamma,
        (const half_t *)beta, (half_t *)dst, (const half_t *)ffn_bias, (half_t *)out, rows_cap, n, eps, 0);
  };
  using std::integral_constant;
  const auto by_tile = [&](auto hidden) {
    if (cols == 64)
      return sliced ? launch(hidden, integral_constant<int, 64>{}, std::true_type{}, std::true_type{})
                    : launch(hidden, integral_constant<int, 64>{}, std::true_type{}, std::false_type{});
    return weight_kn ? launch(hidden, integral_constant<int, 32>{}, std::true_type{}, std::true_type{})
                     : launch(hidden, integral_constant<int, 32>{}, std::false_type{}, std::true_type{});
  };
  return hidden_dim == 768 ? by_tile(integral_constant<int, 768>{}) : by_tile(integral_constant<int, 1024>{});
}
