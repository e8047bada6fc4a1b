// Shared API types of the BERT encoder-layer library, gfx950 build.
//
// Mirrors the public names of the reference's bytetransformer/include/common.h
// (OperationType, Traits, ET_Param, ModelType, ActType, the runtime-error
// convention of common.h:130-138) so that caller code written against the
// reference compiles against this header.  cuBLAS/CUDA types do not exist
// here: streams are hipStream_t and the BLAS-handle slots are opaque pointers
// that the library never dereferences (every GEMM is an in-tree MFMA kernel).
#pragma once
#include <hip/hip_fp16.h>
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdlib>
#include <stdexcept>
#include <string>

#include "bt_hip.h"

namespace bytetransformer {

enum class OperationType { FP32, HALF };

// Opaque stand-in for the reference's cublasHandle_t members.
typedef void *BlasHandle;

template <OperationType OpType>
class Traits;

template <>
class Traits<OperationType::FP32> {
 public:
  typedef float DataType;
  static const int dtype = BT_F32;
  static const int algo = -1;
};

template <>
class Traits<OperationType::HALF> {
 public:
  typedef __half DataType;
  static const int dtype = BT_F16;
  static const int algo = 99;
};

// Packed-token bookkeeping produced by the mask prefix sum.  valid_word_num is
// only filled in when the caller asked the offsets builder for it; the kernels
// read the count from batch_idx[batch_size] on the device.
typedef struct {
  int *batch_idx;
  int *word_idx;
  int valid_word_num;
} ET_Param;

// What a product in `slices` of k will read of a weight, for the attention's warm-up (prefetch_bytes in bt_hip.h): the
// XCDs' shares up to 256 expected rows, for which the products go column by column.
inline unsigned long long prefetch_weight(unsigned long long k, unsigned long long n, bool weight_kn, int slices, long long rows) {
  const unsigned long long bytes = k * n * 2, pitch = (weight_kn ? n : k) * 2;
  const int halvings = slices == 1 ? 0 : slices == 2 ? 1 : slices == 4 ? 2 : slices == 8 ? 3 : -1;
  if (rows > 256 || halvings < 0 || pitch % 64 || pitch / 64 > 0xffff || bytes >> 40) return bytes;
  const unsigned long long cols = weight_kn ? 3 - halvings : halvings;
  return bytes | pitch / 64 << 40 | cols << 56 | (weight_kn ? 0ull : 1ull) << 58;
}

// FFN2 with few rows and a long k runs as a split-k GEMM whose fp32 partial sums the last
// LayerNorm folds in (bt_gemm_splitk_rows / bt_splitk_layernorm).  This is the rule where the kernels
// library has no measurements (bt_gemm_splitk_slices): 4 splits up to 192 expected
// rows, 2 up to 640, none beyond, or when the partials of a launch of that
// capacity exceed the scratch area (4 splits of kSplitKMaxRows rows).  A whole layer in us with k whole / in two
// splits / in four, in stacks of 12 layers (hidden 768) and 24 whose weights no cache holds together; launched
// alone over and over, weights and rows warm, the split of the wide ones looks worse than it is here:
//   hidden 768:  192 rows  36.6 /  34.8 / 34.6; 576 rows  46.2 /  45.9; 640 rows  46.6 /  46.6; 704 rows  54.8 /  56.6
//   hidden 1024: 192 rows  48.1 /  46.7 / 44.4; 576 rows  67.3 /  64.7; 640 rows  68.8 /  65.3; 704 rows  70.1 /  73.7
//   hidden 1280: 192 rows  55.7 /  53.8 / 51.1; 512 rows  81.7 /  83.5; 640 rows  84.2 /  79.8; 704 rows  86.8 /  90.5
//   hidden 2048: 192 rows 100.4 /  92.0 / 88.1; 512 rows 126.8 / 129.9; 640 rows 152.7 / 146.6; 704 rows 155.5 / 174.8
// (weights as stored; pre-packed at 704 rows: hidden 768 49.8 / 51.9, hidden 1024 67.2 / 64.9)
constexpr int kSplitKMaxRows = 512;
inline int splitk_splits(long long rows_cap, long long rows_expected, int k) {
  static const bool enabled = [] {
    const char *e = std::getenv("BT_SPLITK");     // BT_SPLITK=0 turns the split-k path off
    return !(e && e[0] == '0');
  }();
  if (!enabled || k < 2048) return 1;
  if (rows_cap <= kSplitKMaxRows && rows_expected <= 192 && k % (4 * 64) == 0) return 4;
  if (rows_cap <= 2 * kSplitKMaxRows && rows_expected <= 640 && k % (2 * 64) == 0) return 2;
  return 1;
}
inline unsigned long long splitk_scratch_bytes(unsigned long long max_rows,
                                               unsigned long long hidden) {
  const unsigned long long rows = max_rows < (unsigned long long)kSplitKMaxRows
                                      ? max_rows
                                      : (unsigned long long)kSplitKMaxRows;
  return 4ull * rows * hidden * sizeof(float);   // (= 2 splits of up to twice as many rows)
}
// The slices of a layer's FFN2.  `area_bytes` = what the caller can give the partial sums: the activations
// that are dead by then and the scratch behind them.
// `all_live` = the launch has rows_cap rows, not a padded batch's share of them.
inline int ffn2_slices(int rows_cap, bool all_live, int n, int k, unsigned long long area_bytes) {
  const int rule = splitk_splits(rows_cap, all_live ? rows_cap : (rows_cap * 3LL + 4) / 5, k);
  if (k < 2048 || splitk_splits(1, 1, 2048) == 1) return rule;   // (short k, or turned off)
  const unsigned long long fit = area_bytes / ((unsigned long long)rows_cap * n * sizeof(float));
  const int slices = bt_gemm_splitk_slices(rows_cap, all_live ? 1 : 0, n, k, (int)(fit < 16 ? fit : 16));
  return slices > 0 ? slices : rule;
}

// Float layers on products of split operands (bt_gemm_f32_split): from how many rows the launches that split the
// weights, afresh in every layer, cost less than the products gain.  12 layers of hidden 768, split / not, us: 8 x 100
// (480 rows expected) 1512 / 1241, 8 x 160 (768) 1675 / 1336, 10 x 160 (960) 1756 / 1499, 10 x 200 (1200) 1873 / 1904,
// 16 x 128 (1229) 1881 / 2368, 16 x 256 (2458) 2336 / 3062; measured at this width alone.  Follows from sizes alone, never
// from a row hint: both ways are float arithmetic to a few 1e-7, but not the same bits.  From hidden 512 on: there the
// roundings of a sum outweigh those of the pairs, and the result is the nearer one to float64 (distance, pairs / whole
// floats: k = 64 9.8e-8 / 5.5e-8, 512 1.17e-07 / 1.71e-07).
inline bool f32_splits_operands(long long rows_cap, bool all_live, long long hidden, long long inter) {
  return hidden % 64 == 0 && inter % 64 == 0 && hidden >= 512 && hidden <= 4096 && inter <= (1 << 14) &&
         (all_live ? rows_cap : rows_cap * 3 / 5) >= 1220;
}
// What such a layer needs besides its activations: exponents of four sets of rows and of four weights' columns, the
// bounds of FFN1's, and the bits of FFN1's results that stay floats.
struct F32SplitScratch {
  int *x_exps, *att_exps, *ln_exps, *gelu_exps, *w_exps[4];
  float *bounds;
  unsigned *raw;
  int bound_count;
  // (a weight's column has an exponent for every 256 of its rows; a pair of bounds for every 32 columns of those)
  static unsigned long long chunks(unsigned long long k) { return (k + 255) / 256; }
  static unsigned long long bytes(unsigned long long rows, unsigned long long hidden, unsigned long long inter) {
    return (4 * ((rows + 3) / 4 * 4) + chunks(hidden) * (4 * hidden + inter) + chunks(inter) * hidden +
            chunks(hidden) * inter / 16 + rows * (1 + (inter + 1023) / 1024)) * 4;
  }
  F32SplitScratch(void *at, unsigned long long rows, int hidden, int inter) {
    rows = (rows + 3) / 4 * 4;
    int *p = (int *)at;
    const unsigned long long n[4] = {chunks(hidden) * 3 * hidden, chunks(hidden) * hidden, chunks(hidden) * inter, chunks(inter) * hidden};
    for (int i = 0; i < 4; ++i) w_exps[i] = p, p += n[i];
    x_exps = p, att_exps = p + rows, ln_exps = p + 2 * rows, gelu_exps = p + 3 * rows;
    bounds = (float *)(p + 4 * rows);
    bound_count = (int)(chunks(hidden) * inter / 32);
    raw = (unsigned *)(bounds + 2 * bound_count);
  }
};

// Row count that tiles are chosen for.  Without one from the caller the products take 60 % of the
// capacity for a guess and price a tile over 80-120 % of it, which is what a handful of sequence
// lengths spreads over; the mean of 32 or more lies within 7 % and is named as it is (batch 128 of up to
// 128 tokens, hidden 768: 2690 us for 12 layers, 2860 with tiles priced over the spread).
inline int rows_to_plan_for(int given, bool packed, int batch_size, long long rows) {
  if (given > 0 || !packed || batch_size < 32) return given;
  return (int)((rows * 3 + 4) / 5);
}

// Which of a padding-free fp16 layer's four products (QKV, projection, FFN1, FFN2; weights
// [k, n] as stored) run on a k-contiguous copy made afresh in the call, and by which launch:
// copy[i] - by the launch ahead of the layer (bt_layer_prologue), ln_copy[i] - by the first
// LayerNorm's launch (FFN1 and FFN2 only: the products behind it).  A product gets a copy
// when the measured tile table says it gains more than a microsecond beyond the cost of the
// copy.  `live` = expected valid tokens, `padded_rows` = batch x seq_len,
// `first_launch` = 0: the layer has a launch ahead of it in any case, 1: the QKV product could
// count the mask rows itself, so that a layer with nothing for a prologue to do goes without
// it, 2: it does so in any case; `ln_can_copy` = the LayerNorm's launch may carry copies.  Where the prologue is optional it is kept only if the copies that nothing
// else can make (QKV, projection) return what it costs (about 4 us with one round of tiles) -
// it then makes the others as well; without it the FFN copies ride in the LayerNorm's launch
// (or, if they may not, are dropped unless they pay for a prologue: up to 10 k padded rows
// never copying then wins 1.5-1.8 % per forward and loses as much beyond).
// `norm_in_ffn1`: FFN1's launch has the first LayerNorm in it and reads its weight as stored, so it gets no copy, and no
// LayerNorm's launch is there to make one.  Returns the number of prologue copies.
inline int plan_weight_copies(long long live, long long padded_rows, int hidden, int inter,
                              bool split_heads, int first_launch, bool ln_can_copy, bool copy[4],
                              bool ln_copy[4], bool norm_in_ffn1 = false) {
  ln_can_copy = ln_can_copy && !norm_in_ffn1;
  const int n[4] = {3 * hidden, hidden, inter, hidden}, k[4] = {hidden, hidden, hidden, inter};
  const int epilogue[4] = {split_heads ? BT_EPILOGUE_QKV_SPLIT : -1, BT_EPILOGUE_PLAIN,
                           BT_EPILOGUE_BIAS_GELU, BT_EPILOGUE_PLAIN};
  float gain[4] = {0.f, 0.f, 0.f, 0.f}, early = 0.f, total = 0.f;
  bool want[4], want_ln[4];
  for (int i = 0; i < 4; ++i) {
    if (epilogue[i] >= 0 && !(norm_in_ffn1 && i == 2)) gain[i] = bt_gemm_prepack_gain_us(live, n[i], k[i], epilogue[i]);
    want[i] = gain[i] > 1.0f;
    // (the table's gain is less the 0.5 us per megabyte that a copy costs the prologue; the LayerNorm's
    // launch makes one for half of that: 6.7 us without and 7.8 us with FFN1's 4.7 MB at batch 16 x 512)
    want_ln[i] = gain[i] + 0.25e-6f * (float)n[i] * (float)k[i] * 2.f > 1.0f;
    if (want[i]) total += gain[i];
    if (want[i] && i < 2) early += gain[i];
  }
  bool prologue = true;
  if (first_launch == 1)
    prologue = ln_can_copy ? early >= 4.0f : (padded_rows > 10240 ? total > 0.f : total >= 4.0f);
  if (first_launch == 2) prologue = false;
  int count = 0;
  for (int i = 0; i < 4; ++i) {
    copy[i] = prologue && want[i];
    // (measured where the table's gain is smallest, 1.5 us for FFN1 at batch 16 x 512: kernel time
    // -1 % per forward, wall time -0.5 % on one box and +0.6 % on another; with 4.5 us at
    // 16 x 1024, where the copy also replaces the prologue, -2 %)
    ln_copy[i] = !prologue && ln_can_copy && i >= 2 && want_ln[i];
    count += copy[i];
  }
  return count;
}

enum ModelType { Bert };

enum ActType { Relu, Sigmoid, SoftPlus, No };

// Turns a non-zero C-ABI status into the exception the reference's
// check_cuda_error raises (std::runtime_error, "[BT][ERROR] ..." prefix).
inline void check_status(int status, const char *file, int line) {
  if (status != BT_OK) {
    std::string msg = bt_last_error_string();
    if (msg.rfind("[BT][ERROR]", 0) != 0) msg = "[BT][ERROR] " + msg;
    throw std::runtime_error(msg + " " + file + ":" + std::to_string(line) + " \n");
  }
}

#define check_bt_error(val) ::bytetransformer::check_status((val), __FILE__, __LINE__)

}  // namespace bytetransformer
