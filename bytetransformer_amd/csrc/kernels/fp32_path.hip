// The OperationType::FP32 flavour of the encoder layer on gfx950: every tensor
// is float and so is every accumulator.  Three kernels:
//
//   f32_gemm_kernel       C = A[M,K] . W[K,N] (+bias, +tanh-GELU), W row-major as the
//                         caller stores it (no pre-pack: a row-major W tile already is the
//                         MFMA "B" operand), optional row gather on A.  Role of the
//                         reference's cuBLAS calls for float (gemm.cu:32-39) and of
//                         gemm_bias_gelu<float> / add_bias_gelu<float>
//                         (gemm_bias_act.cu:24-75).
//   f32_attention_kernel  fused softmax(scale Q K^T + bias + (mask-1) 10000) V over
//                         token-major [rows, 3H] projections, K / V streamed in 32-key
//                         tiles with an online softmax.  Role of the unfused float path
//                         (attention_nofused.cu:27-114, softmax.h:25-60,103-140) without
//                         its [B,h,S,S] logits buffer and its four transposes.
//   f32_layernorm_kernel  add-bias + residual + LayerNorm, in place on packed rows or
//                         scattered to the padded layout with zero fill
//                         (layernorm.h:20-40, layernorm.cu:89-148 for float).
//
// fp32 MFMA runs at 1/16 of the bf16 rate: the products of the linear layers multiply each float as
// a sum of three bfloat16 instead (see below), the attention stays on v_mfma_f32_32x32x2_f32, compute
// bound with a trivial memory system (one LDS buffer pair, register-staged global loads).
#include "f32_split.h"

namespace bt {

typedef float float2_t __attribute__((ext_vector_type(2)));

namespace {

constexpr float kLog2eF = 1.4426950408889634f;
constexpr float kDeadLogit = -1.0e30f;

// ---------------------------------------------------------------------------
// float operands as bfloat16 triples
// ---------------------------------------------------------------------------
// A float has 24 significand bits, three bfloat16 have 3 x 8: x = h + m + l exactly, with
// h = bf16(x), m = bf16(x - h), l = bf16(x - h - m) (round to nearest, so |m| <= 2^-9 |x| and
// |l| <= 2^-18 |x|; both differences are exact).  That holds from 2^-110 on, where l is a multiple of
// the smallest bfloat16, 2^-133, up to the largest bfloat16; F32SumRange says what happens beyond.
// A product of two floats is then nine bf16
// products, each exact in the MFMA's float accumulator; the three smallest (m l, l m, l l: at most
// 2^-26 of the product) are below the rounding of a float product and are left out.  Six
// v_mfma_f32_32x32x16_bf16 do in 192 clocks what eight v_mfma_f32_32x32x2_f32 do in 512.
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

struct Bf16Triple {   // of two neighbouring elements: h, m and l as packed pairs
  unsigned h, m, l;
};
__device__ __forceinline__ unsigned pack_bf16(float a, float b) {
  return __builtin_bit_cast(unsigned, __builtin_convertvector(float2_t{a, b}, bf16x2_t));
}
__device__ __forceinline__ float bf16_low(unsigned p) { return __builtin_bit_cast(float, p << 16); }
__device__ __forceinline__ float bf16_high(unsigned p) {
  return __builtin_bit_cast(float, p & 0xffff0000u);
}
__device__ __forceinline__ Bf16Triple split_bf16(float a, float b) {
  Bf16Triple t;
  t.h = pack_bf16(a, b);
  const float ra = a - bf16_low(t.h), rb = b - bf16_high(t.h);
  t.m = pack_bf16(ra, rb);
  t.l = pack_bf16(ra - bf16_low(t.m), rb - bf16_high(t.m));
  return t;
}
__device__ __forceinline__ void split_bf16x8(bf16x8_t (&out)[3], const float (&x)[8]) {
  uint4_t v[3];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const Bf16Triple t = split_bf16(x[2 * j], x[2 * j + 1]);
    v[0][j] = t.h, v[1][j] = t.m, v[2][j] = t.l;
  }
#pragma unroll
  for (int pl = 0; pl < 3; ++pl) out[pl] = __builtin_bit_cast(bf16x8_t, v[pl]);
}
// acc += a . b over the 16 k of one step, smallest terms first
__device__ __forceinline__ float16_t mfma_triple(const bf16x8_t (&a)[3], const bf16x8_t (&b)[3],
                                                 float16_t acc) {
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[2], b[0], acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[2], acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[1], acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[0], acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[1], acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[0], acc, 0, 0, 0);
  return acc;
}

// ---------------------------------------------------------------------------
// GEMM
// ---------------------------------------------------------------------------
struct F32GemmArgs {
  const float *a;      // [rows_cap or more, K]
  const float *w;      // [K, N]
  const float *bias;   // [N] or null
  float *c;            // [rows_cap, N]
  const int *valid_rows;
  const int *a_row_index;   // optional gather: A row r is a[a_row_index[r]]
  int rows_cap, N, K;
  int gelu;
};

constexpr int kF32CUs = 256;
constexpr unsigned kF32MaxBytes = 0xffff0000u;   // the largest range that a tile addresses from one base
constexpr unsigned kF32Outside = 0xfffffff0u;   // an offset outside every descriptor: reads as zero
// Largest value over the 64 lanes (values >= 0), wave-uniform: the steps of wave_inclusive_sum.
__device__ __forceinline__ int wave_largest(int v) {
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false));
  return __builtin_amdgcn_readlane(v, 63);
}
template <int N>
__device__ __forceinline__ void f32_wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0F70);
}

// Where the split above does not hold, the sum shows it:
//   * an infinity, or a float past the largest bfloat16 (3.39e38), is no sum of three bfloat16: x - h is
//     inf - inf, and every sum that it enters comes out as NaN.  A product may also pass through an
//     infinity on the way to a finite sum.  A sum that is not finite is formed again.
//   * an operand below 2^-110 is taken to the nearest multiple of 2^-133.  Beside a sum of 2^-60 or more
//     that is lost in float's own rounding unless the other operand is above 2^38; a smaller sum is
//     formed again, except zero (rows of zeros are ordinary: padding).
// "Again" means from the floats themselves by float multiply-adds, whatever float arithmetic makes of
// them.  A launch that has such sums pays a chain of K for each.
// (By the bits without the sign, gathered over all the sums of a lane: 12 layers at batch 16 x 256 take
// 0.5 % longer than without the check, and 1.2 % longer with a branch for each sum.)
struct F32SumRange {
  unsigned largest = 0, smallest = ~0u;   // of 2 |bits|, and of 2 |bits| - 1: zero wraps to the top
  __device__ __forceinline__ void add(float x) {
    const unsigned twice = __builtin_bit_cast(unsigned, x) << 1;
    largest = max(largest, twice);
    smallest = min(smallest, twice - 1);
  }
  __device__ __forceinline__ bool split_held() const {
    constexpr unsigned kInf = 0x7f800000u << 1, kTiny = (127u - 60) << 24;   // of infinity and of 2^-60
    return largest < kInf && smallest >= kTiny - 1;
  }
};
template <int V>   // one column, or four neighbouring ones
__device__ __forceinline__ void f32_dot_again(const float *a_row, const float *w, int K, int N, float (&sum)[V]) {
#pragma unroll
  for (int v = 0; v < V; ++v) sum[v] = 0.f;
  for (int k = 0; k < K; k += 4) {
    const float4_t a = *(const float4_t *)(a_row + k);
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int v = 0; v < V; ++v) sum[v] = __builtin_fmaf(a[e], w[(size_t)(k + e) * N + v], sum[v]);
  }
}
__device__ __forceinline__ const float *f32_a_row(const F32GemmArgs &p, int m) {
  return p.a + (size_t)(p.a_row_index ? p.a_row_index[m] : m) * p.K;
}

// Store of one 32x32 block: accumulator element i is row 8*(i/4) + 4*half + i%4, column l32.
__device__ __forceinline__ void f32_store_block(const F32GemmArgs &p, const float16_t &acc, int m0,
                                                int n0, int M, int l32, int half) {
  const int col = n0 + l32;
  if (col >= p.N) return;
  const float bv = p.bias ? p.bias[col] : 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int row = m0 + 8 * (i >> 2) + 4 * half + (i & 3);
    if (row >= M) continue;
    float sum[1] = {acc[i]};
    F32SumRange range;
    range.add(sum[0]);
    if (!range.split_held()) f32_dot_again(f32_a_row(p, row), p.w + col, p.K, p.N, sum);
    float v = sum[0] + bv;
    if (p.gelu) v = f32_gelu(v);
    p.c[(size_t)row * p.N + col] = v;
  }
}

// One (32 MT) x (32 NT) tile per workgroup; its NW waves take the k range in turn, 16 k ("a slice")
// at a time, and their sums are folded through LDS at the end.  A wave shares nothing with the others
// until then: it copies its own slices global -> LDS (direct-to-LDS loads, no registers, no
// barrier anywhere in the loop) into a private ring of DEPTH slices, reads them back in MFMA order
// as floats and splits them into bf16 triples one slice ahead of the products.  Every element of
// the tile is read from LDS once and split once, which waves side by side on a shared tile would
// do two times each.  What bounds it is the issue port: a 64x64 tile's slice is 24 MFMAs (768 clocks of
// the matrix pipe) and 176 vector instructions of the split, and a SIMD issues them one after the
// other (an MFMA takes about 12 clocks of the port, a vector instruction 4).  2458 rows, hidden 768,
// before (v_mfma_f32_32x32x2_f32, tiles of 128x128 to 64x64) and now: QKV 92 -> 60 us, projection
// 39 -> 23, FFN1 114 -> 78, FFN2 137 -> 71 us (163 TFLOP/s); 32 rows: FFN2 121 -> 25 us.  Relative
// error against float64 at k = 3072: 9.9e-7 -> 4.3e-7.
//
// LDS image of a slice: A as TM rows of 16 floats, the 16-byte chunk of a row XORed with
// (row >> 2) & 3 (16 consecutive rows read one chunk from distinct banks); W as 16 k-rows of TN
// floats such that k-rows e and e + 8, which the two halves of a wave read together, lie on
// distinct banks (64 columns: the upper k-rows' columns XOR 32; 32 columns: the upper k-rows
// exchanged in pairs).
#if defined(__HIP_DEVICE_COMPILE__)
template <int MT, int NT, int NW, int DEPTH, bool RAGGED>
__device__ __forceinline__ void f32_gemm_tile(const F32GemmArgs &p) {
  constexpr int TM = 32 * MT, TN = 32 * NT;
  constexpr int NIA = TM / 16, NIW = TN / 16, NI = NIA + NIW;   // 1 KB load instructions per slice
  constexpr int SLICE = (TM + TN) * 16;                         // floats
  constexpr int ACC = TM * TN;                                  // floats of a wave's sums
  constexpr int REGION = DEPTH * SLICE > ACC ? DEPTH * SLICE : ACC;
  static_assert(NT == 1 || NT == 2, "the W image is laid out for 32 or 64 columns");
  extern __shared__ __attribute__((aligned(1024))) float f32_smem[];

  const int M = p.valid_rows ? min(*p.valid_rows, p.rows_cap) : p.rows_cap;
  int tile_m, tile_n;
  {
    const int tiles_m = (M + TM - 1) / TM, tiles_n = (p.N + TN - 1) / TN;
    const int live = tiles_m * tiles_n, per = (live + 7) >> 3;
    const int bid = (int)blockIdx.x, L = (bid & 7) * per + (bid >> 3);
    if (bid >= per * 8 || L >= live) return;
    if (live < kMostPanelTiles)
      tile_panels<TM, TN>(tiles_m, tiles_n, per).locate(L, tile_m, tile_n);
    else
      tile_m = L / tiles_n, tile_n = L - tile_m * tiles_n;
  }
  const int m0 = tile_m * TM, n0 = tile_n * TN;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l32 = lane & 31, half = lane >> 5;
  float *ring = f32_smem + wave * REGION;

  const int nk = (p.K + 15) >> 4;
  // The rows of A that this tile reads: [first, first + span), at most a descriptor's worth of them.
  // Gathered rows may lie anywhere in an operand whose extent nobody names, so the range comes from the
  // tile's own indices; where they lie further apart (4 GiB), every sum is formed by f32_dot_again.
  int first = m0, span = min(TM, M - m0), index = 0;
  bool far = false;
  if (p.a_row_index) {
    index = p.a_row_index[min(m0 + (lane & (TM - 1)), M - 1)];
    first = 0x7fffffff - wave_largest(0x7fffffff - index);
    span = wave_largest(index) - first + 1;
    far = (unsigned long long)span * p.K * 4 > kF32MaxBytes;
  }
  const int mine = far ? 0 : (nk - wave + NW - 1) / NW;   // slices wave, wave + NW, ...
  const auto rs_a = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p.a + (size_t)first * p.K), 0,
                                                      (int)((unsigned)span * (unsigned)p.K * 4u), 0x00020000);
  const auto rs_w = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float *>(p.w), 0, (int)((unsigned)p.K * (unsigned)p.N * 4u), 0x00020000);
  // byte offsets of this lane's pieces at k = 0.  Rows past M repeat the last live row, columns
  // past N lie outside the descriptor (they read as zero); neither is stored.
  unsigned aoff[NIA], woff[NIW];
#pragma unroll
  for (int i = 0; i < NIA; ++i) {
    const int row = i * 16 + (lane >> 2), chunk = (lane & 3) ^ ((row >> 2) & 3);
    const int src = p.a_row_index ? __shfl(index, row, 64) : min(m0 + row, M - 1);
    aoff[i] = ((unsigned)(src - first) * (unsigned)p.K + 4 * chunk) * 4u;
  }
#pragma unroll
  for (int i = 0; i < NIW; ++i) {
    constexpr int CPR = TN / 4;   // 16-byte chunks per k-row
    const int at = i * 64 + lane, pos = at / CPR, c = at % CPR;
    const int k = NT == 1 ? pos ^ ((pos >> 3) & 1) : pos;
    const int n = 4 * (NT == 2 ? c ^ (8 * ((pos >> 3) & 1)) : c);
    woff[i] = n0 + n < p.N ? ((unsigned)k * p.N + n0 + n) * 4u : kF32Outside;
  }
  // The loads of slice i of this wave.  Past the wave's last slice every offset lies outside: such
  // loads fetch nothing, read as zero and keep the count of loads in flight the same in every step.
  auto issue = [&](int i) {
    const int k0 = (wave + i * NW) * 16;
    const unsigned dead = i < mine ? 0u : kF32Outside;
    float *dst = ring + (i % DEPTH) * SLICE;
    const int a_k = k0 * 4, w_k = (int)((unsigned)k0 * p.N * 4u);
#pragma unroll
    for (int j = 0; j < NIA; ++j) {
      const int row = j * 16 + (lane >> 2), k = k0 + 4 * ((lane & 3) ^ ((row >> 2) & 3));
      // (of a last slice that reaches past k, only what lies before k is fetched)
      const unsigned off = RAGGED && k >= p.K ? kF32Outside : aoff[j] | dead;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rs_a, (__attribute__((address_space(3))) void *)(dst + j * 256), 16, (int)off, a_k, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < NIW; ++j) {
      const int pos = (j * 64 + lane) / (TN / 4), k = k0 + (NT == 1 ? pos ^ ((pos >> 3) & 1) : pos);
      const unsigned off = RAGGED && k >= p.K ? kF32Outside : woff[j] | dead;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rs_w, (__attribute__((address_space(3))) void *)(dst + (NIA + j) * 256), 16, (int)off, w_k,
          0, 0);
    }
  };
  float4_t xa[MT][2];
  float xw[NT][8];
  auto read_slice = [&](int i) {
    const float *src = ring + (i % DEPTH) * SLICE;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int row = mt * 32 + l32;
        xa[mt][j] = *(const float4_t *)(src + row * 16 + 4 * ((2 * half + j) ^ ((row >> 2) & 3)));
      }
    const float *w = src + TM * 16;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if (NT == 2)
          xw[nt][e] = w[(8 * half + e) * TN + ((nt * 32 + l32) ^ (32 * half))];
        else
          xw[nt][e] = w[((8 * half + e) ^ half) * TN + l32];
      }
  };
  struct Operands {
    bf16x8_t a[MT][3], w[NT][3];
  };
  auto split = [&](Operands &o) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const float x[8] = {xa[mt][0][0], xa[mt][0][1], xa[mt][0][2], xa[mt][0][3],
                          xa[mt][1][0], xa[mt][1][1], xa[mt][1][2], xa[mt][1][3]};
      split_bf16x8(o.a[mt], x);
    }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) split_bf16x8(o.w[nt], xw[nt]);
  };

  float16_t acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[mt][nt][i] = 0.f;

  // takes slice i from the ring (its loads are the oldest of DEPTH slices in flight) and sends
  // the loads of slice i + DEPTH after it
  auto take = [&](int i) {
    f32_wait_vmcnt<(DEPTH - 1) * NI>();
    asm volatile("" ::: "memory");
    read_slice(i);
  };
  auto refill = [&](int i) {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the slot has been read
    issue(i + DEPTH);
  };
  auto multiply = [&](const Operands &o) {
#pragma unroll
    for (int t = 0; t < 6; ++t) {
      constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pw[6] = {0, 2, 1, 0, 1, 0};   // smallest terms first
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(o.a[mt][pa[t]], o.w[nt][pw[t]],
                                                                acc[mt][nt], 0, 0, 0);
    }
  };
  if (mine > 0) {
#pragma unroll
    for (int i = 0; i < DEPTH; ++i) issue(i);
    Operands o[2];
    take(0);
    split(o[0]);
    refill(0);
    // slice i is multiplied while slice i + 1 is read and split: one basic block, in which the
    // vector instructions of the split are dealt out between the matrix instructions
    auto step = [&](int i, const Operands &now, Operands &next) {
      take(i + 1);
      multiply(now);
      split(next);
      constexpr int kMfma = 6 * MT * NT, kSplit = (MT + NT) * 44;   // 44 vector instructions per 8 elements
      __builtin_amdgcn_sched_group_barrier(0x100, 2 * MT + 8 * NT, 0);   // the LDS reads first
#pragma unroll
      for (int t = 0; t < kMfma; ++t) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, (kSplit + kMfma - 1) / kMfma, 0);
      }
      refill(i + 1);
    };
    for (int i = 0; i < mine; i += 2) {   // (an odd last slice is followed by an empty one)
      step(i, o[0], o[1]);
      step(i + 1, o[1], o[0]);
    }
    f32_wait_vmcnt<0>();   // the ring is about to be reused
  }

  // fold: every wave leaves its sums in its own region (columns XOR 32 in rows with bit 2 set: the
  // halves of a wave write distinct banks), then takes TM / NW rows of the tile over all regions
  constexpr int XR = NT == 2 ? 32 : 0;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int row = mt * 32 + 8 * (i >> 2) + 4 * half + (i & 3);
        ring[row * TN + ((nt * 32 + l32) ^ (XR * half))] = acc[mt][nt][i];
      }
  __syncthreads();
  constexpr int LPR = TN / 4;            // lanes per row, four columns each
  constexpr int RPP = 64 / LPR;          // rows per pass of a wave
  constexpr int PASSES = TM / (RPP * NW);
  static_assert(TM % (RPP * NW) == 0, "whole passes over the rows of a tile");
  const int row0 = wave * RPP + lane / LPR, c = 4 * (lane % LPR);
  float4_t v[PASSES];
  F32SumRange range;
#pragma unroll
  for (int i = 0; i < PASSES; ++i) {
    const int row = row0 + i * RPP * NW;
    const float *src = f32_smem + row * TN + (c ^ (XR * ((row >> 2) & 1)));
    v[i] = *(const float4_t *)src;
#pragma unroll
    for (int w = 1; w < NW; ++w) v[i] += *(const float4_t *)(src + w * REGION);
#pragma unroll
    for (int e = 0; e < 4; ++e) range.add(v[i][e]);
  }
  const int n = n0 + c;
  if (far || !range.split_held()) {
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
      const int m = m0 + row0 + i * RPP * NW;
      if (m >= M || n >= p.N) continue;
      float sum[4];
      f32_dot_again(f32_a_row(p, m), p.w + n, p.K, p.N, sum);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        F32SumRange one;
        one.add(v[i][e]);
        if (far || !one.split_held()) v[i][e] = sum[e];
      }
    }
  }
#pragma unroll
  for (int i = 0; i < PASSES; ++i) {
    const int m = m0 + row0 + i * RPP * NW;
    if (m >= M || n >= p.N) continue;
    if (p.bias) v[i] += float4_t{p.bias[n], p.bias[n + 1], p.bias[n + 2], p.bias[n + 3]};
    if (p.gelu) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[i][e] = f32_gelu(v[i][e]);
    }
    store_through(p.c + (size_t)m * p.N + n, __builtin_bit_cast(uint4_t, v[i]));
  }
}
#endif

template <int MT, int NT, int NW, int DEPTH, bool RAGGED>
__global__ __launch_bounds__(64 * NW) void f32_gemm_kernel(F32GemmArgs p) {
#if defined(__HIP_DEVICE_COMPILE__)
  f32_gemm_tile<MT, NT, NW, DEPTH, RAGGED>(p);
#endif
}

// Few rows: one 32x32 tile per workgroup, the k range dealt to its NW waves in steps of 16 and
// folded through LDS at the end.  No LDS and no barrier in the loop: a wave takes its operands from
// memory in MFMA order (A: 8 consecutive k of a row per lane, W: one column per lane), DEPTH steps
// ahead.
template <int NW>
__global__ __launch_bounds__(64 * NW) void f32_gemm_skinny_kernel(F32GemmArgs p) {
  constexpr int DEPTH = 4;
  __shared__ float part[NW - 1][16][64];
  const int M = p.valid_rows ? min(*p.valid_rows, p.rows_cap) : p.rows_cap;
  const int m0 = blockIdx.y * 32, n0 = blockIdx.x * 32;
  if (m0 >= M) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l32 = lane & 31, half = lane >> 5;
  const int r = min(m0 + l32, M - 1), n = min(n0 + l32, p.N - 1);
  const float *a_src = p.a + (p.a_row_index ? (size_t)p.a_row_index[r] : (size_t)r) * p.K;
  const float *w_src = p.w + n;
  const int nk = (p.K + 15) / 16;

  float4_t ra[DEPTH][2];
  float rw[DEPTH][8];
  auto fetch = [&](int kt, int s) {
    const int k = 16 * kt + 8 * half;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      ra[s][j] = float4_t{0.f, 0.f, 0.f, 0.f};
      if (k + 4 * j < p.K) ra[s][j] = *(const float4_t *)(a_src + k + 4 * j);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) rw[s][e] = k + e < p.K ? w_src[(size_t)(k + e) * p.N] : 0.f;
  };
  float16_t acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
  for (int s = 0; s < DEPTH - 1; ++s)
    if (wave + s * NW < nk) fetch(wave + s * NW, s);
  for (int kt = wave; kt < nk; kt += DEPTH * NW) {
#pragma unroll
    for (int s = 0; s < DEPTH; ++s) {
      const int at = kt + s * NW;
      if (at < nk) {
        if (at + (DEPTH - 1) * NW < nk) fetch(at + (DEPTH - 1) * NW, (s + DEPTH - 1) % DEPTH);
        bf16x8_t a[3], b[3];
        const float xa[8] = {ra[s][0][0], ra[s][0][1], ra[s][0][2], ra[s][0][3],
                             ra[s][1][0], ra[s][1][1], ra[s][1][2], ra[s][1][3]};
        split_bf16x8(a, xa);
        split_bf16x8(b, rw[s]);
        acc = mfma_triple(a, b, acc);
      }
    }
  }
  if (wave > 0) {
#pragma unroll
    for (int i = 0; i < 16; ++i) part[wave - 1][i][lane] = acc[i];
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int w = 0; w < NW - 1; ++w)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] += part[w][i][lane];
  f32_store_block(p, acc, m0, n0, M, l32, half);
}

// ---------------------------------------------------------------------------
// attention
// ---------------------------------------------------------------------------
struct F32AttArgs {
  const float *qkv;    // [rows, 3H], QKV bias already added
  float *out;          // [rows, H]
  const int *batch_idx;
  const int *seq_order;   // optional: rank -> sequence, longest first
  const float *mask;   // optional [B,S,S]
  const float *bias;   // optional [heads,S,S]
  int B, S, rows_cap, heads;
  float scale;
  int padded_rows;
  int nqb;             // query tiles per sequence
  int balanced;        // 1: the live query tiles are dealt evenly to the CUs (common.h)
  int d;               // head size (a multiple of 8, <= the kernel's D = 32 * ND; the
                       // columns d..D-1 of Q, K and V read as zero)
};

constexpr int kF32KT = 32;   // keys per tile

// One workgroup = NQ waves x 32 queries of one (sequence, head); KS groups of such waves share the keys, group g taking
// the tiles g, g + KS, ..., and fold through LDS.  The logits are computed
// transposed, S^T = K.Q^T (lane = query, 16 keys per lane), so their accumulator is
// directly the "B" operand of O^T = V^T.P^T and the softmax statistics of a query are
// lane-local up to one exchange between the two halves of the wave.  The MFMA's k index
// may be any bijection as long as both operands agree; it is chosen so that Q and K are
// read as float4 (k = half*D/2 + step) and P needs no shuffle (key of step j in half h
// = 8*(j/4) + 4*h + j%4, the accumulator's own row order).
//
// Two waves per SIMD are asked for because the accumulators then stay in the registers that vector
// instructions read.  With one wave they lay in AGPRs: the compiler copied all of them on every turn of the
// loop, and behind it read the last one 7 wait states after the last matrix instruction, which takes 18 -
// wrong last columns at head sizes 96 and 128, another way in every run.  (tests/test_kernel_resources.py
// looks for such reads in every kernel.)
template <int ND, int NQ, int KS>
__global__ __launch_bounds__(64 * NQ * KS, 2) void f32_attention_kernel(F32AttArgs p) {
  constexpr int D = 32 * ND;
  constexpr int THREADS = 64 * NQ * KS, BQ = 32 * NQ;   // 32 queries per wave
  constexpr int STEP = kF32KT * KS;                     // keys of a turn
  constexpr int SK = D + 4, SV = D + 8;
  __shared__ __attribute__((aligned(16))) float smem[STEP * (SK + SV)];
  float *const sK = smem, *const sV = smem + STEP * SK;
  static_assert(KS == 1 || NQ * 64 * (16 * ND + 2) <= STEP * (SK + SV), "a group's sums fit the tiles' place");

  // 1-D grid, XCD-aware: the hardware deals consecutive workgroup ids round-robin to the
  // 8 XCDs; XCD x works on the (sequence, head) pairs p = x (mod 8), the query tiles of
  // one pair back to back (its K / V then come from that XCD's L2), so every XCD sees the
  // same mix of sequence lengths however ragged the batch is.
  // Launches of more than two rounds of workgroups per CU take the balanced work list.
  int b, head, seq_start, len, qb_index;
  if (p.balanced) {
    const AttWork w = att_work_balanced<BQ>(p, blockIdx.x);
    if (!w.exists) return;
    b = w.b, head = w.head, seq_start = w.seq_start, len = w.len, qb_index = w.qb;
  } else {
    const unsigned lin = blockIdx.x, slot = lin >> 3;
    const unsigned pair = (slot / p.nqb) * 8 + (lin & 7);
    if (pair >= (unsigned)(p.B * p.heads)) return;
    const int rank = pair / p.heads;
    head = pair % p.heads;
    b = p.seq_order ? p.seq_order[rank] : rank;
    seq_start = p.batch_idx[b];
    len = p.batch_idx[b + 1] - seq_start;
    qb_index = (int)(slot % p.nqb);
  }
  const int klen = (p.mask && p.padded_rows) ? p.S : len;
  const int row_start = p.padded_rows ? b * p.S : seq_start;
  const int nq = p.padded_rows ? p.S : len;
  const int q0 = qb_index * BQ;
  if (q0 >= nq || klen <= 0) {
    // padded rows of an empty sequence still get defined output: zeros
    if (q0 < nq) {
      const int H = p.heads * p.d;
      for (int i = threadIdx.x; i < BQ * p.d; i += THREADS) {
        const int q = q0 + i / p.d;
        if (q < nq) p.out[(size_t)(row_start + q) * H + head * p.d + i % p.d] = 0.f;
      }
    }
    return;
  }

  const int tid = threadIdx.x, lane = tid & 63, wave_all = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave = KS > 1 ? wave_all % NQ : wave_all, group = KS > 1 ? wave_all / NQ : 0;
  const int l32 = lane & 31, half = lane >> 5;
  const int d = p.d;
  const int H = p.heads * d;
  const size_t ld = (size_t)3 * H;
  const float *Q = p.qkv + (size_t)row_start * ld + head * d;
  const float *K = Q + H;
  const float *V = K + H;

  const int q = q0 + wave * 32 + l32;       // this lane's query
  const bool query_live = q0 + wave * 32 < nq;
  const int qc = min(q, nq - 1);

  // Q^T operand: lane (query, half) holds Q[q][half*D/2 + i]
  float qf[D / 2];
#pragma unroll
  for (int i = 0; i < D / 8; ++i) {
    const int e = half * (D / 2) + 4 * i;
    float4_t v = {0.f, 0.f, 0.f, 0.f};
    if (e < d) v = *(const float4_t *)(Q + (size_t)qc * ld + e);
#pragma unroll
    for (int j = 0; j < 4; ++j) qf[4 * i + j] = v[j];
  }

  // tile staging: 32 KS keys x D floats of K and of V, NV float4 each per thread
  constexpr int CPR = D / 4;   // float4 per row
  constexpr int NV = STEP * CPR / THREADS;
  float4_t rk[NV], rv[NV];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int idx = tid + THREADS * i;
      const int key = min(k0 + idx / CPR, klen - 1);
      const int e = 4 * (idx % CPR);
      const size_t off = (size_t)key * ld + e;
      rk[i] = rv[i] = float4_t{0.f, 0.f, 0.f, 0.f};
      if (e < d) {
        rk[i] = *(const float4_t *)(K + off);
        rv[i] = *(const float4_t *)(V + off);
      }
    }
  };
  auto stash = [&]() {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int idx = tid + THREADS * i;
      *(float4_t *)&sK[(idx / CPR) * SK + 4 * (idx % CPR)] = rk[i];
      *(float4_t *)&sV[(idx / CPR) * SV + 4 * (idx % CPR)] = rv[i];
    }
  };

  float16_t o[ND];
#pragma unroll
  for (int dt = 0; dt < ND; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[dt][i] = 0.f;
  float m_run = kDeadLogit, l_run = 0.f;

  const float c = p.scale * kLog2eF;
  const float *mrow = p.mask ? p.mask + ((size_t)b * p.S + min(q, p.S - 1)) * p.S : nullptr;
  const float *brow = p.bias ? p.bias + ((size_t)head * p.S + min(q, p.S - 1)) * p.S : nullptr;

  const int turns = (klen + STEP - 1) / STEP;
  fetch(0);
  stash();
  __syncthreads();
  const bool has_add = mrow || brow;
  const bool add_vec = (p.S & 3) == 0;
  for (int t = 0; t < turns; ++t) {
    const int k0 = t * STEP + group * kF32KT;
    const bool wave_live = query_live && (KS == 1 || k0 < klen);
    // additive terms of this tile's 16 keys per lane (4 groups of 4 consecutive keys),
    // in the exp2 domain; issued ahead of the next tile's K / V so that the wait for
    // them does not include those
    float4_t add[4];
    if (has_add && wave_live) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int key = k0 + 8 * g + 4 * half;
        float4_t mv = {1.f, 1.f, 1.f, 1.f}, bv = {0.f, 0.f, 0.f, 0.f};
        if (add_vec && key + 3 < p.S) {
          if (mrow) mv = *(const float4_t *)(mrow + key);
          if (brow) bv = *(const float4_t *)(brow + key);
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (key + r < p.S) {
              if (mrow) mv[r] = mrow[key + r];
              if (brow) bv[r] = brow[key + r];
            }
        }
        add[g] = (mv - 1.0f) * (10000.0f * kLog2eF) + bv * kLog2eF;
      }
    }
    if (t + 1 < turns) fetch((t + 1) * STEP);
    if (wave_live) {
      // S^T = K . Q^T : A operand K[key = l32][k = half*D/2 + i]
      float16_t s;
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = 0.f;
      const float *kp = &sK[(group * kF32KT + l32) * SK + half * (D / 2)];
#pragma unroll
      for (int i4 = 0; i4 < D / 8; ++i4) {
        const float4_t kv = *(const float4_t *)(kp + 4 * i4);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[j], qf[4 * i4 + j], s, 0, 0, 0);
      }
      // logits in the exp2 domain; accumulator row i is key k0 + 8*(i/4) + 4*half + i%4
      float x[16];
      float tmax = kDeadLogit;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int key = k0 + 8 * (i >> 2) + 4 * half + (i & 3);
        float v = s[i] * c;
        if (has_add) v += add[i >> 2][i & 3];
        if (key >= klen) v = kDeadLogit;
        x[i] = v;
        tmax = fmaxf(tmax, v);
      }
      tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
      const float m_new = fmaxf(m_run, tmax);
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
      m_run = m_new;
      float psum = 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int key = k0 + 8 * (i >> 2) + 4 * half + (i & 3);
        const float pv = key < klen ? __builtin_amdgcn_exp2f(x[i] - m_new) : 0.f;
        x[i] = pv;
        psum += pv;
      }
      l_run = l_run * alpha + psum;
      // the running maximum of most queries settles after a few tiles: skip the rescale
      // of the accumulators when it moved for no query of the wave
      if (__any(alpha != 1.0f)) {
#pragma unroll
        for (int dt = 0; dt < ND; ++dt)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[dt][i] *= alpha;
      }
      // O^T += V^T . P^T : A operand V[key(j, half)][d = 32*dt + l32], B operand P^T = x[j]
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const float *vp = &sV[(group * kF32KT + 8 * (j >> 2) + 4 * half + (j & 3)) * SV + l32];
#pragma unroll
        for (int dt = 0; dt < ND; ++dt)
          o[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(vp[32 * dt], x[j], o[dt], 0, 0, 0);
      }
    }
    __syncthreads();
    if (t + 1 < turns) {
      stash();
      __syncthreads();
    }
  }

  // The other groups' sums come to the first one's waves by way of the tiles' place, which nobody reads any more.
#pragma unroll
  for (int g = 1; g < KS; ++g) {
    float *const to = smem + wave * 64 * (16 * ND + 2) + lane;
    if (group == g) {
      to[0] = m_run, to[64] = l_run;
#pragma unroll
      for (int dt = 0; dt < ND; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) to[64 * (2 + 16 * dt + i)] = o[dt][i];
    }
    __syncthreads();
    if (group == 0) {
      const float m_new = fmaxf(m_run, to[0]);
      const float mine = __builtin_amdgcn_exp2f(m_run - m_new), theirs = __builtin_amdgcn_exp2f(to[0] - m_new);
      m_run = m_new;
      l_run = l_run * mine + to[64] * theirs;
#pragma unroll
      for (int dt = 0; dt < ND; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[dt][i] = o[dt][i] * mine + to[64 * (2 + 16 * dt + i)] * theirs;
    }
    if (g + 1 < KS) __syncthreads();
  }

  if (group > 0 || !query_live || q >= nq) return;
  const float l_all = l_run + __shfl_xor(l_run, 32, 64);
  const float inv = 1.0f / (l_all + 1e-6f);
  // accumulator element i of d-tile dt: d = 32*dt + 8*(i/4) + 4*half + i%4, query = l32
  float *orow = p.out + (size_t)(row_start + q) * H + head * d;
#pragma unroll
  for (int dt = 0; dt < ND; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float4_t v;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = o[dt][4 * g + r] * inv;
      if (32 * dt + 8 * g + 4 * half < d) *(float4_t *)(orow + 32 * dt + 8 * g + 4 * half) = v;
    }
}

// ---------------------------------------------------------------------------
// add-bias + residual + LayerNorm
// ---------------------------------------------------------------------------
constexpr int kF32LnRows = 4;

// What a LayerNorm whose rows the next product reads as pairs writes beside them.
struct F32LnPairs {
  half_t *pairs;         // [rows][H / 32][64]
  int *exps;             // [rows]
  // exponents for the pairs of GELU(row . W + bias): |row . w| is at most |row|_2 sqrt(H) max |w|
  int *gelu_exps;        // [rows]
  const float *bounds;   // [bound_count][2]: largest |w| and |bias| of some columns each
  int bound_count;
  unsigned *raw;         // [rows][raw_words] cleared for the product that reads the pairs (its rows that stay floats), or null: no marks either
  int raw_words;
};

// One wave per row, float4 per lane, the row in registers between the two passes.
template <int NC, bool RESTORE, bool PAIRS>
__device__ __forceinline__ void f32_layernorm_block(
    const float4_t *src, const float4_t *__restrict__ residual, const float4_t *__restrict__ bias,
    const float4_t *__restrict__ gamma, const float4_t *__restrict__ beta, float4_t *dst,
    const int *__restrict__ idx, const int *__restrict__ residual_row_index, int S, int rows_cap,
    int chunks, float inv_n, float eps, const F32LnPairs &next) {
  const int r = blockIdx.x * kF32LnRows + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (r >= rows_cap) return;
  // what no loaded value points at is requested first: behind the statistics, gamma and beta were one more
  // round trip (rows too wide for the registers keep it)
  constexpr bool kEarly = NC <= 4;
  float4_t bias_v[kEarly ? NC : 1], gamma_v[kEarly ? NC : 1], beta_v[kEarly ? NC : 1];
  if (kEarly) {
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = min(lane + i * kWave, chunks - 1);
      bias_v[i] = bias[c], gamma_v[i] = gamma[c], beta_v[i] = beta[c];
    }
  }
  size_t src_row;
  if (RESTORE) {
    const int b = r / S, s = r - b * S;
    const int start = idx[b], len = idx[b + 1] - start;
    if (s >= len) {
      const float4_t z = {0.f, 0.f, 0.f, 0.f};
      for (int c = lane; c < chunks; c += kWave) store_through(dst + (size_t)r * chunks + c, __builtin_bit_cast(uint4_t, z));
      return;
    }
    src_row = (size_t)start + s;
  } else {
    const int M = idx ? *idx : rows_cap;
    if (r >= M) return;
    src_row = r;
  }
  const float4_t *a = src + src_row * chunks;
  const size_t res_row = residual_row_index ? (size_t)residual_row_index[src_row] : src_row;
  const float4_t *rs = residual + res_row * chunks;
  float4_t v[NC];
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int c = lane + i * kWave;
    v[i] = float4_t{0.f, 0.f, 0.f, 0.f};
    if (c < chunks) {
      v[i] = a[c] + rs[c] + (kEarly ? bias_v[i] : bias[c]);
      sum += v[i][0] + v[i][1] + v[i][2] + v[i][3];
    }
  }
  const float mean = wave_sum(sum) * inv_n;
  float sq = 0.f;
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int c = lane + i * kWave;
    if (c < chunks) {
      v[i] -= mean;
      sq += v[i][0] * v[i][0] + v[i][1] * v[i][1] + v[i][2] * v[i][2] + v[i][3] * v[i][3];
    }
  }
  const float rstd = rsqrtf(wave_sum(sq) * inv_n + eps);
  float4_t *o = dst + (size_t)r * chunks;
  float most = 0.f;
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int c = lane + i * kWave;
    if (c >= chunks) continue;
    v[i] = v[i] * rstd * (kEarly ? gamma_v[i] : gamma[c]) + (kEarly ? beta_v[i] : beta[c]);
    store_through(o + c, __builtin_bit_cast(uint4_t, v[i]));
    if (PAIRS)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = __builtin_fabsf(v[i][e]);
        most = fmaxf(most, x < __builtin_inff() ? x : 0.f);
      }
  }
  if (PAIRS) {
    float w_most = 0.f, bias_most = 0.f;
    for (int i = lane; i < next.bound_count; i += kWave) {
      w_most = fmaxf(w_most, next.bounds[2 * i]);
      bias_most = fmaxf(bias_most, next.bounds[2 * i + 1]);
    }
    const int e = split_exponent(wave_max(most));
    const float scale = split_power(e);
    float norm = 0.f;   // of the scaled row: at most 2^30 H
    bool small = false;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = lane + i * kWave;
      if (c >= chunks) continue;
      const float4_t x = v[i] * scale;
      small = split_store(next.pairs + (size_t)r * chunks * 8, c, x) || small;
      norm += x[0] * x[0] + x[1] * x[1] + x[2] * x[2] + x[3] * x[3];
    }
    // (a bound that is no float is the largest float: finite results fit it, and a row with an infinity or NaN has none)
    const float row_norm = sqrtf(wave_sum(norm) * (float)(chunks * 4)) * split_power(-e);
    const float bound = fminf(row_norm * wave_max(w_most) + wave_max(bias_most), 3.402823466e38f);
    bool marked = false;
    if (next.raw && __builtin_amdgcn_ballot_w64(small) != 0) {
      float score = 0.f;
#pragma unroll
      for (int i = 0; i < NC; ++i)
        if (lane + i * kWave < chunks) score += split_score(v[i], scale);
      marked = wave_sum(score) > 0.f;
    }
    if (lane == 0) {
      next.exps[r] = e + (marked ? kSplitMark : 0);
      next.gelu_exps[r] = split_exponent(bound);
    }
    if (lane < next.raw_words) next.raw[(size_t)r * next.raw_words + lane] = 0;
  }
}

template <int NC, bool RESTORE>
__global__ __launch_bounds__(kF32LnRows *kWave) void f32_layernorm_kernel(
    const float4_t *src, const float4_t *residual, const float4_t *bias, const float4_t *gamma, const float4_t *beta,
    float4_t *dst, const int *idx, const int *residual_row_index, int S, int rows_cap, int chunks, float inv_n,
    float eps) {
  f32_layernorm_block<NC, RESTORE, false>(src, residual, bias, gamma, beta, dst, idx, residual_row_index, S, rows_cap, chunks,
                                          inv_n, eps, F32LnPairs{});
}
template <int NC>
__global__ __launch_bounds__(kF32LnRows *kWave) void f32_layernorm_pairs_kernel(
    const float4_t *src, const float4_t *residual, const float4_t *bias, const float4_t *gamma, const float4_t *beta,
    float4_t *dst, const int *idx, const int *residual_row_index, int rows_cap, int chunks, float inv_n, float eps,
    F32LnPairs next) {
  f32_layernorm_block<NC, false, true>(src, residual, bias, gamma, beta, dst, idx, residual_row_index, 1, rows_cap, chunks, inv_n,
                                       eps, next);
}

template <bool RESTORE>
int launch_f32_ln(const void *src, const void *residual, const void *bias, const void *gamma,
                  const void *beta, void *dst, const int *idx, const int *residual_row_index,
                  int S, int rows_cap, int H, float eps, hipStream_t s, const char *who,
                  const F32LnPairs *next = nullptr) {
  BT_REQUIRE(H > 0 && H % 4 == 0, BT_ERR_UNSUPPORTED, "%s: hidden_dim %d must be a multiple of 4",
             who, H);
  BT_REQUIRE(aligned16({src, residual, bias, gamma, beta, dst}), BT_ERR_INVALID_ARGUMENT,
             "%s: tensor pointers must be 16-byte aligned", who);
  const int chunks = H / 4;
  const int nc = (chunks + kWave - 1) / kWave;
  BT_REQUIRE(nc <= 16, BT_ERR_UNSUPPORTED, "%s: hidden_dim %d exceeds 4096", who, H);
  if (rows_cap == 0) return BT_OK;
  const int grid = (rows_cap + kF32LnRows - 1) / kF32LnRows;
  const float inv_n = 1.0f / (float)H;
  const auto with = [&](auto nc_tag) {
    if constexpr (!RESTORE)
      if (next)
        return Launch<f32_layernorm_pairs_kernel<nc_tag()>>::on(
            s, who, grid, kF32LnRows * kWave, 0, (const float4_t *)src, (const float4_t *)residual, (const float4_t *)bias,
            (const float4_t *)gamma, (const float4_t *)beta, (float4_t *)dst, idx, residual_row_index, rows_cap, chunks,
            inv_n, eps, *next);
    return Launch<f32_layernorm_kernel<nc_tag(), RESTORE>>::on(
        s, who, grid, kF32LnRows * kWave, 0, (const float4_t *)src, (const float4_t *)residual, (const float4_t *)bias,
        (const float4_t *)gamma, (const float4_t *)beta, (float4_t *)dst, idx, residual_row_index, S, rows_cap, chunks,
        inv_n, eps);
  };
  if (nc <= 2) return with(std::integral_constant<int, 2>{});
  if (nc <= 4) return with(std::integral_constant<int, 4>{});
  if (nc <= 8) return with(std::integral_constant<int, 8>{});
  return with(std::integral_constant<int, 16>{});
}

template <int MT, int NT, int NW, int DEPTH, bool RAGGED>
static int launch_f32_gemm_as(const F32GemmArgs &p, hipStream_t s) {
  constexpr int TM = 32 * MT, TN = 32 * NT, SLICE = (TM + TN) * 16;
  constexpr size_t smem = (size_t)NW * (DEPTH * SLICE > TM * TN ? DEPTH * SLICE : TM * TN) * sizeof(float);
  static_assert(smem <= 160 * 1024, "LDS budget");
  const long long tiles = (long long)((p.rows_cap + TM - 1) / TM) * ((p.N + TN - 1) / TN);
  return Launch<f32_gemm_kernel<MT, NT, NW, DEPTH, RAGGED>>::on(s, "bt_gemm_f32", (unsigned)((tiles + 7) / 8 * 8),
                                                                64 * NW, smem, p);
}
template <int MT, int NT, int NW, int DEPTH>
static int launch_f32_gemm(const F32GemmArgs &p, hipStream_t s) {
  return p.K % 16 ? launch_f32_gemm_as<MT, NT, NW, DEPTH, true>(p, s)
                  : launch_f32_gemm_as<MT, NT, NW, DEPTH, false>(p, s);
}

}  // namespace
}  // namespace bt

using namespace bt;

extern "C" int bt_gemm_f32(const void *a, const int *a_row_index, const void *w, const void *bias,
                           void *c, int gelu, const int *valid_rows, int rows_cap, int rows_hint,
                           int n, int k, void *stream) {
  BT_REQUIRE(a && w && c, BT_ERR_INVALID_ARGUMENT, "bt_gemm_f32: null pointer argument");
  BT_REQUIRE(aligned16({a, w, c}), BT_ERR_INVALID_ARGUMENT,
             "bt_gemm_f32: tensor pointers must be 16-byte aligned");
  BT_REQUIRE(rows_cap >= 0 && n > 0 && k > 0, BT_ERR_INVALID_ARGUMENT,
             "bt_gemm_f32: sizes must be positive");
  BT_REQUIRE(n % 4 == 0 && k % 4 == 0, BT_ERR_UNSUPPORTED,
             "bt_gemm_f32: n (%d) and k (%d) must be multiples of 4", n, k);
  BT_REQUIRE(!a_row_index || valid_rows, BT_ERR_INVALID_ARGUMENT,
             "bt_gemm_f32: a_row_index needs valid_rows");
  BT_REQUIRE(!gelu || bias, BT_ERR_INVALID_ARGUMENT, "bt_gemm_f32: gelu needs a bias");
  BT_REQUIRE((long long)rows_cap * n < (1ll << 40), BT_ERR_UNSUPPORTED, "bt_gemm_f32: too large");
  if (rows_cap == 0) return BT_OK;
  F32GemmArgs p{(const float *)a, (const float *)w, (const float *)bias, (float *)c, valid_rows,
                a_row_index, rows_cap, n, k, gelu ? 1 : 0};
  // Tile table: 0: 64x64 | 1: 64x32 | 2: 32x32 (four waves over k each) | 3: the skinny kernel.
  // A tile takes `fixed` us plus, per turn of its four waves over k, `alone` us if it has the CU to
  // itself and else its share of a busy CU, `shared` us: 32x32 while the launch leaves CUs idle, 64x64
  // once the split of the operands has to be amortised.  Over the four products of hidden 512, 768 and
  // 1024 at twelve row counts from 32 to 4800 the choice is the fastest tile or within 2 % of it in
  // 139 of 144, and 7 % slower at worst (profiles/float_product_tiles.txt).
  struct Cand { int id, bm, bn; float fixed, alone, shared; };
  static const Cand cands[3] = {{0, 64, 64, 5.0f, 0.54f, 0.77f}, {1, 64, 32, 4.5f, 0.45f, 0.54f},
                                {2, 32, 32, 4.0f, 0.40f, 0.325f}};
  int tile = option_f32_gemm_tile();
  if (tile < 0) {
    // the row count that matters is the live one; the hint is the caller's estimate of it
    const int rows = (valid_rows && rows_hint > 0 && rows_hint < rows_cap) ? rows_hint : rows_cap;
    const float turns = (float)((k + 63) / 64);
    float best = 0.f;
    for (const Cand &cd : cands) {
      const long long wgs = (long long)((rows + cd.bm - 1) / cd.bm) * ((n + cd.bn - 1) / cd.bn);
      const float load = (float)wgs / (float)kF32CUs;
      const float cost = cd.fixed + turns * fmaxf(cd.alone, load * cd.shared);
      if (tile < 0 || cost < best) {
        best = cost;
        tile = cd.id;
      }
    }
  }
  // the tiled kernels address the weight, and the rows of a tile, with 32-bit byte offsets
  if ((long long)n * k * 4 > kF32MaxBytes || (long long)k * 256 > kF32MaxBytes) tile = 3;
  hipStream_t s = as_stream(stream);
  if (tile == 0) return launch_f32_gemm<2, 2, 4, 2>(p, s);
  if (tile == 1) return launch_f32_gemm<2, 1, 4, 3>(p, s);
  if (tile == 2) return launch_f32_gemm<1, 1, 4, 4>(p, s);
  const dim3 grid((n + 31) / 32, (rows_cap + 31) / 32);
  BT_REQUIRE(grid.y <= 65535, BT_ERR_UNSUPPORTED, "bt_gemm_f32: too many rows");
  f32_gemm_skinny_kernel<8><<<grid, 512, 0, s>>>(p);
  BT_CHECK_LAUNCH("bt_gemm_f32");
  return BT_OK;
}

extern "C" int bt_attention_f32(const void *qkv, void *out, const int *batch_idx,
                                const int *seq_order, const void *atten_mask,
                                const void *attention_bias, int batch_size, int seq_len,
                                int rows_cap, int head_num, int size_per_head, float scale,
                                int padded_rows, void *stream) {
  const char *who = "bt_attention_f32";
  const int rc = check_generic_attention(who, qkv, out, batch_idx, atten_mask, attention_bias, batch_size,
                                         seq_len, rows_cap, head_num, size_per_head, padded_rows);
  if (rc != BT_OK) return rc;
  F32AttArgs p{(const float *)qkv, (float *)out, batch_idx, seq_order, (const float *)atten_mask,
               (const float *)attention_bias, batch_size, seq_len, rows_cap, head_num, scale,
               padded_rows ? 1 : 0};
  p.d = size_per_head;
  // 64 queries whose keys two groups of waves share, or 128 (heads beyond 64 have no room in 64 KB of LDS for two groups'
  // tiles).  A turn is 5000 clocks of dependent matrix instructions, so a launch of few workgroups is as long as its
  // longest sequence has turns: us, 128 queries / shared, 12 heads of 64, lengths 0.2 to 1 of the maximum, 1 x 256
  // 8.5 / 6.8, 2 x 100 8.4 / 6.7, 10 x 200 21.2 / 18.4, 16 x 256 34.3 / 23.4, 4 x 640 62.5 / 58.0, full 1 x 1024 91.0 / 52.0; 24 heads
  // of 32, 7 x 333 27.1 / 17.4.  Up to 64 tokens the second group has next to nothing (1 x 64 5.6 / 6.3, 128 x 20 21.8 / 24.1);
  // beyond two rounds of workgroups they are even (16 x 512 56.8 / 59.2, 32 x 512 121 / 117).  Against float64 the shared sums
  // are the nearer ones (16 x 256 3.7e-7 / 3.4e-7, 1 x 1024 6.5e-7 / 5.0e-7).
  // In a layer of 16 x 256, with the mask's rows, 41.8 / 32.6 us; 12 layers 2936 / 2824.
  const int qb = option_attention_qb();
  const long long blocks128 = (long long)((seq_len + 127) / 128) * head_num * batch_size;
  const bool shared_keys = size_per_head <= 64 && (qb < 0 ? seq_len > 64 && blocks128 <= 2LL * cu_count() : qb == 1);
  const int queries = shared_keys ? 64 : 128;   // of a workgroup
  p.nqb = (seq_len + queries - 1) / queries;
  // the conditions of the fp16 streaming kernel: from the third round of 32 workgroups
  // per XCD on and up to 128 sequences, or always / never by the option
  const unsigned per_xcd = ((unsigned)batch_size * head_num + 7) / 8 * p.nqb;
  const int order = option_attention_xcd_map();
  p.balanced = order == 3 || (order == 2 && per_xcd > 64 && batch_size <= 128);
  const unsigned grid = p.balanced ? (per_xcd + 31) / 32 * 32 * 8 : per_xcd * 8;
  hipStream_t s = as_stream(stream);
  const auto with = [&](auto nd, auto nq, auto ks) {
    return Launch<f32_attention_kernel<nd(), nq(), ks()>>::on(s, who, grid, 256, 0, p);
  };
  using one = std::integral_constant<int, 1>;
  using two = std::integral_constant<int, 2>;
  using four = std::integral_constant<int, 4>;
  switch ((size_per_head + 31) / 32) {
    case 1: return shared_keys ? with(one{}, two{}, two{}) : with(one{}, four{}, one{});
    case 2: return shared_keys ? with(two{}, two{}, two{}) : with(two{}, four{}, one{});
    case 3: return with(std::integral_constant<int, 3>{}, four{}, one{});
    default: return with(four{}, four{}, one{});
  }
}

extern "C" int bt_add_bias_residual_layernorm_f32(void *out, const void *residual,
                                                  const int *residual_row_index, const void *bias,
                                                  const void *gamma, const void *beta,
                                                  const int *valid_rows, int rows_cap,
                                                  int hidden_dim, float eps, void *stream) {
  BT_REQUIRE(out && residual && bias && gamma && beta, BT_ERR_INVALID_ARGUMENT,
             "bt_add_bias_residual_layernorm_f32: null pointer argument");
  BT_REQUIRE(rows_cap >= 0, BT_ERR_INVALID_ARGUMENT,
             "bt_add_bias_residual_layernorm_f32: negative rows_cap");
  BT_REQUIRE(!residual_row_index || valid_rows, BT_ERR_INVALID_ARGUMENT,
             "bt_add_bias_residual_layernorm_f32: residual_row_index needs valid_rows");
  return launch_f32_ln<false>(out, residual, bias, gamma, beta, out, valid_rows,
                              residual_row_index, 1, rows_cap, hidden_dim, eps, as_stream(stream),
                              "bt_add_bias_residual_layernorm_f32");
}

extern "C" int bt_add_bias_residual_layernorm_f32_split(
    void *out, const void *residual, const int *residual_row_index, const void *bias, const void *gamma, const void *beta,
    const int *valid_rows, int rows_cap, int hidden_dim, float eps, void *pairs, int *exps, int *gelu_exps, const float *bounds,
    int bound_count, void *stream) {
  return bt_add_bias_residual_layernorm_f32_split_layer(out, residual, residual_row_index, bias, gamma, beta, valid_rows, rows_cap,
                                                        hidden_dim, eps, pairs, exps, gelu_exps, bounds, bound_count, nullptr, 0,
                                                        stream);
}

extern "C" int bt_add_bias_residual_layernorm_f32_split_layer(
    void *out, const void *residual, const int *residual_row_index, const void *bias, const void *gamma, const void *beta,
    const int *valid_rows, int rows_cap, int hidden_dim, float eps, void *pairs, int *exps, int *gelu_exps, const float *bounds,
    int bound_count, unsigned *raw, int n, void *stream) {
  const char *who = "bt_add_bias_residual_layernorm_f32_split";
  BT_REQUIRE(out && residual && bias && gamma && beta && pairs && exps && gelu_exps && bounds, BT_ERR_INVALID_ARGUMENT,
             "%s: null pointer argument", who);
  BT_REQUIRE(rows_cap >= 0 && bound_count > 0, BT_ERR_INVALID_ARGUMENT, "%s: rows_cap=%d bound_count=%d", who, rows_cap, bound_count);
  BT_REQUIRE(!raw || (n > 0 && split_raw_words(n) <= kWave), BT_ERR_INVALID_ARGUMENT, "%s: n=%d", who, n);   // (a word a lane)
  BT_REQUIRE(!residual_row_index || valid_rows, BT_ERR_INVALID_ARGUMENT, "%s: residual_row_index needs valid_rows", who);
  BT_REQUIRE(hidden_dim % 32 == 0 && aligned16({pairs}), BT_ERR_UNSUPPORTED,
             "%s: hidden_dim=%d must be a multiple of 32, the pairs 16-byte aligned", who, hidden_dim);
  const F32LnPairs next{(half_t *)pairs, exps, gelu_exps, bounds, bound_count, raw, raw ? split_raw_words(n) : 0};
  return launch_f32_ln<false>(out, residual, bias, gamma, beta, out, valid_rows, residual_row_index, 1, rows_cap, hidden_dim,
                              eps, as_stream(stream), who, &next);
}

extern "C" int bt_add_bias_residual_layernorm_restore_f32(
    const void *out, const void *residual, const void *bias, const void *gamma, const void *beta,
    void *out_padded, const int *batch_idx, int batch_size, int seq_len, int hidden_dim, float eps,
    void *stream) {
  BT_REQUIRE(out && residual && bias && gamma && beta && out_padded && batch_idx,
             BT_ERR_INVALID_ARGUMENT,
             "bt_add_bias_residual_layernorm_restore_f32: null pointer argument");
  BT_REQUIRE(batch_size > 0 && seq_len > 0, BT_ERR_INVALID_ARGUMENT,
             "bt_add_bias_residual_layernorm_restore_f32: sizes must be positive");
  BT_REQUIRE((long long)batch_size * seq_len < (1ll << 31), BT_ERR_UNSUPPORTED,
             "bt_add_bias_residual_layernorm_restore_f32: too many rows");
  return launch_f32_ln<true>(out, residual, bias, gamma, beta, out_padded, batch_idx, nullptr,
                             seq_len, batch_size * seq_len, hidden_dim, eps, as_stream(stream),
                             "bt_add_bias_residual_layernorm_restore_f32");
}
