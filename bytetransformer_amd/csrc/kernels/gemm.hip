// fp16 MFMA GEMM family for gfx950: C[rows, N] = A[rows, K] . W[K, N] with
// fp32 accumulation and three fused epilogues (plain store, +bias+tanh-GELU,
// +bias with the Q/K/V head split).  A is consumed k-contiguous as stored; W either
// as the row-major [K, N] matrix itself (its LDS tile is read with the LDS transpose
// read) or through the k-contiguous [N, K] pre-pack made by bt_transpose_weights.
//
// Structure of one workgroup (tile BM x BN, BK = 64):
//   * global -> LDS copies are 16-byte buffer loads with an LDS destination: no
//     staging registers, no ds_write; each wave instruction lands 1 KB = 8 tile
//     rows back to back in LDS.  Small tiles give this job to dedicated loader
//     waves so the computing waves' instruction streams hold MFMAs and LDS
//     reads only;
//   * the LDS image is XOR-swizzled on 16-byte chunks (slot = chunk ^ (row>>1 & 7));
//     the swizzle is applied by choosing which global chunk each lane fetches,
//     and makes the ds_read_b128 operand fetches conflict-free on the 64 banks;
//   * a ring of STAGES tiles, one barrier per k-step, vmcnt-counted waits so
//     later stages stay in flight across the barrier;
//   * v_mfma_f32_16x16x32_f16 with the weight tile as the MFMA "A" operand and
//     the activation tile as "B": a lane's four sums of a block are 4 consecutive
//     output columns of one row; operand fragments are double-buffered over
//     sub-steps of eight products;
//   * epilogue: bias / GELU on the accumulators, then each wave stages 32 rows
//     at a time through a private LDS tile and writes 16-byte, row-contiguous
//     global stores.
//   * workgroup -> tile order is XCD-aware: hardware deals consecutive
//     workgroup ids round-robin to the 8 XCDs, so id%8 selects a contiguous
//     range of the LIVE tiles (live = those below the device-side row count)
//     and the workgroups sharing an XCD's L2 also share operand panels.
//
// Rows are bounded on the device: the live row count is read from
// `valid_rows`; workgroups beyond the live tiles retire at once.
#include "gemm_common.h"
#include "mask_rows.h"

#include <cstring>
#include <type_traits>
#include <utility>

namespace bt {


// kEpiPartial: split-k launch (grid y = split): fp32 partial sums to c32[split][rows_cap][N]
// kEpiBias: + bias, row-major store (the QKV projection of layers whose head size is not 64)
enum Epilogue { kEpiPlain = 0, kEpiBiasGelu = 1, kEpiQkvSplit = 2, kEpiPartial = 3, kEpiBias = 4 };

struct GemmArgs {
  const half_t *a;      // [rows_cap, K]
  const half_t *wt;     // [N, K] (pre-packed), or [K, N] as the layer's weights are stored (w_kn)
  const half_t *bias;   // [N] or null
  half_t *c;            // [rows_cap, N]  (or [3][heads][rows_cap][64] for the QKV split)
  const int *valid_rows;
  const int *a_row_index;   // optional gather: A row r is a[a_row_index[r]] (null = identity)
  int rows_cap, N, K;
  int tiles_n;
  int rows_hint;        // host-side estimate of the live rows (0 = unknown); tile choice only
  float *c32;           // kEpiPartial only: [splits][rows_cap][N]
  int w_kn;             // 1: wt is the row-major [K, N] matrix itself
  // Rows taken straight from the attention mask (the QKV projection of a padding-free
  // layer): A is the padded [mask_B * mask_S, K] tensor, the live rows and their order are
  // what the mask's row lengths say, counted by every workgroup for itself - no launch
  // ahead of the product has to build a row index first.  Workgroup 0 leaves the offsets
  // for the kernels that follow (each pointer may be null).
  const void *mask;     // [mask_B, mask_S, mask_S] or null
  int mask_f32;         // element type: 0 half, 1 float
  int mask_B, mask_S;
  int *out_batch_idx;   // [mask_B + 1]
  int *out_word_idx;    // [mask_B * mask_S]: the complete row map (valid positions, then the padded ones)
  int *out_seq_order;   // [mask_B]
  int tile_grid;        // workgroups of the launch (set by the launcher)
  int splits;           // k slices (set by the launcher; 1 but for kEpiPartial)
  unsigned per_n;       // device only: inverse of tiles_n, for divide()
  unsigned ratio, per_n_second;   // gemm_either_kernel (set by the launcher)
};

// Where a product takes its rows from, as a template parameter: the code that counts the mask rows is 9 KB,
// three quarters of a small kernel, and the kernels of a layer share an instruction cache of 64 KB (12 layers
// without it where no mask is counted: 1 x 32 385 -> 374 us, 4 x 96 430 -> 422, 7 x 217 638 -> 626).

// What a product needs, as leading kernel arguments of their own: the first 64 bytes are in scalar registers when a
// wave starts, where the fields of a struct are memory reads, one more round trip ahead of the first load or store.
// `rows` is valid_rows, or the mask of a launch that counts its rows; `index` is a_row_index, or the counting launch's
// out_batch_idx; k_splits is K | splits << 24; per_n the inverse of the tile columns.
// (With the tile's column count, the row index and the pointers of bias and output behind them, and three
// divisions to find the tile, a small product took 0.3 us longer to its first load.)
#define BT_GEMM_FIRST                                                                              \
  const half_t *a, const half_t *wt, const void *rows, const int *index, const half_t *bias, void *out, \
      int rows_cap, int N, unsigned k_splits, unsigned per_n
#define BT_GEMM_FIRST_NAMES a, wt, rows, index, bias, out, rows_cap, N, k_splits, per_n
template <int MASK, typename Then>
static int with_first_arguments(const GemmArgs &p, Then then) {
  return then(p.a, p.wt, MASK != kMaskNone ? p.mask : (const void *)p.valid_rows,
              MASK != kMaskNone ? (const int *)p.out_batch_idx : p.a_row_index, p.bias, p.c32 ? (void *)p.c32 : (void *)p.c,
              p.rows_cap, p.N, (unsigned)p.K | (unsigned)p.splits << 24, inverse_of((unsigned)p.tiles_n));
}
// ... and what few need.  Every argument byte costs the host: beside ten leading arguments a launch takes
// 3.0 us to issue with 24 bytes more, 3.6 with 48, and 3.8 with the whole of GemmArgs (128), so the fields of a
// launch that counts mask rows, and the grid of one that loops, travel with those launches only.
template <int MASK>
struct GemmTail {
  int tile_grid, mask_B, mask_S;
  int *out_word_idx, *out_seq_order;
};
template <>
struct GemmTail<kMaskNone> {
  int tile_grid;
  unsigned ratio, per_n_second;   // gemm_either_kernel
  int unused;                     // (see Launch: 16 bytes are issued faster than 4)
};
template <int MASK>
static GemmTail<MASK> gemm_tail(const GemmArgs &p) {
  if constexpr (MASK == kMaskNone)
    return {p.tile_grid, p.ratio, p.per_n_second, 0};
  else
    return {p.tile_grid, p.mask_B, p.mask_S, p.out_word_idx, p.out_seq_order};
}
template <int MASK, int BN>
__device__ __forceinline__ GemmArgs gemm_args(BT_GEMM_FIRST, const GemmTail<MASK> &tail) {
  GemmArgs p{};
  p.a = a, p.wt = wt, p.bias = bias, p.c = (half_t *)out, p.c32 = (float *)out;
  p.rows_cap = rows_cap, p.N = N, p.K = (int)(k_splits & 0xffffffu), p.splits = (int)(k_splits >> 24);
  p.tiles_n = (N + BN - 1) / BN, p.per_n = per_n, p.tile_grid = tail.tile_grid;
  if constexpr (MASK == kMaskNone) {
    p.valid_rows = (const int *)rows, p.a_row_index = index;
  } else {
    p.mask = rows, p.out_batch_idx = const_cast<int *>(index);
    p.mask_B = tail.mask_B, p.mask_S = tail.mask_S;
    p.out_word_idx = tail.out_word_idx, p.out_seq_order = tail.out_seq_order;
  }
  return p;
}

// gemm_wave_k: columns of a tile, waves of a workgroup, k-steps in a wave's ring
constexpr int kWaveKCols = 32, kWaveKWaves = 4, kWaveKDepth = 3;

#if defined(__HIP_DEVICE_COMPILE__)
// One stage's loads of one wave: instruction i lands 8 tile rows (1 KB) at
// lds + i * lds_step; the first NIA instructions read A, the rest W.
template <int NI, int NIA, int COUNT = NI>
__device__ __forceinline__ void issue_stage_loads(rsrc_t rs_a, rsrc_t rs_w, const int (&voff)[NI],
                                                  half_t *lds, int lds_step, int k_bytes,
                                                  int k_bytes_w) {
#pragma unroll
  for (int i = 0; i < COUNT; ++i)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(i < NIA ? rs_a : rs_w,
                                             (__attribute__((address_space(3))) void *)(lds + i * lds_step),
                                             16, voff[i], i < NIA ? k_bytes : k_bytes_w, 0, 0);
}

// ---- the epilogue's wave-private staging tile -------------------------------------------
// 32 rows of WTN halfs, written 8 bytes per lane straight from the accumulator layout (lane l
// owns row l & 15 of a 16-row block, the 8-byte half (l >> 4) & 1 of a 16-byte chunk) and read back
// 16 bytes per lane, row-contiguous, for the global stores.  With 128-byte rows (WTN = 64) the tile is
// swizzled instead of padded: chunk ^= (row >> 1) & 7 and half ^= row & 1 put the 16 lanes
// of one write pass on 16 distinct bank pairs; a reader undoes the half swap in registers.
template <int WTN>
struct Staging {
  static constexpr bool kSwizzled = WTN == 64;
  static constexpr int kPitch = kSwizzled ? WTN : WTN + 8;   // halfs
  // where lane (row, half hf of the chunk) writes the 4 halfs of 16-byte chunk `chunk`
  __device__ static __forceinline__ int write_at(int row, int hf, int chunk) {
    if (kSwizzled) return row * kPitch + ((chunk ^ ((row >> 1) & 7)) << 3) + (((hf ^ row) & 1) << 2);
    return row * kPitch + (chunk << 3) + (hf << 2);
  }
  // the 8 halfs of chunk `chunk` of row `row`, in order
  __device__ static __forceinline__ uint4_t read(const half_t *st, int row, int chunk) {
    if (kSwizzled) {
      const uint4_t v = *(const uint4_t *)(st + row * kPitch + ((chunk ^ ((row >> 1) & 7)) << 3));
      return row & 1 ? uint4_t{v[2], v[3], v[0], v[1]} : v;
    }
    return *(const uint4_t *)(st + row * kPitch + (chunk << 3));
  }
};

// ---- a [K, N] weight tile of 256 columns through registers ----------------------------
// The LDS transpose read runs at half the rate of the 16-byte read, and the 256 x 256 tile
// (eight waves that load and compute, LDS reads ~ 3/4 of its MFMA time) is the one shape
// that cannot hide that.  There the 64 x 256 tile of a row-major [K, N] weight is fetched
// into registers instead - each of the 512 lanes takes a block of 4 k-rows x 8 columns, four
// 16-byte loads - transposed in the lane (16 byte permutes) and written k-contiguous with
// eight 8-byte LDS writes into the very image the pre-packed [N, K] layout lands in, so the
// k loop reads both layouts the same way.  Lane -> block: four consecutive lanes take four
// consecutive column blocks (64 contiguous bytes per k-row), the next lanes the next k-rows.
// Which lanes write odd rows first and which even ones, together with the image's swizzle,
// puts the 32 lanes of one write pass on 32 distinct bank pairs.
struct RegW {
  uint4_t r[4];        // k-rows k_base .. k_base + 3, columns n_base .. n_base + 7
  int voff[4];         // byte offsets of the four loads from the tile's first element
  int woff[8];         // LDS offsets (halfs, from the W image of a stage) of the eight writes
  unsigned sel[2];     // permute selectors of even / odd write instructions
};
__device__ __forceinline__ void regw_setup(RegW &w, int wave, int lane, int N, int cols, int BM) {
  // (eight consecutive lanes on whole 128-byte lines measured slower: their writes then
  // collide two ways, and the memory side does not mind the 64-byte pieces)
  const int kq = lane >> 2, ngl = lane & 3, ng = wave * 4 + ngl;
  const int bit = ngl >> 1;
  const int k_base = 4 * kq, n_base = 8 * ng;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    w.voff[i] = n_base < cols ? ((k_base + i) * N + n_base) * (int)sizeof(half_t) : 0x7ffffff0;
  const int c = kq >> 1, h = kq & 1;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int n = n_base + (i ^ bit);
    w.woff[i] = n * kBK + ((c ^ swz(n + BM)) << 3) + h * 4;
  }
  // write i moves column n_base + (i ^ bit): its halfs are the low or the high halves of
  // dword (i >> 1) of the four loads
  w.sel[0] = bit ? 0x07060302u : 0x05040100u;
  w.sel[1] = bit ? 0x05040100u : 0x07060302u;
}
__device__ __forceinline__ void regw_load(RegW &w, rsrc_t rs_w, int k_bytes_w) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
    w.r[i] = __builtin_amdgcn_raw_buffer_load_b128(rs_w, w.voff[i], k_bytes_w, 0);
}
__device__ __forceinline__ void regw_store(const RegW &w, half_t *sW) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const unsigned lo = __builtin_amdgcn_perm(w.r[1][i >> 1], w.r[0][i >> 1], w.sel[i & 1]);
    const unsigned hi = __builtin_amdgcn_perm(w.r[3][i >> 1], w.r[2][i >> 1], w.sel[i & 1]);
    *(uint2_t *)(sW + w.woff[i]) = uint2_t{lo, hi};
  }
}

// ---- a wave's share of a tile: products and stores ----------------------------------------
// 16x16 blocks on v_mfma_f32_16x16x32_f16, the weight as its "A" operand: a lane's four sums of block
// (i, j) are columns 16 i + 4 (lane >> 4) .. + 3 of row 16 j + (lane & 15).
// The chip runs these loops against its power limit (1.8 to 2.1 GHz of 2.4 in forwards of some thousand
// rows), and this instruction does more with it than v_mfma_f32_32x32x16_f16: on operands in
// registers 1870 against 1600 TFLOP/s, with the loop's LDS reads 1585 against 1420 (8 waves, 64x128).
// Products of a forward, with the reads placed by hand (`schedule`): FFN1 at 4800 rows 30.9 -> 29.5 us, at
// 9830 rows 56.6 -> 53.6, FFN2 27.4 -> 24.6 and 46.9 -> 43.9, projection 11.1 -> 9.9.
template <int BM, int BN, int WTM, int WTN, bool TR>
struct WaveTile {
  static constexpr int TM = WTM / 16, TN = WTN / 16;
  // A large wave tile takes its longer side in parts of eight products (the reads for the next eight then
  // fit under them and the fragments requested ahead fit the registers); the other side's fragments serve
  // all parts of 32 k.
  static constexpr bool kByRows = TM > TN;
  static constexpr int PARTS = TM * TN <= 8 ? 1 : TM * TN / 8;
  static_assert((kByRows ? TM : TN) % PARTS == 0, "whole parts");
  static constexpr int PM = kByRows ? TM / PARTS : TM, PN = kByRows ? TN : TN / PARTS;
  static constexpr int SUBSTEPS = kBK / 32 * PARTS;
  float4_t acc[TN][TM];
  half8_t fw[2][PN], fa[2][PM];

  // the sums start from the bias of their columns (n: column of this lane's first sum in block 0)
  template <bool BIAS>
  __device__ __forceinline__ void start(const half_t *bias, int n, int n_last) {
#pragma unroll
    for (int i = 0; i < TN; ++i) {
      float4_t init = {0.f, 0.f, 0.f, 0.f};
      if (BIAS) {
        const half4_t b = *(const half4_t *)(bias + min(n + i * 16, n_last));
#pragma unroll
        for (int e = 0; e < 4; ++e) init[e] = (float)b[e];
      }
#pragma unroll
      for (int j = 0; j < TM; ++j) acc[i][j] = init;
    }
  }

  // fragments of sub-step u (32 k, one part) of the k-step whose tiles lie at sA; the wave tile starts at
  // row m_w and column n_w of the tile
  __device__ __forceinline__ void load(const half_t *sA, int m_w, int n_w, int lane, int u) {
    const half_t *sW = sA + BM * kBK;
    const int ks = u / PARTS, part = u % PARTS;
    const int fr = lane & 15, chunk = 4 * ks + (lane >> 4);
    if (!kByRows || part == 0) {
#pragma unroll
      for (int i = 0; i < PN; ++i) {
        const int n = n_w + ((kByRows ? 0 : part * PN) + i) * 16;
        fw[(kByRows ? ks : u) & 1][i] = TR ? load_kn_frag<BN>(sW, n, 32 * ks, lane)
                                           : *(const half8_t *)(sW + (n + fr) * kBK + ((chunk ^ swz(n + fr + BM)) * 8));
      }
    }
    if (kByRows || part == 0) {
#pragma unroll
      for (int j = 0; j < PM; ++j) {
        const int r = m_w + ((kByRows ? part * PM : 0) + j) * 16 + fr;
        fa[(kByRows ? u : ks) & 1][j] = *(const half8_t *)(sA + r * kBK + ((chunk ^ swz(r)) * 8));
      }
    }
  }

  // Where the LDS reads of a k-step go: those of sub-step u + 1 are spread over the products of sub-step
  // u, one read (two transpose reads where there are more reads than products) ahead of every few of them.
  template <int U>
  __device__ __forceinline__ static void schedule_substep() {
    constexpr bool kNext = U + 1 < SUBSTEPS, kFirst = (U + 1) % PARTS == 0;
    constexpr int R = (kNext && (!kByRows || kFirst) ? PN * (TR ? 2 : 1) : 0) + (kNext && (kByRows || kFirst) ? PM : 0);
    constexpr int P = PN * PM, G = R < P ? (R > 0 ? R : 1) : P;   // groups of reads and products
    if constexpr (R > 0) {
#pragma unroll
      for (int g = 0; g < G; ++g) {
        __builtin_amdgcn_sched_group_barrier(kSchedLdsRead, (R + G - 1) / G, 0);
        __builtin_amdgcn_sched_group_barrier(kSchedMfma, P / G, 0);
      }
    }
    if constexpr (R == 0 || P % G != 0) __builtin_amdgcn_sched_group_barrier(kSchedMfma, R == 0 ? P : P % G, 0);
  }
  template <int... U>
  __device__ __forceinline__ static void schedule(std::integer_sequence<int, U...>) {
    __builtin_amdgcn_sched_group_barrier(kSchedLdsRead, PN * (TR ? 2 : 1) + PM, 0);
    (schedule_substep<U>(), ...);
  }

  // one k-step; `between(u)` runs ahead of the products of sub-step u
  template <typename Between>
  __device__ __forceinline__ void step(const half_t *sA, int m_w, int n_w, int lane, Between between) {
    load(sA, m_w, n_w, lane, 0);
#pragma unroll
    for (int u = 0; u < SUBSTEPS; ++u) {
      if (u + 1 < SUBSTEPS) load(sA, m_w, n_w, lane, u + 1);
      between(u);
      const int ks = u / PARTS, part = u % PARTS;
      const int bw = (kByRows ? ks : u) & 1, ba = (kByRows ? u : ks) & 1;
#pragma unroll
      for (int i = 0; i < PN; ++i)
#pragma unroll
        for (int j = 0; j < PM; ++j) {
          float4_t &sum = acc[(kByRows ? 0 : part * PN) + i][(kByRows ? part * PM : 0) + j];
          sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(fw[bw][i], fa[ba][j], sum, 0, 0, 0);
        }
    }
    schedule(std::make_integer_sequence<int, SUBSTEPS>{});
  }

  // 32 rows at a time through the wave-private staging tile `st`; (m_first, n_first): the wave tile's
  // corner in C
  template <int EPI>
  __device__ __forceinline__ void store(const GemmArgs &p, half_t *st, int m_first, int n_first, int M,
                                        int lane) {
    constexpr int CPRW = WTN / 8;   // 16-byte chunks per staged row
    constexpr int RPS = 64 / CPRW;  // rows per store instruction
    const int sr = lane / CPRW, sc = (lane % CPRW) * 8;
#pragma unroll
    for (int j = 0; j < TM; ++j) {
#pragma unroll
      for (int i = 0; i < TN; ++i) {
        float4_t v = acc[i][j];
        if (EPI == kEpiBiasGelu) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = gelu_tanh_f32(v[e]);
        }
        *(half4_t *)(st + Staging<WTN>::write_at((j & 1) * 16 + (lane & 15), (lane >> 4) & 1, i * 2 + (lane >> 5))) =
            half4_t{(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]};
      }
      if ((j & 1) == 0) continue;
#pragma unroll
      for (int r0 = 0; r0 < 32; r0 += RPS) {
        const int r = r0 + sr;
        if (sr >= RPS || r >= 32) continue;   // lanes left over when 64 % CPRW != 0
        const int m = m_first + (j - 1) * 16 + r, n = n_first + sc;
        const uint4_t v = Staging<WTN>::read(st, r, sc >> 3);
        if (m < M && n < p.N) {
          if (EPI == kEpiQkvSplit) {
            // column n = which*H + g*64 + dd  ->  [which*heads + g][m][dd]
            store_through(p.c + ((size_t)(n >> 6) * p.rows_cap + m) * 64 + (n & 63), v);
          } else {
            store_through(p.c + (size_t)m * p.N + n, v);
          }
        }
      }
    }
  }
};

// XCD-aware tile order over the live tiles of M rows: position `bid` of `end`; false: it has no tile.  The k slices of a
// split launch follow each other in it.  (As rows of the grid they left the workgroups of the dead rows
// between them, and the live ones of the second slice came to lie on the CUs of the first: 230 of 384 rows,
// hidden 768, FFN2 in two slices with the LayerNorm behind it 13.6 -> 11.1 us.)
constexpr int kColumnRows = 256;   // rows of the launches whose 32-row tiles go column by column
template <int BM, int BN>
__device__ __forceinline__ bool tile_at(const GemmArgs &p, int M, int bid, int &split, int &tile_m, int &tile_n) {
  const int tiles_m = (M + BM - 1) / BM;
  const int tiles = tiles_m * p.tiles_n;
  const int live = tiles * p.splits;
  const int per = (live + 7) >> 3;
  int L = (bid & 7) * per + (bid >> 3);
  if (bid >= per * 8 || L >= live) return false;
  split = 0;
  if (p.splits > 1)
    for (; L >= tiles; L -= tiles) ++split;
  if (BM == 32 && tiles_m > 1 && live < kMostPanelTiles) {
    // A few hundred rows: the launch is as long as it takes to fetch the weight, and in row-major
    // order every XCD fetches all of it (256 rows, QKV at hidden 768: 28 MB in all against
    // 7 MB in panels; 12 layers at batch 1 x 256: -8 %).  Up to 256 rows the order is column by column: an XCD has an
    // eighth of the weight to itself however many the rows, the eighth that the attention's launch has put into
    // its L2 (warm_slice).  12 layers in panels (two or three tile rows row-major, as one always is) and so, us: as
    // stored 1 x 64 346 -> 342, 1 x 128 376 -> 369, pre-packed 2 x 64 361 -> 354; 8 x 64, some 300 rows, 440 -> 444.  With
    // the larger tiles neither gains anything (64 x 64: 1 x 256 416 -> 422) and the index arithmetic costs up to 1 %.
    if (tiles_m <= kColumnRows / BM) {
      const int column = divide_small(L, tiles_m);
      tile_m = L - column * tiles_m;
      tile_n = column;
    } else {
      tile_panels<BM, BN>(tiles_m, p.tiles_n, per).locate(L, tile_m, tile_n);
    }
  } else {
    tile_m = (int)divide((unsigned)L, (unsigned)p.tiles_n, p.per_n);
    tile_n = L - tile_m * p.tiles_n;
  }
  return true;
}

template <int BM, int BN, int STAGES, int WM, int WN, int NP, int EPI, bool WKN, int MASK, bool LOOP>
__device__ __forceinline__ int gemm_tile(const GemmArgs &p, const int bid) {
  constexpr int BK = kBK;
  constexpr int NW = WM * WN;                   // waves that run the MFMAs
  constexpr int NL = NP > 0 ? NP : NW;          // waves that issue the global loads
  constexpr int WTM = BM / WM, WTN = BN / WN;   // wave tile
  constexpr int ROWS = BM + BN;                 // A rows then W rows in one stage
  constexpr int NI = ROWS / 8 / NL;             // load instructions per loading wave per stage
  constexpr int NIA = BM / 8 / NL;              // ... of which the first NIA fetch A rows
  constexpr int STAGE_HALFS = ROWS * BK;
  static_assert(BM % (8 * NL) == 0 && BN % (8 * NL) == 0, "tile rows must split evenly over the loading waves");
  static_assert(STAGES >= 2 && STAGES <= 5 && (STAGES - 2) * NI < 64, "pipeline depth");
  constexpr int YOUNG = STAGES - 2;   // stages that may still be in flight at a barrier
  // a [K, N] weight tile goes through registers (see RegW) where every wave loads and computes
  constexpr bool kRegW = WKN && NP == 0 && BN == 256 && NW == 8 && STAGES == 2;

  extern __shared__ __attribute__((aligned(1024))) half_t gemm_smem[];
  half_t *smem = gemm_smem;

  int tid = threadIdx.x;
  if constexpr (LOOP) asm volatile("" : "+v"(tid));   // (so that its uses are not computed ahead of the loop and kept)
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int M;
  MaskRows mr{};
  if constexpr (MASK != kMaskNone) {
    // the last ring stage is first written after the first barrier of the k loop, which
    // every wave reaches only after it has read the lengths
    mr = mask_rows_setup<MASK>(p, wave, NW + NP, lane, (int *)(smem + (STAGES - 1) * STAGE_HALFS));
    M = min(mr.M, p.rows_cap);
    if (bid == 0 && wave < NW) mask_rows_write(p, mr, tid, NW * 64, lane);
  } else {
    M = p.valid_rows ? min(*p.valid_rows, p.rows_cap) : p.rows_cap;
  }

  int split, tile_m, tile_n;
  if (!tile_at<BM, BN>(p, M, bid, split, tile_m, tile_n)) return 0;
  const int end = ((M + BM - 1) / BM * p.tiles_n * p.splits + 7) / 8 * 8;
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  // slice y of a split-k launch: the k range [y, y + 1) * K / splits
  const int nk = EPI == kEpiPartial ? divide_small(p.K / BK, p.splits) : p.K / BK;
  const int k_first = EPI == kEpiPartial ? split * nk * BK : 0;

  // ---- loading side ---------------------------------------------------------
  // Global -> LDS copies are buffer loads with the LDS destination: descriptor and
  // k offset in scalar registers, one fixed 32-bit byte offset per lane and load.
  // (Beside a wave that keeps the MFMA pipe full this form issues at the full
  // 64 B/clk of the vector memory path; the flat-address form drops to half.)
  // Load instruction i of loading wave w fills tile rows [(i*NL + w)*8, +8); a lane
  // fetches the chunk that the swizzle places in its slot.  Rows past the last live one and
  // columns past the end of the weight fall outside the descriptor and read as zero.  (Nothing has
  // written the dead rows in this call: they would come from HBM, and the last row of tiles would take up to
  // twice as long as the others for them.  Six heads of 128, 8 x 300, 1416 rows, FFN2: the loops of that tile row 15.6 us,
  // of the others 8.1 to 9.1; 12 layers 861 -> 783 us, twelve heads, 19 x 26, 479 -> 463.)
  //
  // With NP == 0 every wave loads its share and then computes.  With NP > 0 the
  // last NP waves only load: the vector-memory unit accepts one 1 KB instruction
  // per 16 clocks, and a wave that has to push its loads through that queue at the
  // top of every k-step cannot feed the MFMA pipe meanwhile; for small tiles
  // (load clocks ~ MFMA clocks) that serialisation costs half of the throughput.
  const bool loader = NP == 0 || wave >= NW;
  const int lw = NP == 0 ? wave : wave - NW;    // index among the loading waves
  const bool gather = MASK != kMaskNone || p.a_row_index != nullptr;
  const rsrc_t rs_a =
      gather ? make_rsrc(p.a + k_first, ((size_t)p.rows_cap * p.K - k_first) * sizeof(half_t))
             : make_rsrc(p.a + (size_t)m0 * p.K + k_first,
                         ((size_t)(M - m0) * p.K - k_first) * sizeof(half_t));
  // the weight tile: BN rows of 64 k ([N, K] pre-pack), or 64 k-rows of BN columns ([K, N]);
  // 1 KB per load instruction either way
  const rsrc_t rs_w =
      WKN ? make_rsrc(p.wt + (size_t)k_first * p.N + n0,
                      ((size_t)(p.K - k_first) * p.N - n0) * sizeof(half_t))
          : make_rsrc(p.wt + (size_t)n0 * p.K + k_first,
                      ((size_t)(p.N - n0) * p.K - k_first) * sizeof(half_t));
  int voff[NI];
  if (loader) {
    MaskRowSpan span{};
    if constexpr (MASK != kMaskNone) span = mask_rows_span(mr, p.mask_B, lane, m0, min(m0 + BM, M) - 1);
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int r = (i * NL + lw) * 8 + (lane >> 3);
      const int kc = (lane & 7) ^ swz(r);
      int row = i < NIA ? r : r - BM;
      if (i < NIA && gather) {   // live rows only hold valid indices
        const int live_row = min(m0 + r, M - 1);
        row = MASK != kMaskNone ? mask_rows_map(mr, span, live_row) : p.a_row_index[live_row];
      }
      voff[i] = (row * p.K + kc * 8) * (int)sizeof(half_t);
      if (WKN && i >= NIA) voff[i] = kn_load_offset<BN>((i - NIA) * NL + lw, lane, p.N, p.N - n0);
    }
  }
  const int w_step_bytes = (WKN ? BK * p.N : BK) * (int)sizeof(half_t);   // one k-step further
  RegW rw;
  if (kRegW) regw_setup(rw, wave, lane, p.N, p.N - n0, BM);
#define BT_ISSUE_LOADS(kt, stage)                                                              \
  issue_stage_loads<NI, NIA, kRegW ? NIA : NI>(                                                \
      rs_a, rs_w, voff, smem + (stage)*STAGE_HALFS + lw * 8 * BK, NL * 8 * BK,                 \
      (kt)*BK * (int)sizeof(half_t), (kt)*w_step_bytes)
  // Register-staged weight tile: one register set.  The loads of k-step s + 1 go out early in
  // step s - 1 (right after the registers have been emptied into LDS), have the rest of that
  // step and the start of step s to arrive, and are written to LDS early in step s, behind
  // the first quarter of its MFMAs: neither the loads nor the writes are waited for where
  // they were issued.  In vmcnt terms every wait is "at most the NIA youngest outstanding":
  // at the top of a step those are the weight loads (the A tile's direct-to-LDS loads are
  // older), at the write they are the A tile's loads of the next step.
#define BT_LOAD_W(kt) regw_load(rw, rs_w, (kt)*w_step_bytes)
#define BT_STORE_W(stage) regw_store(rw, smem + (stage)*STAGE_HALFS + BM * BK)
  static_assert(!kRegW || NIA == 4, "the weight tile's four loads per lane pair with four A loads");

  if (loader) {
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s)
      if (s < nk) BT_ISSUE_LOADS(s, s);
    if (kRegW) {
      BT_LOAD_W(0);
      wait_vmcnt<0>();
      BT_STORE_W(0);
      if (nk > 1) BT_LOAD_W(1);
    }
  }

  if (NP > 0 && wave >= NW) {
    // pure loader: one barrier per k-step, in step with the computing waves
    int stage = 0;
    for (int kt = 0; kt < nk; ++kt) {
      wait_stages<NI, YOUNG>(nk - 1 - kt);       // this wave's part of tile kt has landed
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();               // tile kt is complete; stage of tile kt-1 is free
      asm volatile("" ::: "memory");
      if (kt + STAGES - 1 < nk) {
        int ps = stage + STAGES - 1;
        if (ps >= STAGES) ps -= STAGES;
        BT_ISSUE_LOADS(kt + STAGES - 1, ps);
      }
      if (++stage == STAGES) stage = 0;
    }
    __builtin_amdgcn_s_barrier();                 // pairs with the barrier before the epilogue
    return end;
  }

  // ---- computing side -------------------------------------------------------
  const int wm = wave / WN, wn = wave % WN;
  constexpr bool kHasBias = EPI == kEpiBiasGelu || EPI == kEpiQkvSplit || EPI == kEpiBias;
  WaveTile<BM, BN, WTM, WTN, WKN && !kRegW> tile;
  tile.template start<kHasBias>(p.bias, n0 + wn * WTN + (lane >> 4) * 4, p.N - 4);
  int stage = 0;
  for (int kt = 0; kt < nk; ++kt) {
    // tile kt has landed for this wave once only the younger stages' loads are outstanding
    if (kRegW) {
      // this wave's A loads of tile kt and its LDS writes of the W tile; the weight loads of
      // tile kt + 1 stay in flight
      if (kt + 1 < nk)
        __builtin_amdgcn_s_waitcnt(0x0074);   // vmcnt(4) lgkmcnt(0)
      else
        __builtin_amdgcn_s_waitcnt(0x0070);   // vmcnt(0) lgkmcnt(0)
    } else if (NP == 0)
      wait_stages<NI, YOUNG>(nk - 1 - kt);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();   // everyone's tile is in LDS; stage (kt-1) is free again
    asm volatile("" ::: "memory");
    if (NP == 0 && kt + STAGES - 1 < nk) {
      int ps = stage + STAGES - 1;
      if (ps >= STAGES) ps -= STAGES;
      BT_ISSUE_LOADS(kt + STAGES - 1, ps);
    }
    tile.step(smem + stage * STAGE_HALFS, wm * WTM, wn * WTN, lane, [&](int u) {
      if (kRegW && u == 2 && kt + 1 < nk) {
        wait_vmcnt<NIA>();            // the weight registers of step kt + 1 (older than its A loads)
        BT_STORE_W(stage ^ 1);
        if (kt + 2 < nk) BT_LOAD_W(kt + 2);
      }
    });
    if (++stage == STAGES) stage = 0;
  }

#undef BT_ISSUE_LOADS
#undef BT_LOAD_W
#undef BT_STORE_W
  // ---- epilogue -------------------------------------------------------------
  constexpr int EP = Staging<WTN>::kPitch;   // pitch (halfs) of the wave-private staging tile
  static_assert((size_t)NW * 32 * EP <= (size_t)STAGES * STAGE_HALFS, "staging fits the ring");
  __builtin_amdgcn_s_barrier();   // all waves are done with the last stage
  if (EPI == kEpiPartial) {
    // fp32 partial sums straight from the accumulators: 16 bytes per lane and block
    float *dst = p.c32 + (size_t)split * p.rows_cap * p.N;
#pragma unroll
    for (int j = 0; j < WTM / 16; ++j) {
      const int m = m0 + wm * WTM + j * 16 + (lane & 15);
#pragma unroll
      for (int i = 0; i < WTN / 16; ++i) {
        const int n = n0 + wn * WTN + i * 16 + (lane >> 4) * 4;
        if (m < M && n < p.N)
          store_through(dst + (size_t)m * p.N + n, __builtin_bit_cast(uint4_t, tile.acc[i][j]));
      }
    }
    return end;
  }
  tile.template store<EPI>(p, smem + wave * 32 * EP, m0 + wm * WTM, n0 + wn * WTN, M, lane);
  return end;
}

// ---- persistent form ---------------------------------------------------------------
// The launch has about one workgroup per CU and every workgroup takes SEVERAL tiles of its
// XCD's range, running ONE software pipeline over all their k-steps: the loads of the next
// tile's first stages are in flight while the current tile's accumulators are stored, and
// a tile's stores drain to memory under the next tile's products instead of in one burst of
// the whole launch at its end.  (One tile per workgroup leaves the matrix pipe idle from
// the first store instruction on: with 228 tiles on 256 CUs the last 7 us of the 31 us of
// the FFN1 product at batch 16 x 512 are 29.5 MB of stores.)  The grid no longer depends
// on the row count: a workgroup counts its tiles from the device-side row count.
template <int BM, int BN, int STAGES, int WM, int WN, int NP, int EPI, bool WKN, int MASK>
__device__ __forceinline__ void gemm_tiles_flat(const GemmArgs &p) {
  constexpr int BK = kBK;
  constexpr int NW = WM * WN;
  constexpr int NL = NP > 0 ? NP : NW;
  constexpr int WTM = BM / WM, WTN = BN / WN;
  constexpr int ROWS = BM + BN;
  constexpr int NI = ROWS / 8 / NL;
  constexpr int NIA = BM / 8 / NL;
  constexpr int STAGE_HALFS = ROWS * BK;
  static_assert(BM % (8 * NL) == 0 && BN % (8 * NL) == 0, "tile rows must split evenly over the loading waves");
  static_assert(STAGES >= 2 && STAGES <= 5 && (STAGES - 2) * NI < 64, "pipeline depth");
  static_assert(EPI != kEpiPartial, "split-k launches keep one tile per workgroup");
  constexpr int YOUNG = STAGES - 2;
  constexpr int EP = Staging<WTN>::kPitch;   // pitch (halfs) of the wave-private staging tile
  static_assert((size_t)NW * 32 * EP <= (size_t)STAGE_HALFS, "staging fits one stage of the ring");

  extern __shared__ __attribute__((aligned(1024))) half_t gemm_smem[];
  half_t *smem = gemm_smem;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int bid = (int)blockIdx.x;
  int M;
  MaskRows mr{};
  if constexpr (MASK != kMaskNone) {
    // (the last ring stage: first written after the first barrier of the k loop)
    mr = mask_rows_setup<MASK>(p, wave, NW + NP, lane, (int *)(smem + (STAGES - 1) * STAGE_HALFS));
    M = min(mr.M, p.rows_cap);
    if (bid == 0 && wave < NW) mask_rows_write(p, mr, tid, NW * 64, lane);
  } else {
    M = p.valid_rows ? min(*p.valid_rows, p.rows_cap) : p.rows_cap;
  }

  // XCD x owns the contiguous range [x * per, (x + 1) * per) of the live tiles; its
  // workgroups take them round-robin
  const auto tile_row = [&](int L) { return (int)divide((unsigned)L, (unsigned)p.tiles_n, p.per_n); };
  const int live = ((M + BM - 1) / BM) * p.tiles_n;
  const int per = (live + 7) >> 3;
  const int wgx = p.tile_grid >> 3;                      // workgroups per XCD
  const int lo = (bid & 7) * per;
  const int hi = min(lo + per, live);
  const int L0 = lo + (bid >> 3);
  if (L0 >= hi) return;
  const int n_my = (hi - L0 + wgx - 1) / wgx;
  const int nk = p.K / BK;
  const int total = n_my * nk;                           // k-steps of this workgroup

  // ---- loading side: a cursor (tile, k-step) STAGES - 1 steps ahead of the products ----
  const bool loader = NP == 0 || wave >= NW;
  const int lw = NP == 0 ? wave : wave - NW;
  const bool gather = MASK != kMaskNone || p.a_row_index != nullptr;
  rsrc_t rs_a = make_rsrc(p.a, 0), rs_w = make_rsrc(p.wt, 0);
  constexpr bool kHasBias = EPI == kEpiBiasGelu || EPI == kEpiQkvSplit || EPI == kEpiBias;
  // The bias of a tile's columns reaches the computing waves through LDS, fetched by the
  // first loading wave together with the tile's first k-step: a global load in a computing
  // wave after its stores would wait for every one of them to complete - the very wait this
  // form of the kernel exists to avoid.  (Only the first tile's bias is loaded directly.)
  // It is requested as soon as the cursor moves to the tile, one k-step ahead of the tile's
  // first loads (so that the wait for those loads' predecessors covers it), and the cursor
  // runs STAGES - 1 k-steps ahead of the products: with k = 64 (one k-step per tile) up to
  // STAGES biases are waiting to be read, hence STAGES buffers, taken in turn.
  half_t *s_bias = smem + STAGES * STAGE_HALFS;          // [STAGES][BN]
  const rsrc_t rs_bias = make_rsrc(kHasBias ? p.bias : p.wt, kHasBias ? (size_t)p.N * sizeof(half_t) : 0);
  int voff[NI];
  int idx_next[NIA];   // gathered A rows of the tile after the one being loaded
  int ld_L = L0, ld_kt = 0, ld_left = loader ? total : 0;
  int ld_slot = 0;     // bias buffer of the tile being set up: its position in the sequence mod STAGES
  auto fetch_indices = [&](int Lt) {
    const int m0 = tile_row(Lt) * BM;
    MaskRowSpan span{};
    if constexpr (MASK != kMaskNone) span = mask_rows_span(mr, p.mask_B, lane, m0, min(m0 + BM, M) - 1);
#pragma unroll
    for (int i = 0; i < NIA; ++i) {
      const int r = (i * NL + lw) * 8 + (lane >> 3);
      const int live_row = min(m0 + r, M - 1);   // live rows only hold valid indices
      idx_next[i] = MASK != kMaskNone ? mask_rows_map(mr, span, live_row) : p.a_row_index[live_row];
    }
  };
  auto load_setup = [&](int Lt, bool more, bool bias_to_lds) {
    const int tm = tile_row(Lt), tn = Lt - tm * p.tiles_n;
    const int m0 = tm * BM, n0 = tn * BN;
    if (kHasBias && bias_to_lds && lw == 0) {
      // 4 bytes per lane and instruction: 128 columns each
#pragma unroll
      for (int i = 0; i < BN / 128; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rs_bias,
            (__attribute__((address_space(3))) void *)(s_bias + ld_slot * BN + i * 128), 4,
            (lane + i * 64) * 4, n0 * (int)sizeof(half_t), 0, 0);
    }
    rs_a = gather ? make_rsrc(p.a, (size_t)p.rows_cap * p.K * sizeof(half_t))
                  : make_rsrc(p.a + (size_t)m0 * p.K, (size_t)(M - m0) * p.K * sizeof(half_t));
    rs_w = WKN ? make_rsrc(p.wt + n0, ((size_t)p.K * p.N - n0) * sizeof(half_t))
               : make_rsrc(p.wt + (size_t)n0 * p.K, (size_t)(p.N - n0) * p.K * sizeof(half_t));
    if (WKN && (p.N % BN) != 0) {
      // the column mask of the weight loads depends on the tile's first column
#pragma unroll
      for (int i = NIA; i < NI; ++i)
        voff[i] = kn_load_offset<BN>((i - NIA) * NL + lw, lane, p.N, p.N - n0);
    }
    if (gather) {
#pragma unroll
      for (int i = 0; i < NIA; ++i) {
        const int r = (i * NL + lw) * 8 + (lane >> 3);
        const int kc = (lane & 7) ^ swz(r);
        voff[i] = (idx_next[i] * p.K + kc * 8) * (int)sizeof(half_t);
      }
      if (more) fetch_indices(Lt + wgx);
    }
  };
  if (loader) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int r = (i * NL + lw) * 8 + (lane >> 3);
      const int kc = (lane & 7) ^ swz(r);
      const int row = i < NIA ? r : r - BM;
      voff[i] = (row * p.K + kc * 8) * (int)sizeof(half_t);
      if (WKN && i >= NIA) voff[i] = kn_load_offset<BN>((i - NIA) * NL + lw, lane, p.N, BN);
    }
    if (gather) fetch_indices(L0);
    load_setup(L0, n_my > 1, false);
  }
  // issues the loads of the cursor's k-step into `stage` and moves the cursor on
  auto issue_next = [&](int stage) {
    if (ld_left == 0) return;
    issue_stage_loads<NI, NIA>(rs_a, rs_w, voff, smem + stage * STAGE_HALFS + lw * 8 * BK,
                               NL * 8 * BK, ld_kt * BK * (int)sizeof(half_t),
                               ld_kt * (WKN ? BK * p.N : BK) * (int)sizeof(half_t));
    --ld_left;
    if (++ld_kt == nk) {
      ld_kt = 0;
      ld_L += wgx;
      if (++ld_slot == STAGES) ld_slot = 0;
      if (ld_left) load_setup(ld_L, ld_left > nk, true);
    }
  };
  if (loader) {
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s) issue_next(s);
  }

  if (NP > 0 && wave >= NW) {
    // pure loader: one barrier per k-step in step with the computing waves, one more at
    // the end of every tile (the computing waves then overlay the consumed stage)
    int stage = 0, kt = 0;
    for (int g = 0; g < total; ++g) {
      wait_stages<NI, YOUNG>(total - 1 - g);
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      int ps = stage + STAGES - 1;
      if (ps >= STAGES) ps -= STAGES;
      issue_next(ps);
      if (++kt == nk) {
        kt = 0;
        __builtin_amdgcn_s_barrier();
      }
      if (++stage == STAGES) stage = 0;
    }
    return;
  }

  // ---- computing side ---------------------------------------------------------------
  const int wm = wave / WN, wn = wave % WN;
  WaveTile<BM, BN, WTM, WTN, WKN> tile;
  const int n_lane = wn * WTN + (lane >> 4) * 4;
  int cL = L0, c_slot = 0;
  // the first tile's bias straight from memory
  tile.template start<kHasBias>(p.bias, (cL - tile_row(cL) * p.tiles_n) * BN + n_lane, p.N - 4);

  int stage = 0, kt = 0;
  for (int g = 0; g < total; ++g) {
    if (NP == 0) wait_stages<NI, YOUNG>(total - 1 - g);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();   // everyone's k-step g is in LDS; the stage of step g-1 is free again
    asm volatile("" ::: "memory");
    if (NP == 0) {
      int ps = stage + STAGES - 1;
      if (ps >= STAGES) ps -= STAGES;
      issue_next(ps);
    }
    tile.step(smem + stage * STAGE_HALFS, wm * WTM, wn * WTN, lane, [](int) {});
    if (++kt == nk) {
      // ---- this tile is complete: store it, start the next from its bias ----
      kt = 0;
      const int tm = tile_row(cL), tn = cL - tm * p.tiles_n;
      const int m0 = tm * BM, n0 = tn * BN;
      __builtin_amdgcn_s_barrier();   // all waves are done reading this stage: it becomes the staging area
      tile.template store<EPI>(p, smem + stage * STAGE_HALFS + wave * 32 * EP, m0 + wm * WTM, n0 + wn * WTN, M, lane);
      cL += wgx;
      if (++c_slot == STAGES) c_slot = 0;
      // (from LDS, where the loading side has put it)
      if (g + 1 < total) tile.template start<kHasBias>(s_bias + c_slot * BN, n_lane, BN - 4);
    }
    if (++stage == STAGES) stage = 0;
  }
}

#endif  // __HIP_DEVICE_COMPILE__

// ---- launches of more capacity than rows -------------------------------------------------
// A workgroup that finds no rows needs as much LDS as one that does, and waits for it: with workgroups for the
// padded batch (16 x 512, 4800 of 8192 rows) QKV took 23.1 us instead of 20.9, FFN1 27.6 (26.0), the projection
// 9.5 (8.5), FFN2 26.3 (24.7); 12 layers there 1362 -> 1331 us, at 16 x 1024 2495 -> 2479.  Where one workgroup
// fills a CU and there would be a third of a round too many, a launch therefore has workgroups for the
// expected rows, in whole rounds, and one whose position is followed by further ones (the rows were more) goes on to them.  `tile` returns the number of
// positions (0: none here).  Everywhere else a kernel without the loop is 0.2 us faster.
// Nothing of a tile stays in registers for the next.
template <typename Tile>
__device__ __forceinline__ void for_each_tile(const GemmArgs &p, Tile tile) {
  for (int bid = (int)blockIdx.x;;) {
    const int end = tile(bid);
    bid += p.tile_grid;
    if (bid >= end) return;
    __syncthreads();   // every wave is done with the LDS of this tile
  }
}

template <int BM, int BN, int STAGES, int WM, int WN, int NP, int EPI, bool WKN, int MASK>
__global__ __launch_bounds__((WM * WN + NP) * 64) void gemm_flat_kernel(BT_GEMM_FIRST, GemmTail<MASK> tail) {
#if defined(__HIP_DEVICE_COMPILE__)
  gemm_tiles_flat<BM, BN, STAGES, WM, WN, NP, EPI, WKN, MASK>(gemm_args<MASK, BN>(BT_GEMM_FIRST_NAMES, tail));
#endif
}

template <int BM, int BN, int STAGES, int WM, int WN, int NP, int EPI, bool WKN, int MASK, bool LOOP>
__global__ __launch_bounds__((WM * WN + NP) * 64) void gemm_kernel(BT_GEMM_FIRST, GemmTail<MASK> tail) {
#if defined(__HIP_DEVICE_COMPILE__)
  const GemmArgs p = gemm_args<MASK, BN>(BT_GEMM_FIRST_NAMES, tail);
  if constexpr (LOOP)
    for_each_tile(p, [&](int bid) { return gemm_tile<BM, BN, STAGES, WM, WN, NP, EPI, WKN, MASK, LOOP>(p, bid); });
  else
    gemm_tile<BM, BN, STAGES, WM, WN, NP, EPI, WKN, MASK, LOOP>(p, (int)blockIdx.x);
#endif
}
// Without a mask to count and tiles to go on to there is no tail.
template <int BM, int BN, int STAGES, int WM, int WN, int NP, int EPI, bool WKN>
__global__ __launch_bounds__((WM * WN + NP) * 64) void gemm_short_kernel(BT_GEMM_FIRST) {
#if defined(__HIP_DEVICE_COMPILE__)
  gemm_tile<BM, BN, STAGES, WM, WN, NP, EPI, WKN, kMaskNone, false>(gemm_args<kMaskNone, BN>(BT_GEMM_FIRST_NAMES, {}),
                                                                    (int)blockIdx.x);
#endif
}

// ---- one of two tiles ------------------------------------------------------------------
// Products whose live rows only the device knows.  A tile is as good as the rounds of the chip that it takes, so the
// one that suits up to 120 % of an expected row count takes 5 to 12 % longer than the best where fewer rows come, and
// at the far side of a round's end the other way about.  Where two tiles of one workgroup size are each the better one
// for some of the likely rows, the launch has both, and takes the one whose rounds cost less.
// ratio: 256 x the second one's cost of a round over the first one's.
// 12 layers without a row count, one tile and one of two, us (the rows of one draw of lengths): encoder 12 x 380 874 -> 835,
// with a bias 895 -> 855, 16 x 1024 2687 -> 2597, 20 x 200 845 -> 822, 6 x 250 515 -> 493, per-layer entry 12 x 380 981 -> 938,
// 16 x 512 1644 -> 1592; other lengths gain less, none at those of 100 x 120, and FFN2's slices at six heads of 128, 8 x 300,
// 821 -> 825; where the rows are known nothing
// changes, and a launch of two is asked to be 2.5 % better on the average of the likely rows (kPairMargin).  Of the
// pairs whose workgroups go together these five have nearly all there is to gain.  Which is taken changes no bit.
template <int BM_, int BN_, int STAGES_, int WM_, int WN_, int NP_>
struct TileShape {
  static constexpr int BM = BM_, BN = BN_, STAGES = STAGES_, WM = WM_, WN = WN_, NP = NP_;
  static constexpr int kThreads = (WM * WN + NP) * 64;
  static constexpr size_t kLds = (size_t)STAGES * (BM + BN) * kBK * sizeof(half_t);
};
constexpr int kEitherCus = 256;   // (of a chip with more or fewer the launcher makes no use of this)
__host__ __device__ __forceinline__ int rounds_of(int rows, int bm, int tiles_n, int splits) {
  return ((rows + bm - 1) / bm * tiles_n * splits + kEitherCus - 1) / kEitherCus;
}
__host__ __device__ __forceinline__ bool second_is_faster(int first_rounds, int second_rounds, unsigned ratio) {
  return (unsigned)second_rounds * ratio < (unsigned)first_rounds * 256u;
}
template <typename A, typename B, int EPI, bool WKN>
__global__ __launch_bounds__(A::kThreads > B::kThreads ? A::kThreads : B::kThreads) void gemm_either_kernel(BT_GEMM_FIRST, GemmTail<kMaskNone> tail) {
#if defined(__HIP_DEVICE_COMPILE__)
  GemmArgs p = gemm_args<kMaskNone, A::BN>(BT_GEMM_FIRST_NAMES, tail);
  const int M = min(*p.valid_rows, p.rows_cap), second_n = (p.N + B::BN - 1) / B::BN;
  constexpr bool LOOP = EPI != kEpiPartial;
  const auto run = [&](auto shape) {
    using T = decltype(shape);
    if (threadIdx.x >= T::kThreads) return;   // (whole waves; a barrier counts those that are left)
    const auto tile = [&](int bid) {
      return gemm_tile<T::BM, T::BN, T::STAGES, T::WM, T::WN, T::NP, EPI, WKN, kMaskNone, LOOP>(p, bid);
    };
    if constexpr (LOOP)
      for_each_tile(p, tile);
    else
      tile((int)blockIdx.x);
  };
  if (second_is_faster(rounds_of(M, A::BM, p.tiles_n, p.splits), rounds_of(M, B::BM, second_n, p.splits), tail.ratio)) {
    p.tiles_n = second_n, p.per_n = tail.per_n_second;
    run(B{});
  } else {
    run(A{});
  }
#endif
}

// ---- a few rows: the waves share the k range, not the tile ----------------------------
// One 32x32 tile per workgroup.  Its waves take the k-steps in turn (wave w: steps w, w + NW, ...),
// each through a ring of its own that it fills and reads alone, so the loop has no barrier; their
// sums are folded through LDS at the end, in wave order.  What bounds such a launch is the chain of
// k-steps of one tile (barrier, LDS read, MFMAs: 0.18 us each in the 32x64 tile); here a wave has a
// quarter of them, and with K = 768 all of its loads are in flight at once.  Projection of 230 rows at
// hidden 768: 5.0 -> 4.4 us; 12 layers at batch 1 x 32 407 -> 397 us, 1 x 256 482 -> 476, captured
// encoder at 4 x 96 469 -> 458.  Tried and slower: 32x64 tiles (half as many workgroups: 1 x 32 394 us
// against 372 on one box), six or eight waves (a captured 4 x 96: 416 against 413), and a ring of 6 to 10
// steps under the 32x64 tile (no gain to -8 %).
#if defined(__HIP_DEVICE_COMPILE__)
// The weight operand of 16 k out of a [K, N] image (load_kn_frag, as assembly: in front of the compiler's
// own transpose read it waits for every direct-to-LDS load of this wave, that is, for the k-steps
// requested ahead), and the wait for it while LEFT younger LDS operations may be outstanding.
template <int KSTEP>
__device__ __forceinline__ void kn_read_step(uint2_t (&w)[2], unsigned at) {
  constexpr int kRow = kWaveKCols * (int)sizeof(half_t);
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(w[0]) : "v"(at), "n"(KSTEP * 16 * kRow));
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(w[1]) : "v"(at), "n"((KSTEP * 16 + 4) * kRow));
}
template <int LEFT>
__device__ __forceinline__ half8_t lds_wait_operand(uint2_t (&w)[2]) {
  asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(w[0]), "+v"(w[1]) : "n"(LEFT));
  return __builtin_bit_cast(half8_t, uint4_t{w[0][0], w[0][1], w[1][0], w[1][1]});
}

template <int EPI, bool WKN, int MASK>
__device__ __forceinline__ void gemm_wave_k(const GemmArgs &p) {
  constexpr int BM = 32, BN = kWaveKCols, BK = kBK, NW = kWaveKWaves, DEPTH = kWaveKDepth;
  constexpr int KS = BK / 16;
  constexpr int NIA = BM / 8, NI = (BM + BN) / 8;   // 1 KB load instructions per k-step
  constexpr int STEP_HALFS = (BM + BN) * BK;
  static_assert(BN == 32 && KS == 4, "one MFMA block; the loop body names its four k parts");
  static_assert(NW == 4, "a wave for each of the four quads of sums");
  static_assert((DEPTH - 1) * NI < 64, "pipeline depth");
  static_assert(BM * BN * sizeof(float) <= DEPTH * STEP_HALFS * sizeof(half_t), "sums fit the ring");
  extern __shared__ __attribute__((aligned(1024))) half_t gemm_smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int bid = (int)blockIdx.x;
  half_t *ring = gemm_smem + wave * DEPTH * STEP_HALFS;
  int M;
  MaskRows mr{};
  if constexpr (MASK != kMaskNone) {
    mr = mask_rows_setup<MASK>(p, wave, NW, lane, (int *)(gemm_smem + NW * DEPTH * STEP_HALFS));
    M = min(mr.M, p.rows_cap);
    if (bid == 0) mask_rows_write(p, mr, tid, NW * 64, lane);
  } else {
    M = p.valid_rows ? min(*p.valid_rows, p.rows_cap) : p.rows_cap;
  }
  int split, tile_m, tile_n;
  if (!tile_at<BM, BN>(p, M, bid, split, tile_m, tile_n)) return;
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const int nk = EPI == kEpiPartial ? divide_small(p.K / BK, p.splits) : p.K / BK;
  const int k_first = EPI == kEpiPartial ? split * nk * BK : 0;
  const int mine = (nk - wave + NW - 1) / NW;   // (0 where there are fewer steps than waves)

  const bool gather = MASK != kMaskNone || p.a_row_index != nullptr;
  const rsrc_t rs_a =
      gather ? make_rsrc(p.a + k_first, ((size_t)p.rows_cap * p.K - k_first) * sizeof(half_t))
             : make_rsrc(p.a + (size_t)m0 * p.K + k_first,
                         ((size_t)(M - m0) * p.K - k_first) * sizeof(half_t));
  const rsrc_t rs_w =
      WKN ? make_rsrc(p.wt + (size_t)k_first * p.N + n0,
                      ((size_t)(p.K - k_first) * p.N - n0) * sizeof(half_t))
          : make_rsrc(p.wt + (size_t)n0 * p.K + k_first,
                      ((size_t)(p.N - n0) * p.K - k_first) * sizeof(half_t));
  int voff[NI];
  {
    MaskRowSpan span{};
    if constexpr (MASK != kMaskNone) span = mask_rows_span(mr, p.mask_B, lane, m0, min(m0 + BM, M) - 1);
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int r = i * 8 + (lane >> 3);
      const int kc = (lane & 7) ^ swz(r);
      int row = i < NIA ? r : r - BM;
      if (i < NIA && gather) {
        const int live_row = min(m0 + r, M - 1);
        row = MASK != kMaskNone ? mask_rows_map(mr, span, live_row) : p.a_row_index[live_row];
      }
      voff[i] = (row * p.K + kc * 8) * (int)sizeof(half_t);
      if (WKN && i >= NIA) voff[i] = kn_load_offset<BN>(i - NIA, lane, p.N, p.N - n0);
    }
  }
  const int w_step_bytes = (WKN ? BK * p.N : BK) * (int)sizeof(half_t);
  constexpr bool kHasBias = EPI == kEpiBiasGelu || EPI == kEpiQkvSplit || EPI == kEpiBias;
  const int n = n0 + wave * 8 + (lane >> 5) * 4;   // of the sums that this lane stores
  half4_t bias = {0, 0, 0, 0};
  if (kHasBias) bias = *(const half4_t *)(p.bias + min(n, p.N - 4));   // (ahead of the operands: it has long arrived)
  auto issue = [&](int i, int slot) {
    const int kt = wave + i * NW;
    issue_stage_loads<NI, NIA>(rs_a, rs_w, voff, ring + slot * STEP_HALFS, 8 * BK,
                               kt * BK * (int)sizeof(half_t), kt * w_step_bytes);
  };
#pragma unroll
  for (int s = 0; s < DEPTH; ++s)
    if (s < mine) issue(s, s);

  float16_t acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.f;
  const int fr_row = lane & 31, fr_kc = lane >> 5;
  unsigned kn_at;   // byte offset of this lane's first transpose read, from the weight image
  {
    const int lq = lane & 15, g2 = lane >> 4;
    const int k_row = 8 * (g2 >> 1) + (lq >> 2), col = 16 * (g2 & 1) + 4 * (lq & 3);
    kn_at = (k_row * BN + col) * (int)sizeof(half_t);
  }
  int slot = 0;
  for (int s = 0; s < mine; ++s) {
    wait_stages<NI, DEPTH - 1>(mine - 1 - s);
    asm volatile("" ::: "memory");
    const half_t *sA = ring + slot * STEP_HALFS, *sB = sA + BM * BK;
    half8_t fa[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      fa[ks] = *(const half8_t *)(sA + fr_row * BK + (((2 * ks + fr_kc) ^ swz(fr_row)) * 8));
    if constexpr (WKN) {
      const unsigned at =
          (unsigned)(unsigned long long)(__attribute__((address_space(3))) const half_t *)sB + kn_at;
      uint2_t w[KS][2];
      kn_read_step<0>(w[0], at);
      kn_read_step<1>(w[1], at);
      kn_read_step<2>(w[2], at);
      kn_read_step<3>(w[3], at);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(lds_wait_operand<6>(w[0]), fa[0], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(lds_wait_operand<4>(w[1]), fa[1], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(lds_wait_operand<2>(w[2]), fa[2], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(lds_wait_operand<0>(w[3]), fa[3], acc, 0, 0, 0);
    } else {
      half8_t fw[KS];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        fw[ks] = *(const half8_t *)(sB + fr_row * BK + (((2 * ks + fr_kc) ^ swz(fr_row + BM)) * 8));
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(fw[ks], fa[ks], acc, 0, 0, 0);
    }
    if (s + DEPTH < mine) {
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the slot has been read
      issue(s + DEPTH, slot);
    }
    if (++slot == DEPTH) slot = 0;
  }

  // fold: quad q of a wave's sums (columns 8 q + 4 (lane >> 5) .. + 3 of row lane & 31) lies at 1 KB q
  // of its ring, 16 bytes per lane; wave q adds quad q over the waves and stores it
  {
    float4_t *own = (float4_t *)ring;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      own[q * 64 + lane] = float4_t{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
  }
  __syncthreads();
  float4_t v = ((const float4_t *)gemm_smem)[wave * 64 + lane];
#pragma unroll
  for (int w = 1; w < NW; ++w)
    v += ((const float4_t *)(gemm_smem + w * DEPTH * STEP_HALFS))[wave * 64 + lane];
  const int m = m0 + fr_row;
  if (m >= M || n >= p.N) return;
  if (EPI == kEpiPartial) {
    store_through(p.c32 + ((size_t)split * p.rows_cap + m) * p.N + n, __builtin_bit_cast(uint4_t, v));
    return;
  }
  if (kHasBias) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] += (float)bias[e];
  }
  if (EPI == kEpiBiasGelu) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = gelu_tanh_f32(v[e]);
  }
  half_t *dst = EPI == kEpiQkvSplit ? p.c + ((size_t)(n >> 6) * p.rows_cap + m) * 64 + (n & 63)
                                    : p.c + (size_t)m * p.N + n;
  store_through(dst, __builtin_bit_cast(uint2_t, half4_t{(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]}));
}
#endif  // __HIP_DEVICE_COMPILE__

template <int EPI, bool WKN, int MASK>
__global__ __launch_bounds__(kWaveKWaves * 64) void gemm_wave_k_kernel(BT_GEMM_FIRST, GemmTail<MASK> tail) {
#if defined(__HIP_DEVICE_COMPILE__)
  gemm_wave_k<EPI, WKN, MASK>(gemm_args<MASK, kWaveKCols>(BT_GEMM_FIRST_NAMES, tail));
#endif
}
template <int EPI, bool WKN>
__global__ __launch_bounds__(kWaveKWaves * 64) void gemm_wave_k_short_kernel(BT_GEMM_FIRST) {
#if defined(__HIP_DEVICE_COMPILE__)
  gemm_wave_k<EPI, WKN, kMaskNone>(gemm_args<kMaskNone, kWaveKCols>(BT_GEMM_FIRST_NAMES, {}));
#endif
}

// Plain products whose live rows only the device knows: tile 14 where they fit one round of it, else tile 4
// (see takes_wave_k).  The top bits of k_splits bring the most tile rows of tile 14.
template <bool WKN>
__global__ __launch_bounds__(kWaveKWaves * 64) void gemm_few_rows_kernel(BT_GEMM_FIRST) {
#if defined(__HIP_DEVICE_COMPILE__)
  GemmArgs p = gemm_args<kMaskNone, kWaveKCols>(BT_GEMM_FIRST_NAMES, {});
  const int most_rows = p.splits * 32;
  p.splits = 1;
  if (*p.valid_rows <= most_rows) {
    gemm_wave_k<kEpiPlain, WKN, kMaskNone>(p);
  } else {
    p.tiles_n = (p.N + 63) / 64;
    p.per_n = 0xffffffffu / (unsigned)p.tiles_n;
    gemm_tile<32, 64, 4, 1, 2, 2, kEpiPlain, WKN, kMaskNone, false>(p, (int)blockIdx.x);
  }
#endif
}

// ---- weight pre-pack: wt[n][k] = w[k][n] for up to four matrices in one launch ---
struct TransposeJob {
  const half_t *w;
  half_t *wt;
  int K, N;
  int tiles_n, tile_begin;   // 64x64 tiles: tiles along n, first global tile id
};
struct TransposeArgs {
  TransposeJob job[4];
  int njobs;
};

__global__ __launch_bounds__(256) void transpose_kernel(TransposeArgs a) {
  __shared__ half_t tile[64][kTransposePitch];
  int j = 0;
#pragma unroll
  for (int i = 1; i < 4; ++i)
    if (i < a.njobs && (int)blockIdx.x >= a.job[i].tile_begin) j = i;
  const TransposeJob jb = a.job[j];
  const int t = blockIdx.x - jb.tile_begin;
  transpose_tile_64(jb.w, jb.wt, jb.K, jb.N, (t / jb.tiles_n) * 64, (t % jb.tiles_n) * 64, tile,
                    threadIdx.x, true);
}

static long long estimated_rows(const GemmArgs &p);
// Workgroups of a launch whose kernel can go on to further tiles (see for_each_tile): for the expected rows, of
// which a fifth more may come where the number is a guess, in whole rounds of the chip; `all` at most.
static int launched_tiles(const GemmArgs &p, int bm, int all) {
  const bool guess = (p.valid_rows || p.mask) && p.rows_hint <= 0;
  const long long rows = guess ? (estimated_rows(p) * 6 + 4) / 5 : estimated_rows(p);
  const long long expected = (rows + bm - 1) / bm * p.tiles_n * p.splits, round = cu_count();
  const long long rounds = (expected + round - 1) / round * round;
  return rounds < all ? (int)rounds : all;
}

// Calls `launch` with the weight layout and the source of the rows as compile-time constants.
template <int EPI, typename Then>
static int by_layout(const GemmArgs &p, Then then) {
  auto with = [&](auto mask) { return p.w_kn ? then(std::true_type{}, mask) : then(std::false_type{}, mask); };
  if constexpr (EPI == kEpiQkvSplit || EPI == kEpiBias) {
    if (p.mask && p.mask_f32) return with(std::integral_constant<int, kMaskF32>{});
    if (p.mask) return with(std::integral_constant<int, kMaskF16>{});
  }
  return with(std::integral_constant<int, kMaskNone>{});
}

template <int BM, int BN, int STAGES, int WM, int WN, int NP, int EPI, bool WKN, int MASK, bool LOOP>
static int launch_gemm_kernel(const GemmArgs &p, hipStream_t s, size_t smem) {
  return with_first_arguments<MASK>(p, [&](auto... first) {
    if constexpr (MASK == kMaskNone && !LOOP)
      return Launch<gemm_short_kernel<BM, BN, STAGES, WM, WN, NP, EPI, WKN>>::on(
          s, "gemm_kernel", p.tile_grid, (WM * WN + NP) * 64, smem, first...);
    else
      return Launch<gemm_kernel<BM, BN, STAGES, WM, WN, NP, EPI, WKN, MASK, LOOP>>::on(
          s, "gemm_kernel", p.tile_grid, (WM * WN + NP) * 64, smem, first..., gemm_tail<MASK>(p));
  });
}

template <int BM, int BN, int STAGES, int WM, int WN, int NP, int EPI, bool WKN, int MASK>
static int launch_gemm_tile_as(GemmArgs p, hipStream_t s, int splits) {
  constexpr size_t smem = (size_t)STAGES * (BM + BN) * kBK * sizeof(half_t);
  static_assert(smem <= 160 * 1024, "LDS budget");
  const int tiles_m = (p.rows_cap + BM - 1) / BM;
  p.tiles_n = (p.N + BN - 1) / BN;
  p.splits = splits;
  p.tile_grid = (tiles_m * p.tiles_n * splits + 7) / 8 * 8;
  if constexpr (smem > 80 * 1024 && EPI != kEpiPartial) {
    const int launched = launched_tiles(p, BM, p.tile_grid) / 8 * 8;
    if (p.tile_grid - launched > cu_count() / 3) {   // (32 or 48 fewer: 7 x 217 -0.5 %, heads of 128 -0.6 %)
      p.tile_grid = launched;
      return launch_gemm_kernel<BM, BN, STAGES, WM, WN, NP, EPI, WKN, MASK, true>(p, s, smem);
    }
  }
  return launch_gemm_kernel<BM, BN, STAGES, WM, WN, NP, EPI, WKN, MASK, false>(p, s, smem);
}

template <int BM, int BN, int STAGES, int WM, int WN, int NP, int EPI>
static int launch_gemm_tile(GemmArgs p, hipStream_t s, int splits = 1) {
  return by_layout<EPI>(p, [&](auto wkn, auto mask) {
    return launch_gemm_tile_as<BM, BN, STAGES, WM, WN, NP, EPI, wkn(), mask()>(p, s, splits);
  });
}

template <typename A, typename B, int EPI>
static int launch_gemm_either(GemmArgs p, hipStream_t s, unsigned ratio, int splits = 1) {
  constexpr size_t smem = A::kLds > B::kLds ? A::kLds : B::kLds;
  constexpr int kThreads = A::kThreads > B::kThreads ? A::kThreads : B::kThreads;
  static_assert(smem <= 160 * 1024, "LDS budget");
  p.splits = splits, p.ratio = ratio;
  const auto grid = [&](int bm, int bn) {
    p.tiles_n = (p.N + bn - 1) / bn;
    const int all = ((p.rows_cap + bm - 1) / bm * p.tiles_n * splits + 7) / 8 * 8;
    return EPI == kEpiPartial ? all : launched_tiles(p, bm, all) / 8 * 8;
  };
  const int second = grid(B::BM, B::BN);
  p.per_n_second = inverse_of((unsigned)p.tiles_n);
  const int first = grid(A::BM, A::BN);
  p.tile_grid = first > second ? first : second;
  const auto launch = [&](auto wkn) {
    return with_first_arguments<kMaskNone>(p, [&](auto... arguments) {
      return Launch<gemm_either_kernel<A, B, EPI, wkn()>>::on(s, "gemm_either_kernel", p.tile_grid, kThreads, smem, arguments...,
                                                              gemm_tail<kMaskNone>(p));
    });
  };
  return p.w_kn ? launch(std::true_type{}) : launch(std::false_type{});
}
using Tile1 = TileShape<128, 128, 3, 2, 2, 4>;
using Tile2 = TileShape<256, 128, 3, 4, 2, 4>;
using Tile3 = TileShape<256, 192, 2, 4, 2, 4>;
using Tile9 = TileShape<64, 64, 4, 2, 2, 4>;
using Tile10 = TileShape<64, 128, 3, 2, 2, 4>;
using Tile11 = TileShape<96, 128, 3, 3, 2, 4>;
using Tile12 = TileShape<128, 192, 3, 2, 2, 4>;

template <int EPI, bool WKN, int MASK>
static int launch_gemm_wave_k_as(GemmArgs p, hipStream_t s, int splits) {
  // (and 256 bytes for the lengths of a launch that counts the mask rows)
  constexpr size_t smem = (size_t)kWaveKWaves * kWaveKDepth * (32 + kWaveKCols) * kBK * sizeof(half_t) + 256;
  static_assert(smem <= 160 * 1024, "LDS budget");
  p.tiles_n = (p.N + kWaveKCols - 1) / kWaveKCols;
  p.splits = splits;
  p.tile_grid = ((p.rows_cap + 31) / 32 * p.tiles_n * splits + 7) / 8 * 8;
  return with_first_arguments<MASK>(p, [&](auto... first) {
    if constexpr (MASK == kMaskNone)
      return Launch<gemm_wave_k_short_kernel<EPI, WKN>>::on(s, "gemm_wave_k_kernel", p.tile_grid, kWaveKWaves * 64, smem, first...);
    else
      return Launch<gemm_wave_k_kernel<EPI, WKN, MASK>>::on(s, "gemm_wave_k_kernel", p.tile_grid, kWaveKWaves * 64, smem,
                                                            first..., gemm_tail<MASK>(p));
  });
}

template <int EPI>
static int launch_gemm_wave_k(GemmArgs p, hipStream_t s, int splits = 1) {
  return by_layout<EPI>(p, [&](auto wkn, auto mask) {
    return launch_gemm_wave_k_as<EPI, wkn(), mask()>(p, s, splits);
  });
}

template <bool WKN>
static int launch_gemm_few_rows_as(GemmArgs p, hipStream_t s) {
  constexpr size_t smem = (size_t)kWaveKWaves * kWaveKDepth * (32 + kWaveKCols) * kBK * sizeof(half_t);
  static_assert(smem >= 4 * (32 + 64) * kBK * sizeof(half_t), "room for the ring of tile 4");
  p.tiles_n = (p.N + kWaveKCols - 1) / kWaveKCols;
  // (one round of either tile: what the few rows take, or the capacity in the wider tiles)
  p.splits = cu_count() / p.tiles_n;   // tile rows of one round, at most 255 of them
  if (p.splits > 255) p.splits = 255;
  const int few = p.splits * p.tiles_n, wide = (p.rows_cap + 31) / 32 * ((p.N + 63) / 64);
  const int grid = ((few > wide ? few : wide) + 7) / 8 * 8;
  return with_first_arguments<kMaskNone>(p, [&](auto... first) {
    return Launch<gemm_few_rows_kernel<WKN>>::on(s, "gemm_few_rows_kernel", grid, kWaveKWaves * 64, smem, first...);
  });
}
static int launch_gemm_few_rows(const GemmArgs &p, hipStream_t s) {
  return p.w_kn ? launch_gemm_few_rows_as<true>(p, s) : launch_gemm_few_rows_as<false>(p, s);
}

// Persistent launch: about one workgroup per CU (a multiple of 8, one share per XCD), each
// looping over its tiles on the device.
template <int BM, int BN, int STAGES, int WM, int WN, int NP, int EPI, bool WKN, int MASK>
static int launch_gemm_flat_as(GemmArgs p, hipStream_t s) {
  constexpr size_t smem = (size_t)STAGES * (BM + BN) * kBK * sizeof(half_t) + STAGES * BN * sizeof(half_t);
  static_assert(smem <= 160 * 1024, "LDS budget");
  const int tiles_m = (p.rows_cap + BM - 1) / BM;
  p.tiles_n = (p.N + BN - 1) / BN;
  const long long tiles = (long long)tiles_m * p.tiles_n;
  const int per_cu = smem <= 80 * 1024 ? 2 : 1;          // workgroups that fit one CU's LDS
  long long wgs = (long long)cu_count() * per_cu;
  if (wgs > tiles) wgs = tiles;
  p.tile_grid = (int)((wgs + 7) / 8 * 8);
  p.splits = 1;
  return with_first_arguments<MASK>(p, [&](auto... first) {
    return Launch<gemm_flat_kernel<BM, BN, STAGES, WM, WN, NP, EPI, WKN, MASK>>::on(
        s, "gemm_flat_kernel", p.tile_grid, (WM * WN + NP) * 64, smem, first..., gemm_tail<MASK>(p));
  });
}

template <int BM, int BN, int STAGES, int WM, int WN, int NP, int EPI>
static int launch_gemm_flat(GemmArgs p, hipStream_t s) {
  return by_layout<EPI>(p, [&](auto wkn, auto mask) {
    return launch_gemm_flat_as<BM, BN, STAGES, WM, WN, NP, EPI, wkn(), mask()>(p, s);
  });
}

int cu_count() {
  static const int cus = [] {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        n <= 0)
      n = 256;
    return n;
  }();
  return cus;
}

// Live rows the tile choice is made for: the exact count when every row is live, the
// caller's hint when it has one, else 60 % of the capacity (the fill the padding-free
// path is built for).
static long long estimated_rows(const GemmArgs &p) {
  if (!p.valid_rows && !p.mask) return p.rows_cap;
  if (p.rows_hint > 0) return p.rows_hint < p.rows_cap ? p.rows_hint : p.rows_cap;
  return (p.rows_cap * 3LL + 4) / 5;
}

#include "gemm_tuned.inc"

// Measured times of every tile for this weight shape at the first table row of at least m
// rows, or nullptr when the shape is not in the table or m lies outside it (the analytic
// model then decides alone).  The rows are at most kTunedStep apart where most launches are, the
// height of the tallest tile (and closer below, where smaller tiles matter), so the row used has the same number
// of row tiles as m or one more: run time moves in steps with the number of rounds of workgroups, and
// interpolating between two row counts on either side of such a step would describe neither.
static const float *tuned_times(long long m, int n, int k, int epi, int kn, int full) {
  if (cu_count() != 256) return nullptr;     // the table was measured on a 256-CU part
  if (m > kTunedRows[kTunedPoints - 1]) return nullptr;
  // (the token-major QKV projection differs from the head-major one in where it stores)
  if (epi == kEpiBias) epi = kEpiQkvSplit;
  for (const TunedShape &ts : kTunedShapes) {
    if (ts.n != n || ts.k != k || ts.epi != epi || ts.kn != kn || ts.full != full) continue;
    int at = 0;
    while (at < kTunedPoints - 1 && kTunedRows[at] < m) ++at;
    return ts.us[at];
  }
  return nullptr;
}

// The row counts a tile is priced at.  A launch over padded sequences whose caller named no row
// count holds 60 % of its capacity give or take: the mean of a handful of sequence lengths is off
// by 10-20 %.  A tile priced at the middle alone may fit one round of the chip there and need two
// a few rows later (7 sequences of up to 844 tokens, narrow products: 17.4 us a launch with the tile
// this picks, 23.3 us with the one that was fastest at 60 %), so it is priced over the spread.
struct LikelyRows {
  long long rows[5];
  float weight[5];
  int count;
  explicit LikelyRows(const GemmArgs &p) {
    const long long m = estimated_rows(p);
    const bool guess = (p.valid_rows || p.mask) && p.rows_hint <= 0;
    count = guess ? 5 : 1;
    for (int i = 0; i < count; ++i) {
      rows[i] = guess ? (m * (8 + i) + 9) / 10 : m;
      weight[i] = !guess ? 1.f : i == 2 ? 1.f / 3.f : 1.f / 6.f;
    }
  }
};

struct TileModel {
  int id, bm, bn;
  float step_us, fixed_us;   // one k-step of one tile; launch, fill and epilogue of one tile
  float shared_us;           // > 0: one k-step's share of a CU that several tiles occupy
};

// Fitted to the table's measurements.  Both were taken of these tiles on 32x32x16 instructions, with stores that
// stayed in the L2 and a workgroup for every tile of the capacity; the kernels have become 4 to 13 % faster since, not all
// tiles alike, and how far the choice is from the fastest tile of today has not been measured.
static const TileModel kTileModels[] = {
    {0, 256, 256, 1.45f, 5.7f, 0.f},     {13, 192, 192, 0.95f, 4.7f, 0.f},  {3, 256, 192, 1.10f, 4.35f, 0.f},
    {12, 128, 192, 0.64f, 4.6f, 0.f},    {2, 256, 128, 0.79f, 4.4f, 0.f},   {1, 128, 128, 0.467f, 3.4f, 0.f},
    {5, 128, 128, 0.66f, 3.6f, 0.70f},   {11, 96, 128, 0.41f, 3.0f, 0.f},   {10, 64, 128, 0.267f, 2.67f, 0.43f},
    {9, 64, 64, 0.20f, 2.63f, 0.265f},   {4, 32, 64, 0.175f, 2.75f, 0.19f}};

// Workgroups that count the mask rows first (bt_gemm_qkv_bias_split_mask_rows) do so once per tile in
// every tile but the persistent ones: each round past the first pays for it.  Batch 16 x 1024, hidden
// 768: 256x192 in two rounds 40.8 us by the table, which counts no mask, and 51.5 in the layer;
// persistent 256x128 43.2 and 47.9.
constexpr float kMaskRoundUs = 3.f;
static float mask_rounds_us(int id, long long m, int n) {
  for (const TileModel &c : kTileModels) {
    if (c.id != id) continue;
    const long long tiles = ((m + c.bm - 1) / c.bm) * ((n + c.bn - 1) / c.bn);
    const long long at_once = (long long)cu_count() * (c.shared_us > 0.f ? 2 : 1);
    return tiles > at_once ? kMaskRoundUs * (float)((tiles - 1) / at_once) : 0.f;
  }
  return 0.f;   // a persistent form
}

// Time of one launch of n columns and k reduction: fixed + k-steps x step time, where a step takes
// `step_us` while every CU has one tile at most and then grows in whole rounds or, where several
// workgroups share a CU, with its load.
static float model_us(const TileModel &c, long long m, int n, int k) {
  const int cus = cu_count();
  const float nk = (float)(k / kBK);
  const long long tiles = ((m + c.bm - 1) / c.bm) * ((n + c.bn - 1) / c.bn);
  if (c.shared_us > 0.f) {
    const float load = (float)tiles / (float)cus * c.shared_us;
    return c.fixed_us + nk * (load > c.step_us ? load : c.step_us);
  }
  return (float)((tiles + cus - 1) / cus) * (nk * c.step_us + c.fixed_us - 1.8f) + 1.8f;
}

static int fastest_by_model(const LikelyRows &likely, int n, int k, bool mask) {
  int best_id = 0;
  float best = 0.f;
  for (const TileModel &c : kTileModels) {
    float t = 0.f;
    for (int i = 0; i < likely.count; ++i)
      t += likely.weight[i] * (model_us(c, likely.rows[i], n, k) + (mask ? mask_rounds_us(c.id, likely.rows[i], n) : 0.f));
    if (best == 0.f || t < best) {
      best = t;
      best_id = c.id;
    }
  }
  return best_id;
}

// The table's times of every tile over the likely rows (0 = not measured at all of them); false
// when the table does not cover the launch.
static bool tuned_mean(const LikelyRows &likely, int n, int k, int epi, int kn, int full, float *us) {
  for (int i = 0; i < likely.count; ++i) {
    const float *at = tuned_times(likely.rows[i], n, k, epi, kn, full);
    if (!at) return false;
    for (int t = 0; t < kTunedTiles; ++t)
      us[t] = at[t] > 0.f && (i == 0 || us[t] > 0.f) ? (i == 0 ? 0.f : us[t]) + likely.weight[i] * at[t] : 0.f;
  }
  return true;
}

// The fastest tile for the likely rows: the model's, unless the table knows a clear win.
static int fastest_tile(const GemmArgs &p, int epi) {
  const LikelyRows likely(p);
  float us[kTunedTiles];
  int choice = fastest_by_model(likely, p.N, p.K, p.mask != nullptr);
  // the table overrides the model only for a clear win: the timings come from a loop
  // of identical launches, and differences of a few per cent do not carry over to the
  // layer sequence
  // (a launch whose estimated live rows fill its capacity to within one tile row is looked
  // up among the all-live measurements)
  if (tuned_mean(likely, p.N, p.K, epi, p.w_kn, estimated_rows(p) + kTunedStep > p.rows_cap, us)) {
    if (p.mask)
      for (int t = 0; t < kTunedTiles; ++t)
        for (int i = 0; us[t] > 0.f && i < likely.count; ++i)
          us[t] += likely.weight[i] * mask_rounds_us(t, likely.rows[i], p.N);
    int tuned = -1;
    for (int t = 0; t < kTunedTiles; ++t)
      if (us[t] > 0.f && (tuned < 0 || us[t] < us[tuned])) tuned = t;
    const float t_model = us[choice];
    const float margin = 1.f - 0.01f * (float)option_gemm_table_margin();
    if (tuned >= 0 && tuned != choice && (t_model <= 0.f || us[tuned] < margin * t_model))
      choice = tuned;
  }
  return choice;
}

// The pairs that a launch may have (gemm_either_kernel), and what is asked of one beyond the fastest tile's time.
struct TilePair {
  int first, first_bm, first_bn, second, second_bm, second_bn;
};
static const TilePair kTilePairs[] = {
    {9, 64, 64, 10, 64, 128}, {10, 64, 128, 1, 128, 128}, {10, 64, 128, 11, 96, 128},
    {1, 128, 128, 12, 128, 192}, {2, 256, 128, 3, 256, 192}};
constexpr float kPairMargin = 0.975f, kPairChoiceUs = 0.1f;

// The fastest pair for `count` likely rows, given the times of both tiles at each: its number from 1 on (0: none below
// `most_us`), and the ratio by which the device picks.
template <typename Us>
static int fastest_pair(const LikelyRows &likely, int n, int splits, int pairs, float most_us, unsigned &ratio, Us us) {
  int best = 0;
  for (int q = 0; q < pairs; ++q) {
    const TilePair &c = kTilePairs[q];
    float first[5], second[5], first_round = 0.f, second_round = 0.f;
    int first_rounds[5], second_rounds[5];
    for (int i = 0; i < likely.count; ++i) {
      first[i] = us(c.first, i), second[i] = us(c.second, i);
      first_rounds[i] = rounds_of((int)likely.rows[i], c.first_bm, (n + c.first_bn - 1) / c.first_bn, splits);
      second_rounds[i] = rounds_of((int)likely.rows[i], c.second_bm, (n + c.second_bn - 1) / c.second_bn, splits);
      first_round += likely.weight[i] * first[i] / (float)first_rounds[i];
      second_round += likely.weight[i] * second[i] / (float)second_rounds[i];
    }
    const unsigned r = (unsigned)(256.f * second_round / first_round + 0.5f);
    float t = kPairChoiceUs;
    for (int i = 0; i < likely.count; ++i)
      t += likely.weight[i] * (second_is_faster(first_rounds[i], second_rounds[i], r) ? second[i] : first[i]);
    if (t < most_us && r < (1u << 20)) best = q + 1, most_us = t, ratio = r;
  }
  return best;
}

// For a launch that knows no row count: its tile | its pair << 4 | the pair's ratio << 8.
static int tile_or_pair(const GemmArgs &p, int epi) {
  const LikelyRows likely(p);
  const int tile = fastest_tile(p, epi);
  const float *table[5];
  for (int i = 0; i < likely.count; ++i)
    table[i] = tuned_times(likely.rows[i], p.N, p.K, epi, p.w_kn, estimated_rows(p) + kTunedStep > p.rows_cap);
  const auto us = [&](int id, int i) {
    if (table[i] && table[i][id] > 0.f) return table[i][id];
    for (const TileModel &c : kTileModels)
      if (c.id == id) return model_us(c, likely.rows[i], p.N, p.K);
    return 0.f;
  };
  float one = 0.f;
  for (int i = 0; i < likely.count; ++i) one += likely.weight[i] * us(tile, i);
  unsigned ratio = 0;
  const int pair = fastest_pair(likely, p.N, 1, 5, kPairMargin * one, ratio, us);
  return tile | pair << 4 | (int)(ratio << 8);
}

// How a product runs on tile 14, whose waves share k and add up in an order of their own: a row count that a
// caller knows in one call and not in the next must not change a bit, so this follows from sizes, and from the
// live rows themselves.  A workgroup fills its CU's LDS, so its tiles have to fit one round: us of tile 14 / tile
// 4 in one round and in two, projection at hidden 768 4.4 / 4.8 (320 rows), 6.6 / 4.8 (352); hidden 1024 5.1 / 5.6
// (256), 7.2 / 5.6 (288); hidden 512 3.8 / 4.1 (512); QKV at hidden 768 4.3 / 4.6 (32 rows), 4.8 / 4.8 (96), 6.7 / 4.7
// (128); FFN1 4.9 / 5.1 (32), 5.1 / 5.2 (64), 8.2 / 5.3 (96).  A plain product of a padded batch whose capacity
// does not fit, but fits in tile 4, finds its rows on the device, where the kernel takes the one or the other (four
// sequences of 96, all full: 4.9 us a projection in place of 6.7 without a row count; with one, 12 layers 483
// and 486 us).  In the products with more columns, whose gain is small, the second tile's code costs more than
// that (with it in both, 4 x 32 406 -> 416 us).  With fewer than four k-steps a wave has nothing to do.
enum WaveK { kWaveKNo, kWaveKYes, kWaveKDevice };
static WaveK takes_wave_k(const GemmArgs &p, bool plain) {
  const long long tiles_m = (p.rows_cap + 31) / 32, tiles_n = (p.N + kWaveKCols - 1) / kWaveKCols;
  if (p.K < kWaveKWaves * kBK || tiles_n > cu_count()) return kWaveKNo;
  if (tiles_m * tiles_n <= cu_count()) return kWaveKYes;
  return plain && p.valid_rows && tiles_m * ((p.N + 63) / 64) <= cu_count() ? kWaveKDevice : kWaveKNo;
}

bool product_takes_wave_k(int rows_cap, int n, int k) {
  GemmArgs p{};
  p.rows_cap = rows_cap, p.N = n, p.K = k;
  return takes_wave_k(p, false) == kWaveKYes;
}

// What a question about sizes was answered before, on this thread: a forward asks the same few in every layer,
// and pricing them anew costs the host 0.3 to 0.9 us each, while issuing a launch takes 3 to 4.
template <int KEYS, typename Ask>
static int remembered(const int (&sizes)[KEYS], Ask ask) {
  struct Entry {
    int sizes[KEYS], answer;
    bool known;
  };
  thread_local Entry entries[32];   // (of this question alone: one table per `Ask`)
  unsigned at = 0;
  for (int v : sizes) at = (at ^ (unsigned)v) * 0x9e3779b1u;
  Entry &e = entries[at >> 27];
  if (!e.known || memcmp(e.sizes, sizes, sizeof(sizes)) != 0) {
    e.answer = ask();
    memcpy(e.sizes, sizes, sizeof(sizes));
    e.known = true;
  }
  return e.answer;
}

// ---- products in k slices ----------------------------------------------------------------
// FFN2 of up to two thousand rows is a few dozen tiles with a k loop four times as long as the other
// products': k slices give the idle CUs a share of it, and the LayerNorm that reads the result anyway adds
// the slices up.  The pair's time is, within 3 % (84 pairs of tile and slices, hidden 768 and 1024, 32
// to 2736 rows), that of the tile - fixed + k-steps of a slice x step - plus what the LayerNorm reads.
// Tile 14 is priced by what layers with it take (hidden 1024, 64 rows, two slices / four, us: 40.1 / 38.0, the
// 32x64 tile 42.0 / 38.5): launched alone, its weight warm, the number of slices seems to make no difference.
// Pairs of FFN2 and LayerNorm, k whole -> in slices, us: hidden 768, 230 rows 14.7 -> 10.3 (four slices of
// 64x64 tiles; two of 32x64 tiles 10.7), 768 rows 16.1 -> 12.8, 911 rows 16.2 -> 14.4, 1500 rows 20.2 -> 16.7,
// 2000 rows 21.1 -> 19.5; hidden 1024, 640 rows 17.8 -> 14.8, 1300 rows 25.0 -> 21.3.
struct SliceModel {
  int id, bm, bn;
  float fixed_us, step_us;   // launch and LayerNorm of few rows included
  int busy_cus;              // (a tile that fills its CU finds some CU busy at the last few per cent: 252
};                           // workgroups 21.6 us, 216 16.7; the short ones of tile 14 fill the chip, 256)
static const SliceModel kSliceModels[] = {
    {14, 32, kWaveKCols, 8.00f, 0.080f, 0}, {4, 32, 64, 8.37f, 0.115f, 0},
    {9, 64, 64, 9.04f, 0.111f, 0},          {10, 64, 128, 9.37f, 0.195f, 0},
    {11, 96, 128, 10.39f, 0.242f, 16},      {1, 128, 128, 10.53f, 0.231f, 16},
    {12, 128, 192, 12.05f, 0.321f, 16}};
constexpr int kMostSlices = 4;
// Beyond this many results the slices cost the memory system more than the idle CUs give.  Layers of rows
// that are all live, 600 MB of weights walked through, k whole / in two slices, us: hidden 512 (k 2048)
// 1024 rows 43.5 / 43.0, 1088 rows 46.6 / 47.2, 1984 rows 49.1 / 50.9; hidden 576 1024 rows 45.9 / 46.7, 1600
// rows 56.9 / 58.4; hidden 640 (k 2560) 1984 rows 63.1 / 62.4; hidden 768 2112 rows 74.2 / 72.5, 2400 rows
// 76.7 / 75.5, 2600 rows 94.1 / 94.2; hidden 1024 1600 rows 90.7 / 87.2, 1984 rows 90.2 / 91.2, 2600
// rows 118.9 / 128.6.
static float sliced_results(int k) { return k < 2560 ? 0.55e6f : 1.9e6f; }
// What a tile's launch takes beyond the LayerNorm and the launches themselves, so again in a second round.
constexpr float kPairUs = 6.f;

static float slice_pair_us(const SliceModel &c, long long m, int n, int k, int splits) {
  const long long tiles = ((m + c.bm - 1) / c.bm) * ((n + c.bn - 1) / c.bn) * splits;
  const long long at_once = cu_count() - c.busy_cus;
  const float rounds = (float)((tiles + at_once - 1) / at_once);
  const float mn = (float)m * (float)n * 1e-6f, extra = (float)(splits - 1);
  return kPairUs + rounds * (c.fixed_us - kPairUs + c.step_us * (float)(k / kBK) / (float)splits) + 2.16f * mn +
         0.49f * mn * extra - (splits > 1 ? 0.86f + 0.12f * (extra - 1.f) : 0.f);
}

// The fastest tile for a number of slices, and the pair's time with it.
static const SliceModel &fastest_sliced(const LikelyRows &likely, int n, int k, int splits, float *us) {
  const SliceModel *best = nullptr;
  for (const SliceModel &c : kSliceModels) {
    if (splits == 1 && c.id == 14) continue;   // (measured in slices only)
    float t = 0.f;
    for (int i = 0; i < likely.count; ++i) t += likely.weight[i] * slice_pair_us(c, likely.rows[i], n, k, splits);
    if (!best || t < *us) best = &c, *us = t;
  }
  return *best;
}

template <int EPI>
static int launch_gemm(GemmArgs p, hipStream_t s) {
  // Tile table (rows x cols, ring depth, computing wave grid, loader waves):
  //   0: 256x256, 2, 2x4, 0   wide outputs: one tile per CU, every wave loads and computes
  //   1: 128x128, 3, 2x2, 4   narrow outputs (projection, FFN2) and small problems
  //   2: 256x128, 3, 4x2, 4   narrow outputs with enough rows to fill the chip
  //   3: 256x192, 2, 4x2, 4   outputs that split into 192-wide panels but not into a
  //                           full wave of 256-wide ones (QKV at hidden 768); 141 registers
  //                           leave room for the loader waves (-2 to -4 % against unified)
  //   4:  32x64,  4, 1x2, 2   a few hundred rows or fewer: the k loop of one tile is the
  //                           whole run time, and a small tile has the shortest k-step
  //   5: 128x128, 2, 2x2, 4   tile 1 with a two-deep ring: 64 KB of LDS, so two workgroups
  //                           share a CU and one's fill and epilogue hide under the other's
  //                           k loop; pays when tile 1 would need several rounds
  //   6, 7, 8                 tiles 2, 1 and 0 in the persistent form (gemm_tiles_flat); never
  //                           the model's choice, only the measured table's, and there
  //                           within a few per cent of the one-tile-per-workgroup form
  //   9:  64x64,  4, 2x2, 4   } one round of tiles on 256 CUs between the shapes above: a launch is
  //  10:  64x128, 3, 2x2, 4   } as long as its largest tile while it fits one round, so the tile
  //  11:  96x128, 3, 3x2, 4   } that just fills the chip wins.  Hidden 768, weights in the
  //  12: 128x192, 3, 2x2, 4   } memory-side cache, best of tiles 0-8 and now: FFN2 at 920 rows 17.0 ->
  //  13: 192x192, 2, 3x2, 4   } 13.0 us (9), at 2000 rows 20.6 -> 17.5 (10), at 5600 rows 35.6 -> 30.2
  //                           (12); QKV at 3600 rows 19.6 -> 18.6 (13), at 1300 rows 9.6 -> 9.1 (11)
  //  14:  32x32, four waves over k (gemm_wave_k), where takes_wave_k() says so
  // The choice minimises the time of the launch: for the weight shapes of BERT-base and BERT-large
  // by a table of measured times (gemm_tuned.inc) where it names a clearly faster tile, else by the
  // model of model_us().
  int choice = option_gemm_tile();
  if (choice < 0) {
    const WaveK few = takes_wave_k(p, EPI == kEpiPlain);
    if (few == kWaveKDevice) return launch_gemm_few_rows(p, s);
    if (few == kWaveKYes) choice = 14;
  }
  if (choice < 0 && p.valid_rows && !p.mask && p.rows_hint <= 0 && cu_count() == kEitherCus) {
    const int answer = remembered({p.rows_cap, p.N, p.K, p.w_kn, option_gemm_table_margin()}, [&] { return tile_or_pair(p, EPI); });
    const unsigned ratio = (unsigned)answer >> 8;
    choice = answer & 15;
    switch (answer >> 4 & 15) {
      case 1: return launch_gemm_either<Tile9, Tile10, EPI>(p, s, ratio);
      case 2: return launch_gemm_either<Tile10, Tile1, EPI>(p, s, ratio);
      case 3: return launch_gemm_either<Tile10, Tile11, EPI>(p, s, ratio);
      case 4: return launch_gemm_either<Tile1, Tile12, EPI>(p, s, ratio);
      case 5: return launch_gemm_either<Tile2, Tile3, EPI>(p, s, ratio);
      default: break;
    }
  }
  if (choice < 0) choice = fastest_tile(p, EPI);
  switch (choice) {
    case 14:
      return launch_gemm_wave_k<EPI>(p, s);
    case 0:
      return launch_gemm_tile<256, 256, 2, 2, 4, 0, EPI>(p, s);
    case 2:
      return launch_gemm_tile<256, 128, 3, 4, 2, 4, EPI>(p, s);
    case 3:
      return launch_gemm_tile<256, 192, 2, 4, 2, 4, EPI>(p, s);
    case 4:
      return launch_gemm_tile<32, 64, 4, 1, 2, 2, EPI>(p, s);
    case 5:
      return launch_gemm_tile<128, 128, 2, 2, 2, 4, EPI>(p, s);
    case 6:
      return launch_gemm_flat<256, 128, 3, 4, 2, 4, EPI>(p, s);
    case 7:
      return launch_gemm_flat<128, 128, 3, 2, 2, 4, EPI>(p, s);
    case 8:
      return launch_gemm_flat<256, 256, 2, 2, 4, 0, EPI>(p, s);
    case 9:
      return launch_gemm_tile<64, 64, 4, 2, 2, 4, EPI>(p, s);
    case 10:
      return launch_gemm_tile<64, 128, 3, 2, 2, 4, EPI>(p, s);
    case 11:
      return launch_gemm_tile<96, 128, 3, 3, 2, 4, EPI>(p, s);
    case 12:
      return launch_gemm_tile<128, 192, 3, 2, 2, 4, EPI>(p, s);
    case 13:
      return launch_gemm_tile<192, 192, 2, 3, 2, 4, EPI>(p, s);
    default:
      return launch_gemm_tile<128, 128, 3, 2, 2, 4, EPI>(p, s);
  }
}

static int check_gemm_args(const char *who, const void *a, const void *wt, const void *c,
                           int rows_cap, int n, int k, int weight_kn) {
  BT_REQUIRE(a && wt && c, BT_ERR_INVALID_ARGUMENT, "%s: null pointer argument", who);
  BT_REQUIRE(aligned16({a, wt, c}), BT_ERR_INVALID_ARGUMENT,
             "%s: tensor pointers must be 16-byte aligned", who);
  BT_REQUIRE(rows_cap >= 0 && n > 0 && k > 0, BT_ERR_INVALID_ARGUMENT,
             "%s: rows_cap=%d n=%d k=%d out of range", who, rows_cap, n, k);
  BT_REQUIRE(k % 64 == 0, BT_ERR_UNSUPPORTED, "%s: k=%d must be a multiple of 64", who, k);
  BT_REQUIRE(n % 8 == 0, BT_ERR_UNSUPPORTED, "%s: n=%d must be a multiple of 8", who, n);
  // a 256-row tile is addressed with 32-bit byte offsets from its first row
  BT_REQUIRE(k <= (1 << 21), BT_ERR_UNSUPPORTED, "%s: k=%d is beyond 2^21", who, k);
  BT_REQUIRE(weight_kn == 0 || weight_kn == 1, BT_ERR_INVALID_ARGUMENT,
             "%s: weight_kn=%d must be 0 ([n, k] pre-pack) or 1 ([k, n] as stored)", who, weight_kn);
  // a [k, n] weight is addressed with 32-bit byte offsets from its first row
  BT_REQUIRE(!weight_kn || (long long)n * k * 2 <= 0x7fffffffLL, BT_ERR_UNSUPPORTED,
             "%s: a [k, n] weight of %d x %d halfs is beyond 2 GiB", who, k, n);
  return BT_OK;
}

}  // namespace bt

using namespace bt;

extern "C" int bt_transpose_weights(int count, const void *const *w, void *const *wt,
                                    const int *k, const int *n, void *stream) {
  BT_REQUIRE(count >= 1 && count <= 4, BT_ERR_INVALID_ARGUMENT,
             "bt_transpose_weights: count=%d outside [1, 4]", count);
  BT_REQUIRE(w && wt && k && n, BT_ERR_INVALID_ARGUMENT,
             "bt_transpose_weights: null pointer argument");
  TransposeArgs a;
  a.njobs = count;
  int tiles = 0;
  for (int i = 0; i < count; ++i) {
    BT_REQUIRE(w[i] && wt[i], BT_ERR_INVALID_ARGUMENT,
               "bt_transpose_weights: null matrix pointer #%d", i);
    BT_REQUIRE(k[i] > 0 && n[i] > 0 && k[i] % 8 == 0 && n[i] % 8 == 0, BT_ERR_UNSUPPORTED,
               "bt_transpose_weights: k=%d n=%d must be positive multiples of 8", k[i], n[i]);
    a.job[i] = TransposeJob{(const half_t *)w[i], (half_t *)wt[i], k[i], n[i],
                            (n[i] + 63) / 64, tiles};
    tiles += ((n[i] + 63) / 64) * ((k[i] + 63) / 64);
  }
  for (int i = count; i < 4; ++i) a.job[i] = a.job[0];
  return Launch<transpose_kernel>::on(as_stream(stream), "transpose_kernel", tiles, 256, 0, a);
}

extern "C" int bt_transpose_weight(const void *w, void *wt, int k, int n, void *stream) {
  const void *ws[1] = {w};
  void *wts[1] = {wt};
  return bt_transpose_weights(1, ws, wts, &k, &n, stream);
}

extern "C" float bt_gemm_prepack_gain_us(long long rows, int n, int k, int epilogue) {
  const int forced = option_layer_prepack();
  if (forced >= 0) return forced ? 1e9f : -1e9f;
  // (asked for the padded batch: the layer's launches are sized for batch x seq_len rows)
  const float *nk = tuned_times(rows, n, k, epilogue, 0, 0), *kn = tuned_times(rows, n, k, epilogue, 1, 0);
  if (!nk || !kn) return 0.f;
  float best_nk = 0.f, best_kn = 0.f;
  for (int t = 0; t < kTunedTiles; ++t) {
    if (nk[t] > 0.f && (best_nk == 0.f || nk[t] < best_nk)) best_nk = nk[t];
    if (kn[t] > 0.f && (best_kn == 0.f || kn[t] < best_kn)) best_kn = kn[t];
  }
  if (best_nk == 0.f || best_kn == 0.f) return 0.f;
  // the copy is made inside the layer's first launch, beside the offsets: measured in the
  // layer sequence it adds about 0.5 us per megabyte of weight to that launch (2.4 us for
  // FFN1 of BERT-base, 7.4 us for all four matrices)
  const float pack_us = 0.5e-6f * (float)n * (float)k * sizeof(half_t);
  return best_kn - best_nk - pack_us;
}

extern "C" int bt_gemm_prepack_pays(long long rows, int n, int k, int epilogue) {
  return bt_gemm_prepack_gain_us(rows, n, k, epilogue) > 1.0f ? 1 : 0;   // asked to return a microsecond more
}

extern "C" int bt_gemm(const void *a, const void *wt, void *c, const int *valid_rows,
                       int rows_cap, int rows_hint, int n, int k, int weight_kn, void *stream) {
  int rc = check_gemm_args("bt_gemm", a, wt, c, rows_cap, n, k, weight_kn);
  if (rc) return rc;
  if (rows_cap == 0) return BT_OK;
  GemmArgs p{(const half_t *)a, (const half_t *)wt, nullptr, (half_t *)c, valid_rows, nullptr,
             rows_cap,          n,                  k,       0,           rows_hint,
             nullptr,           weight_kn};
  return launch_gemm<kEpiPlain>(p, as_stream(stream));
}

// The number of slices changes the order of the sums, so it follows from the sizes of the call alone, not from
// a row count that a caller may know in one call and not in the next: a padded batch is taken to be 60 %
// full or, less likely, full.
static int fastest_slices(int rows_cap, bool all_live, int n, int k, int most) {
  GemmArgs p{};
  p.rows_cap = rows_cap;
  const LikelyRows full(p);
  p.rows_cap = (int)((rows_cap * 3LL + 4) / 5);
  const LikelyRows part(p);
  const float fills = all_live ? 1.f : 1.f / 3.f;
  if ((float)(all_live ? full : part).rows[0] * (float)n > sliced_results(k)) return 1;
  int best = 1;
  float best_us = 0.f;
  for (int s = 1; s <= kMostSlices && (s == 1 || s <= most); ++s) {
    if (k / kBK % s != 0) continue;
    float at_full = 0.f, at_part = 0.f;
    fastest_sliced(full, n, k, s, &at_full);
    fastest_sliced(part, n, k, s, &at_part);
    const float us = fills * at_full + (1.f - fills) * at_part;
    // (asked to be worth it)
    if (s == 1 || us < (best == 1 ? 0.97f : 1.f) * best_us) best = s, best_us = us;
  }
  return best;
}

extern "C" int bt_gemm_splitk_slices(int rows_cap, int all_live, int n, int k, int most) {
  if (rows_cap <= 0 || n <= 0 || k < kBK || k % kBK != 0) return 1;
  if (cu_count() != 256) return 0;
  return remembered({rows_cap, all_live ? 1 : 0, n, k, most},
                    [&] { return fastest_slices(rows_cap, all_live != 0, n, k, most); });
}

// For a launch in slices: its tile | its pair << 4 | the pair's ratio << 8.
static int sliced_tile_or_pair(const GemmArgs &p, int splits) {
  float us = 0.f;
  const LikelyRows likely(p);
  const int named = fastest_sliced(likely, p.N, p.K, splits, &us).id;
  if (p.rows_hint <= 0) {
    unsigned ratio = 0;
    const auto at = [&](int id, int i) {
      for (const SliceModel &c : kSliceModels)
        if (c.id == id) return slice_pair_us(c, likely.rows[i], p.N, p.K, splits);
      return 0.f;
    };
    const bool either = p.valid_rows && named != 14 && splits > 1 && cu_count() == kEitherCus;
    const int pair = either ? fastest_pair(likely, p.N, splits, 3, kPairMargin * us, ratio, at) : 0;
    return named | pair << 4 | (int)(ratio << 8);
  }
  // (the waves of tile 14 add up in an order of their own: not for a row count's sake either)
  GemmArgs unnamed = p;
  unnamed.rows_hint = 0;
  const int without = fastest_sliced(LikelyRows(unnamed), p.N, p.K, splits, &us).id;
  return (named == 14) != (without == 14) ? without : named;
}

extern "C" int bt_gemm_tiles(int epilogue, int rows_cap, int n, int k, int weight_kn, int splits, int *tiles) {
  const char *who = "bt_gemm_tiles";
  BT_REQUIRE(tiles, BT_ERR_INVALID_ARGUMENT, "%s: null pointer argument", who);
  BT_REQUIRE(epilogue >= kEpiPlain && epilogue <= kEpiPartial && rows_cap > 0 && n > 0 && k >= kBK && k % kBK == 0,
             BT_ERR_INVALID_ARGUMENT, "%s: epilogue=%d rows_cap=%d n=%d k=%d", who, epilogue, rows_cap, n, k);
  const int some = 0;
  GemmArgs p{};
  p.valid_rows = &some;   // (not read: it says that the launch finds its rows on the device)
  p.rows_cap = rows_cap, p.N = n, p.K = k, p.w_kn = weight_kn;
  int answer;
  if (epilogue == kEpiPartial) {
    BT_REQUIRE(splits >= 1 && splits <= 16 && k % (splits * kBK) == 0, BT_ERR_INVALID_ARGUMENT, "%s: splits=%d", who, splits);
    answer = sliced_tile_or_pair(p, splits);
  } else {
    const WaveK few = takes_wave_k(p, epilogue == kEpiPlain);
    if (few != kWaveKNo) {
      tiles[0] = 14, tiles[1] = few == kWaveKDevice ? 4 : -1, tiles[2] = 0;
      return BT_OK;
    }
    answer = cu_count() == kEitherCus ? tile_or_pair(p, epilogue) : fastest_tile(p, epilogue);
  }
  const int pair = answer >> 4 & 15;
  tiles[0] = pair ? kTilePairs[pair - 1].first : answer & 15;
  tiles[1] = pair ? kTilePairs[pair - 1].second : -1;
  tiles[2] = (int)((unsigned)answer >> 8);
  return BT_OK;
}

extern "C" int bt_gemm_splitk(const void *a, const void *wt, void *partials, int splits,
                              const int *valid_rows, int rows_cap, int n, int k, int weight_kn,
                              void *stream) {
  return bt_gemm_splitk_rows(a, wt, partials, splits, valid_rows, rows_cap, 0, n, k, weight_kn, stream);
}

extern "C" int bt_gemm_splitk_rows(const void *a, const void *wt, void *partials, int splits,
                                   const int *valid_rows, int rows_cap, int rows_hint, int n, int k,
                                   int weight_kn, void *stream) {
  int rc = check_gemm_args("bt_gemm_splitk", a, wt, partials, rows_cap, n, k, weight_kn);
  if (rc) return rc;
  BT_REQUIRE(splits >= 1 && splits <= 16 && k % (splits * kBK) == 0, BT_ERR_INVALID_ARGUMENT,
             "bt_gemm_splitk: splits=%d must lie in [1, 16] and divide k / 64 = %d", splits,
             k / kBK);
  if (rows_cap == 0) return BT_OK;
  GemmArgs p{(const half_t *)a, (const half_t *)wt, nullptr, nullptr, valid_rows, nullptr,
             rows_cap,          n,                  k,       0,       rows_hint,  (float *)partials,
             weight_kn};
  hipStream_t st = as_stream(stream);
  const int answer = remembered({rows_cap, valid_rows != nullptr, rows_hint, n, k, splits}, [&] { return sliced_tile_or_pair(p, splits); });
  const unsigned ratio = (unsigned)answer >> 8;
  if ((answer >> 4 & 15) == 1) return launch_gemm_either<Tile9, Tile10, kEpiPartial>(p, st, ratio, splits);
  if ((answer >> 4 & 15) == 2) return launch_gemm_either<Tile10, Tile1, kEpiPartial>(p, st, ratio, splits);
  if ((answer >> 4 & 15) == 3) return launch_gemm_either<Tile10, Tile11, kEpiPartial>(p, st, ratio, splits);
  const int tile = answer & 15;
  switch (tile) {
    case 14: return launch_gemm_wave_k<kEpiPartial>(p, st, splits);
    case 4: return launch_gemm_tile<32, 64, 4, 1, 2, 2, kEpiPartial>(p, st, splits);
    case 9: return launch_gemm_tile<64, 64, 4, 2, 2, 4, kEpiPartial>(p, st, splits);
    case 10: return launch_gemm_tile<64, 128, 3, 2, 2, 4, kEpiPartial>(p, st, splits);
    case 11: return launch_gemm_tile<96, 128, 3, 3, 2, 4, kEpiPartial>(p, st, splits);
    case 12: return launch_gemm_tile<128, 192, 3, 2, 2, 4, kEpiPartial>(p, st, splits);
    default: return launch_gemm_tile<128, 128, 3, 2, 2, 4, kEpiPartial>(p, st, splits);
  }
}

extern "C" int bt_gemm_bias_gelu(const void *a, const void *wt, const void *bias, void *c,
                                 const int *valid_rows, int rows_cap, int rows_hint, int n, int k,
                                 int weight_kn, void *stream) {
  int rc = check_gemm_args("bt_gemm_bias_gelu", a, wt, c, rows_cap, n, k, weight_kn);
  if (rc) return rc;
  BT_REQUIRE(bias, BT_ERR_INVALID_ARGUMENT, "bt_gemm_bias_gelu: null bias");
  if (rows_cap == 0) return BT_OK;
  GemmArgs p{(const half_t *)a, (const half_t *)wt, (const half_t *)bias, (half_t *)c, valid_rows,
             nullptr,           rows_cap,           n,                    k,           0,
             rows_hint,         nullptr,            weight_kn};
  return launch_gemm<kEpiBiasGelu>(p, as_stream(stream));
}

extern "C" int bt_gemm_qkv_bias_split(const void *a, const int *a_row_index, const void *wt_qkv,
                                      const void *bias_qkv, void *qkv_heads,
                                      const int *valid_rows, int rows_cap, int rows_hint,
                                      int head_num, int size_per_head, int weight_kn,
                                      void *stream) {
  BT_REQUIRE(head_num > 0, BT_ERR_INVALID_ARGUMENT, "bt_gemm_qkv_bias_split: head_num=%d",
             head_num);
  BT_REQUIRE(size_per_head > 0, BT_ERR_INVALID_ARGUMENT,
             "bt_gemm_qkv_bias_split: size_per_head=%d", size_per_head);
  const int H = head_num * size_per_head;
  int rc = check_gemm_args("bt_gemm_qkv_bias_split", a, wt_qkv, qkv_heads, rows_cap, 3 * H, H,
                           weight_kn);
  if (rc) return rc;
  BT_REQUIRE(bias_qkv, BT_ERR_INVALID_ARGUMENT, "bt_gemm_qkv_bias_split: null bias");
  if (rows_cap == 0) return BT_OK;
  BT_REQUIRE(!a_row_index || valid_rows, BT_ERR_INVALID_ARGUMENT,
             "bt_gemm_qkv_bias_split: a_row_index needs valid_rows (only live rows are indexed)");
  // gathered rows are addressed with 32-bit byte offsets from the start of `a`
  BT_REQUIRE(!a_row_index || (long long)rows_cap * H * 2 <= 0x7fffffffLL, BT_ERR_UNSUPPORTED,
             "bt_gemm_qkv_bias_split: a gathered input of %d x %d halfs is beyond 2 GiB", rows_cap, H);
  GemmArgs p{(const half_t *)a, (const half_t *)wt_qkv, (const half_t *)bias_qkv,
             (half_t *)qkv_heads, valid_rows, a_row_index, rows_cap, 3 * H, H, 0, rows_hint,
             nullptr, weight_kn};
  // the head-major split is the layout of the fp16 attention kernels, which are built for
  // 64-wide heads; any other head size keeps the projections token-major [rows_cap, 3H]
  // for bt_attention_generic_f16
  if (size_per_head != 64) return launch_gemm<kEpiBias>(p, as_stream(stream));
  return launch_gemm<kEpiQkvSplit>(p, as_stream(stream));
}

extern "C" int bt_gemm_qkv_mask_rows_supported(int batch_size, int seq_len, int mask_dtype) {
  if (batch_size <= 0 || batch_size > kMaskRowsMaxBatch || seq_len <= 0) return 0;
  if (mask_dtype != BT_F16 && mask_dtype != BT_F32) return 0;
  // every workgroup reads row 0 of every sequence's mask: keep that to 64 KB
  return (long long)batch_size * seq_len * (mask_dtype == BT_F32 ? 4 : 2) <= 64 * 1024;
}

extern "C" int bt_gemm_qkv_bias_split_mask_rows(
    const void *from_tensor, const void *atten_mask, int mask_dtype, int batch_size, int seq_len,
    const void *wt_qkv, const void *bias_qkv, void *qkv_heads, int *batch_idx, int *word_idx,
    int *seq_order, int rows_hint, int head_num, int size_per_head, int weight_kn,
    void *stream) {
  const char *who = "bt_gemm_qkv_bias_split_mask_rows";
  BT_REQUIRE(head_num > 0 && size_per_head > 0, BT_ERR_INVALID_ARGUMENT,
             "%s: head_num=%d size_per_head=%d", who, head_num, size_per_head);
  BT_REQUIRE(batch_size > 0 && seq_len > 0, BT_ERR_INVALID_ARGUMENT,
             "%s: batch_size=%d seq_len=%d must be positive", who, batch_size, seq_len);
  BT_REQUIRE(bt_gemm_qkv_mask_rows_supported(batch_size, seq_len, mask_dtype), BT_ERR_UNSUPPORTED,
             "%s: batch_size=%d seq_len=%d mask_dtype=%d is outside what "
             "bt_gemm_qkv_mask_rows_supported allows", who, batch_size, seq_len, mask_dtype);
  const int H = head_num * size_per_head;
  const int rows_cap = batch_size * seq_len;
  int rc = check_gemm_args(who, from_tensor, wt_qkv, qkv_heads, rows_cap, 3 * H, H, weight_kn);
  if (rc) return rc;
  BT_REQUIRE(bias_qkv && atten_mask && batch_idx, BT_ERR_INVALID_ARGUMENT,
             "%s: null pointer argument", who);
  BT_REQUIRE(aligned16({atten_mask}), BT_ERR_INVALID_ARGUMENT,
             "%s: tensor pointers must be 16-byte aligned", who);
  // gathered rows are addressed with 32-bit byte offsets from the start of the input
  BT_REQUIRE((long long)rows_cap * H * 2 <= 0x7fffffffLL, BT_ERR_UNSUPPORTED,
             "%s: a gathered input of %d x %d halfs is beyond 2 GiB", who, rows_cap, H);
  GemmArgs p{(const half_t *)from_tensor, (const half_t *)wt_qkv, (const half_t *)bias_qkv,
             (half_t *)qkv_heads, nullptr, nullptr, rows_cap, 3 * H, H, 0, rows_hint,
             nullptr, weight_kn};
  p.mask = atten_mask;
  p.mask_f32 = mask_dtype == BT_F32;
  p.mask_B = batch_size, p.mask_S = seq_len;
  p.out_batch_idx = batch_idx, p.out_word_idx = word_idx, p.out_seq_order = seq_order;
  if (size_per_head != 64) return launch_gemm<kEpiBias>(p, as_stream(stream));
  return launch_gemm<kEpiQkvSplit>(p, as_stream(stream));
}
