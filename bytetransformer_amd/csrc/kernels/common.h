// Shared device helpers for the gfx950 kernels: vector types, wave64
// reductions, error plumbing for the C ABI.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <hip/hip_fp16.h>

#include <cstdarg>
#include <cstdint>
#include <initializer_list>
#include <cstdio>
#include <type_traits>

#include "bt_hip.h"

namespace bt {

constexpr int kWave = 64;

typedef _Float16 half_t;
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef __fp16 fp16x4_t __attribute__((ext_vector_type(4)));   // element type of the LDS transpose-read builtin
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef float float16_t __attribute__((ext_vector_type(16)));
typedef unsigned int uint4_t __attribute__((ext_vector_type(4)));
typedef unsigned int uint2_t __attribute__((ext_vector_type(2)));

// ---- error plumbing -------------------------------------------------------
void set_error(const char *fmt, ...);
int hip_fail(hipError_t e, const char *what);

#define BT_REQUIRE(cond, code, ...) \
  do {                              \
    if (!(cond)) {                  \
      ::bt::set_error(__VA_ARGS__); \
      return (code);                \
    }                               \
  } while (0)

#define BT_CHECK_LAUNCH(what)                     \
  do {                                            \
    hipError_t e__ = hipGetLastError();           \
    if (e__ != hipSuccess)                        \
      return ::bt::hip_fail(e__, what);           \
  } while (0)

// ---- launches ---------------------------------------------------------------
// A launch through the kernel's function handle, its arguments packed here.  Issuing a launch is what the host
// does all day (12 layers at 1 x 32 are 84 of them, and take the GPU no longer than the host), and as <<<>>> with
// a parameter each it looks the symbol up and copies argument by argument: us to issue an empty kernel of one / ten /
// sixteen arguments 2.9 / 3.2 / 3.6 as <<<>>>, 2.7 / 2.95 / 3.2 so; 68 bytes of arguments 3.8 and 3.5, so the
// products and the LayerNorm of half-precision layers end at 64 or a multiple of 16 beyond.  (Others do not, the float
// LayerNorm's 84 bytes among them: those layers are not bound by the host.)
// The handle, and the dynamic LDS limit beyond 64 KB, belong to the kernel on one device: they are looked up once
// for each (a lost race only repeats an idempotent call).
constexpr int kMaxDevices = 64;
constexpr size_t kMostLds = 160 * 1024;
template <auto Kernel>
struct Launch;
template <typename... P, void (*Kernel)(P...)>
struct Launch<Kernel> {
  // 0 or a BT status
  static int on(hipStream_t s, const char *what, unsigned grid, unsigned threads, size_t lds, P... args) {
    hipFunction_t f = nullptr;
    int rc = function(&f, s, what, lds > 64 * 1024);
    if (rc != BT_OK) return rc;
    alignas(16) unsigned char packed[kBytes];
    size_t at = 0;
    (pack(packed, at, args), ...);
    size_t bytes = kBytes;
    void *config[] = {HIP_LAUNCH_PARAM_BUFFER_POINTER, packed, HIP_LAUNCH_PARAM_BUFFER_SIZE, &bytes, HIP_LAUNCH_PARAM_END};
    const hipError_t e = hipModuleLaunchKernel(f, grid, 1, 1, threads, 1, 1, (unsigned)lds, s, nullptr, config);
    return e == hipSuccess ? BT_OK : hip_fail(e, what);
  }

 private:
  // (every argument at the next multiple of its alignment, as the kernel's argument segment lies)
  static constexpr size_t total() {
    size_t at = 0;
    ((at = (at + alignof(P) - 1) / alignof(P) * alignof(P) + sizeof(P)), ...);
    return at;
  }
  static constexpr size_t kBytes = total();
  template <typename T>
  static void pack(unsigned char *to, size_t &at, const T &v) {
    at = (at + alignof(T) - 1) / alignof(T) * alignof(T);
    __builtin_memcpy(to + at, &v, sizeof(T));
    at += sizeof(T);
  }
  // The kernel on the stream's device (a launch by <<<>>> goes there too, whatever the current device is).
  static int function(hipFunction_t *f, hipStream_t s, const char *what, bool large_lds) {
    static std::atomic<hipFunction_t> known[2][kMaxDevices];   // with the limit as it is, and raised
    int dev = 0;
    const bool named = reinterpret_cast<uintptr_t>(s) <= 2;   // null, hipStreamLegacy, hipStreamPerThread: the current device's
    hipError_t e = named ? hipGetDevice(&dev) : hipStreamGetDevice(s, &dev);
    if (e != hipSuccess) return hip_fail(e, what);
    const bool kept = dev >= 0 && dev < kMaxDevices;
    if (kept && (*f = known[large_lds][dev].load(std::memory_order_acquire))) return BT_OK;
    int current = dev;
    if ((e = hipGetDevice(&current)) == hipSuccess && current != dev) e = hipSetDevice(dev);
    if (e == hipSuccess && large_lds)
      e = hipFuncSetAttribute((const void *)Kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMostLds);
    if (e == hipSuccess) e = hipGetFuncBySymbol(f, (const void *)Kernel);
    if (current != dev) (void)hipSetDevice(current);
    if (e != hipSuccess) return hip_fail(e, what);
    if (kept) known[large_lds][dev].store(*f, std::memory_order_release);
    return BT_OK;
  }
};

// ---- tuning options (bt_set_option) ----------------------------------------
int option_gemm_tile();      // -1 = heuristic, else index into the tile table
int option_gemm_table_margin();   // per cent by which a measured tile must beat the model's choice
int option_layer_prepack();  // -1 = by the measured table, 0 = never, 1 = always
int option_attention_qb();   // -1 = heuristic, 1 or 2 = query blocks per wave
int option_f32_gemm_tile();  // -1 = heuristic, else index into the float GEMM's tile table
int option_attention_xcd_map();     // workgroup order of the attention kernels: 0 plain, 1 XCD-aware, 2 balanced (default), 3 balanced always
int option_prefetch();       // 1 = honour the prefetch hints of the attention entries (default), 0 = ignore
int option_attention_key_split();  // streaming attention, 64-query tiles: -1 heuristic, 0 four waves, 1 eight waves over two key halves
int option_prefetch_min_grid();   // attention launches of fewer workgroups bring workgroups of their own for the cache warm-up (default 512)

int cu_count();   // of the part that the process started on

inline hipStream_t as_stream(void *s) { return reinterpret_cast<hipStream_t>(s); }

// Every kernel moves tensors in 16-byte pieces: all tensor pointers of an entry point must
// be 16-byte aligned (null counts as aligned: nullable arguments are checked elsewhere).
inline bool aligned16(std::initializer_list<const void *> ptrs) {
  for (const void *p : ptrs)
    if (reinterpret_cast<uintptr_t>(p) & 15) return false;
  return true;
}

// Arguments of the token-major attention entries (float, and fp16 of any head size).
inline int check_generic_attention(const char *who, const void *qkv, const void *out, const int *batch_idx,
                                   const void *atten_mask, const void *attention_bias, int batch_size,
                                   int seq_len, int rows_cap, int head_num, int size_per_head,
                                   int padded_rows) {
  BT_REQUIRE(qkv && out && batch_idx, BT_ERR_INVALID_ARGUMENT, "%s: null pointer argument", who);
  BT_REQUIRE(aligned16({qkv, out, atten_mask, attention_bias}), BT_ERR_INVALID_ARGUMENT,
             "%s: tensor pointers must be 16-byte aligned", who);
  BT_REQUIRE(batch_size > 0 && seq_len > 0 && head_num > 0 && rows_cap >= 0,
             BT_ERR_INVALID_ARGUMENT, "%s: sizes must be positive", who);
  BT_REQUIRE(size_per_head > 0 && size_per_head % 8 == 0 && size_per_head <= 128,
             BT_ERR_UNSUPPORTED, "%s: size_per_head %d (supported: multiples of 8 up to 128)",
             who, size_per_head);
  BT_REQUIRE(batch_size <= 65535 && head_num <= 65535, BT_ERR_UNSUPPORTED,
             "%s: batch_size / head_num exceed the grid limit", who);
  BT_REQUIRE(!padded_rows || (long long)batch_size * seq_len <= rows_cap, BT_ERR_INVALID_ARGUMENT,
             "%s: padded rows need rows_cap >= batch_size * seq_len", who);
  return BT_OK;
}

// ---- wave64 reductions ----------------------------------------------------
// Sum over the 64 lanes, as a wave-uniform value, with data-parallel-primitive adds only (the steps of
// wave_inclusive_sum): a step is a few clocks, where one through the LDS pipe takes over a hundred.
__device__ __forceinline__ float wave_sum(float v) {
#if defined(__HIP_DEVICE_COMPILE__)
  const auto moved = [](float x, auto ctrl, auto rows) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(ctrl)::value,
                                                                 decltype(rows)::value, 0xf, true));
  };
  using all = std::integral_constant<int, 0xf>;
  v += moved(v, std::integral_constant<int, 0x111>{}, all{});   // row_shr:1
  v += moved(v, std::integral_constant<int, 0x112>{}, all{});   // row_shr:2
  v += moved(v, std::integral_constant<int, 0x114>{}, all{});   // row_shr:4
  v += moved(v, std::integral_constant<int, 0x118>{}, all{});   // row_shr:8
  v += moved(v, std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{});   // row_bcast:15 -> rows 1, 3
  v += moved(v, std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{});   // row_bcast:31 -> rows 2, 3
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
#else
  return v;
#endif
}

// Largest over the 64 lanes of values that are not negative, wave-uniform, by the same steps.
__device__ __forceinline__ float wave_max(float v) {
#if defined(__HIP_DEVICE_COMPILE__)
  const auto moved = [](float x, auto ctrl, auto rows) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(ctrl)::value,
                                                                 decltype(rows)::value, 0xf, true));
  };
  using all = std::integral_constant<int, 0xf>;
  v = fmaxf(v, moved(v, std::integral_constant<int, 0x111>{}, all{}));
  v = fmaxf(v, moved(v, std::integral_constant<int, 0x112>{}, all{}));
  v = fmaxf(v, moved(v, std::integral_constant<int, 0x114>{}, all{}));
  v = fmaxf(v, moved(v, std::integral_constant<int, 0x118>{}, all{}));
  v = fmaxf(v, moved(v, std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{}));
  v = fmaxf(v, moved(v, std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{}));
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
#else
  return v;
#endif
}

// ---- wave-uniform values ----------------------------------------------------
// x / d for any 32-bit x, where inverse = floor(2^32 / d)  (2^32 - 1 for d = 1)
__device__ __forceinline__ unsigned divide(unsigned x, unsigned d, unsigned inverse) {
  const unsigned q = (unsigned)((unsigned long long)x * inverse >> 32);   // the quotient or one less
  return q + (x - q * d >= d ? 1u : 0u);
}
inline unsigned inverse_of(unsigned d) { return d > 1 ? (unsigned)((1ull << 32) / d) : 0xffffffffu; }
// x / d for wave-uniform 0 <= x < 2^21 and 0 < d, neither known to the host: a quarter of the instructions of a division.
__device__ __forceinline__ int divide_small(int x, int d) {
  int q = __builtin_amdgcn_readfirstlane((int)((float)x * __builtin_amdgcn_rcpf((float)d)));   // the quotient, one more or one less
  q -= q * d > x ? 1 : 0;
  return q + (x - q * d >= d ? 1 : 0);
}
// A load into scalar registers, of what nothing in this launch writes, at a wave-uniform address.
template <typename T>
__device__ __forceinline__ T scalar_load(const T *from) {
#if defined(__HIP_DEVICE_COMPILE__)
  return *(const __attribute__((address_space(4))) T *)from;
#else
  return *from;
#endif
}

// Inclusive prefix sum across the 64 lanes of a wave.
__device__ __forceinline__ int wave_inclusive_scan(int v, int lane) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    int t = __shfl_up(v, o, 64);
    if (lane >= o) v += t;
  }
  return v;
}


// Inclusive prefix sum over the 64 lanes with data-parallel-primitive adds only: four
// shifts inside each row of 16, then lane 15 of rows 0 / 2 into rows 1 / 3 and lane 31
// into the upper half.
__device__ __forceinline__ int wave_inclusive_sum(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);   // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);   // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);   // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);   // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 -> rows 1, 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 -> rows 2, 3
  return v;
}

// Sum over the 64 lanes, as a wave-uniform value.
__device__ __forceinline__ int wave_total(int v) {
  return __builtin_amdgcn_readlane(wave_inclusive_sum(v), 63);
}

// Number of row elements >= 0.5 (the length rule of the offsets, remove_padding.h:36-86),
// counted by one wave for R mask rows at a time (row r may be null: length 0).
// A mask row that has not been touched since the last layer comes from HBM: the wave
// fetches it with 16-byte loads, 4 per lane in flight over the R rows (R rows of up to
// 2048 / R halfs are one round trip; element by element a 512-token row was eight
// dependent ones).  Rows may start at any element; the last piece of a row that does not divide lies
// over the one before it and counts what that one has not (element by element, as those rows were read before, each
// was up to 16 dependent round trips: 12 layers, operator, 12 x 380 857 -> 820 us, 16 x 250 931 -> 908, 24 x 100 707 -> 694).
template <typename T, int R>
__device__ __forceinline__ void wave_row_lengths(const T *const *row, int S, int lane,
                                                 int (&count)[R]) {
  constexpr int kVec = 16 / (int)sizeof(T);
  constexpr int kUnroll = 4 / R;
  static_assert(R == 1 || R == 2 || R == 4, "rows per call");
#pragma unroll
  for (int r = 0; r < R; ++r) count[r] = 0;
  if (S > kWave) {   // (else an element a lane)
    typedef uint4_t any_element __attribute__((aligned(2)));
    for (int j0 = 0; j0 < S; j0 += kWave * kVec * kUnroll) {
      uint4_t raw[R][kUnroll];
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
          const int j = j0 + (u * kWave + lane) * kVec;
          raw[r][u] = uint4_t{0u, 0u, 0u, 0u};
          if (row[r] && j < S) raw[r][u] = *(const any_element *)(row[r] + min(j, S - kVec));
        }
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
          const T *e = (const T *)&raw[r][u];
#pragma unroll
          for (int i = 0; i < kVec; ++i) count[r] += (float)e[i] >= 0.5f;
          const int again = j0 + (u * kWave + lane) * kVec - (S - kVec);   // elements that the piece before has
          if (again > 0 && again < kVec)
#pragma unroll
            for (int i = 0; i < kVec - 1; ++i) count[r] -= i < again && (float)e[i] >= 0.5f;
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) count[r] = wave_total(count[r]);
    return;
  }
  float e[R];
#pragma unroll
  for (int r = 0; r < R; ++r) e[r] = row[r] && lane < S ? (float)row[r][lane] : 0.f;
#pragma unroll
  for (int r = 0; r < R; ++r) count[r] = __popcll(__ballot(e[r] >= 0.5f));
}
template <typename T>
__device__ __forceinline__ int wave_row_length(const T *__restrict__ row, int S, int lane) {
  const T *const rows[1] = {row};
  int count[1];
  wave_row_lengths<T, 1>(rows, S, lane, count);
  return count[0];
}

// ---- 64 x 64 tile of the weight pre-pack: wt[n][k] = w[k][n] ---------------------------
// 256 threads (t = 0..255) move one tile through `tile`; both sides are 16-byte accesses.
// `live` = false keeps a thread group in step (it meets the barrier) without touching memory.
constexpr int kTransposePitch = 64 + 2;
__device__ __forceinline__ void transpose_tile_64(const half_t *__restrict__ w,
                                                  half_t *__restrict__ wt, int K, int N, int k0,
                                                  int n0, half_t (*tile)[kTransposePitch], int t,
                                                  bool live) {
  // read 64 k-rows x 128 B: thread -> (row = t/8 + 32*i, 16-byte chunk t%8)
  const int r = t >> 3, c = (t & 7) * 8;
  if (live) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int k = k0 + r + 32 * i, n = n0 + c;
      uint4_t v = {0u, 0u, 0u, 0u};
      if (k < K && n < N) v = *(const uint4_t *)(w + (size_t)k * N + n);
      const half_t *h = (const half_t *)&v;
#pragma unroll
      for (int e = 0; e < 8; ++e) tile[r + 32 * i][c + e] = h[e];
    }
  }
  __syncthreads();
  if (live) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int n = n0 + r + 32 * i, k = k0 + c;
      if (n < N && k < K) {
        half8_t o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = tile[c + e][r + 32 * i];
        *(half8_t *)(wt + (size_t)n * K + k) = o;
      }
    }
  }
}

// ---- jobs that ride along with a layer's first launch ----------------------------------
// k-contiguous copies [N, K] of up to four [K, N] weight matrices, and ranges whose
// 128-byte lines are touched once so that later launches find them in the memory-side cache.
struct WeightJobs {
  const half_t *w[4];        // [K, N] as the caller stores them
  half_t *wt[4];             // [N, K] copies to make
  int K[4], N[4];
  int tiles_n[4];            // 64 x 64 tiles along n
  int tile_end[4];           // tiles up to and including matrix i
  int count;                 // 0 = none
  // range r holds the 128-byte lines [warm_end[r - 1], warm_end[r]) of the concatenation
  const char *warm[4];
  unsigned warm_end[4];
};
// Fills `out` from the tail arguments of the C entries that take such jobs (checks them and
// reports errors under the name `who`; returns a BT status).  With the `prefetch` option off
// the ranges to warm are dropped.
int make_weight_jobs(const char *who, WeightJobs *out, int weight_count, const void *const *w,
                     void *const *wt, const int *k, const int *n, int warm_count,
                     const void *const *warm, const unsigned long long *warm_bytes);

// U tiles at a time per group of 256 threads (t = thread index in the group): tiles t0 .. t0 +
// U - 1 of the concatenated tile list of the jobs (ids from pw.tile_end[pw.count - 1] on do not
// exist).  All the loads of the U tiles are in flight together, so a group that has several
// tiles to move pays one memory round trip for U of them.  `tiles` holds U consecutive LDS
// tiles of this group.  The whole workgroup must call it together (two barriers inside).
template <int U>
__device__ __forceinline__ void transpose_tiles_64(const WeightJobs &pw, int t0,
                                                   half_t (*tiles)[kTransposePitch], int t) {
  const int r = t >> 3, c = (t & 7) * 8;
  const int t_end = pw.tile_end[pw.count - 1];
  uint4_t v[U][2];
  const half_t *src[U];
  half_t *dst[U];
  int K[U], N[U], k0[U], n0[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int tile = t0 + u;
    int j = 0, first = 0;
#pragma unroll
    for (int q = 1; q < 4; ++q)
      if (q < pw.count && tile >= pw.tile_end[q - 1]) {
        j = q;
        first = pw.tile_end[q - 1];
      }
    const int tl = tile - first;
    src[u] = pw.w[j], dst[u] = pw.wt[j], K[u] = tile < t_end ? pw.K[j] : 0, N[u] = pw.N[j];
    k0[u] = (tl / pw.tiles_n[j]) * 64, n0[u] = (tl % pw.tiles_n[j]) * 64;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int k = k0[u] + r + 32 * i, n = n0[u] + c;
      v[u][i] = uint4_t{0u, 0u, 0u, 0u};
      if (k < K[u] && n < N[u]) v[u][i] = *(const uint4_t *)(src[u] + (size_t)k * N[u] + n);
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const half_t *h = (const half_t *)&v[u][i];
#pragma unroll
      for (int e = 0; e < 8; ++e) tiles[u * 64 + r + 32 * i][c + e] = h[e];
    }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < U; ++u) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int n = n0[u] + r + 32 * i, k = k0[u] + c;
      if (n < N[u] && k < K[u]) {
        half8_t o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = tiles[u * 64 + c + e][r + 32 * i];
        *(half8_t *)(dst[u] + (size_t)n * K[u] + k) = o;
      }
    }
  }
  __syncthreads();
}

// One dword of the lines l, l + stride, ... below `last` (range r holds the 128-byte lines
// [end[r - 1], end[r]) of a concatenation of four).  Ordinary loads, two in flight, so that the compiler
// knows which registers they return to: as assembly whose result nobody reads, their register was
// reused for the next turn's address while the load was under way, an illegal access once in a long while.
// (One / two / four in flight, 12 layers in us: 1 x 32 360 / 366 / 379, 1 x 256 443 / 449 / 461, captured 4 x
// 96 417 / 414 / 418, 6 x 250 under its mask 779 / 772 / 761.)
__device__ __forceinline__ void touch_lines(const char *const (&base)[4], const unsigned (&end)[4], unsigned l,
                                            unsigned last, unsigned stride) {
  constexpr int kFlight = 2;
  unsigned long long at[4];   // where line 0 of the concatenation would lie, counted back from range r
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    at[r] = (unsigned long long)base[r] - (r ? end[r - 1] : 0u) * 128ull;
    asm volatile("" : "+s"(at[r]));   // (in registers: selected by line, the compiler loads it again for each)
  }
  for (; l < last; l += kFlight * stride) {
    unsigned got[kFlight];
#pragma unroll
    for (int u = 0; u < kFlight; ++u) {
      const unsigned line = min(l + u * stride, last - 1);
      unsigned long long from = at[0];
#pragma unroll
      for (int r = 1; r < 4; ++r) from = line >= end[r - 1] ? at[r] : from;
      // (in the global address space by name; ranges may start at any byte)
      typedef unsigned any_byte __attribute__((aligned(1)));
      got[u] = *(const __attribute__((address_space(1))) any_byte *)(from + line * 128ull);
    }
    asm volatile("" ::"v"(got[0]), "v"(got[1]));   // (both have returned)
  }
}

// The same for lines 0 .. lines - 1, at(l) each, by workgroup `mine` of `per` (THREADS threads each).
template <int THREADS, typename At>
__device__ __forceinline__ void touch_lines(unsigned lines, unsigned mine, unsigned per, At at) {
  constexpr int kFlight = 2;
  for (unsigned l = mine * THREADS + __builtin_amdgcn_workitem_id_x(); l < lines; l += kFlight * per * THREADS) {
    unsigned got[kFlight];
#pragma unroll
    for (int u = 0; u < kFlight; ++u) {
      typedef unsigned any_byte __attribute__((aligned(1)));
      const unsigned line = min(l + u * per * THREADS, lines - 1);
      got[u] = *(const __attribute__((address_space(1))) any_byte *)at(line);
    }
    asm volatile("" ::"v"(got[0]), "v"(got[1]));   // (both have returned)
  }
}

// ---- which tile a position of the XCD-aware order is ---------------------------------------
// XCD x works on the positions [x * per, (x + 1) * per) and every XCD has an L2 of its own, so
// what the launch fetches from the memory side is, per XCD, the distinct rows of A plus the
// distinct columns of W in its range.  The order therefore walks the tile grid in panels of
// `gn` tile columns (row tiles outermost inside a panel) such that a range of `per` positions
// is close to a square of operand elements: gn BN = (per / gn) BM.  Plain row-major order
// (gn = tiles_n) makes every XCD read the whole weight as soon as a range is a tile row
// long: 28 MB instead of 7 MB for the QKV product of 256 rows at hidden 768.
constexpr int kMostPanelTiles = 1 << 20;
struct TilePanels {
  int tiles_m, tiles_n, gn;
  __device__ __forceinline__ void locate(int L, int &tile_m, int &tile_n) const {   // L < kMostPanelTiles
    const int panel = divide_small(L, tiles_m * gn);
    const int r = L - panel * tiles_m * gn;
    const int w = min(gn, tiles_n - panel * gn);   // the last panel may be narrower
    tile_m = divide_small(r, w);
    tile_n = panel * gn + r - tile_m * w;
  }
};
template <int BM, int BN>
__device__ __forceinline__ TilePanels tile_panels(int tiles_m, int tiles_n, int per) {
  int gn = (int)(__builtin_amdgcn_sqrtf((float)per * ((float)BM / (float)BN)) + 0.5f);
  gn = max(gn, divide_small(per + tiles_m - 1, tiles_m));   // a range taller than the grid is wider instead
  return TilePanels{tiles_m, tiles_n, __builtin_amdgcn_readfirstlane(max(1, min(gn, tiles_n)))};
}

// blockIdx.x and threadIdx.x without the call that some floating-point flags keep from being inlined
// (attention.hip): behind it the workgroup's number counts as a vector value, and every address and branch
// at the head of a kernel with it.
__device__ __forceinline__ unsigned workgroup_id() { return __builtin_amdgcn_workgroup_id_x(); }
__device__ __forceinline__ unsigned thread_id() { return __builtin_amdgcn_workitem_id_x(); }

// ---- balanced work list of the streaming attention kernels -------------------------
// Within an XCD the hardware deals consecutive workgroups to its 32 CUs round-robin
// (slot s of the XCD lands on CU s % 32), and a launch of a few workgroups per CU is
// resident at once, so the static order alone decides what each CU gets.  With a fixed
// number of query-tile slots per sequence the tile index is s % 4 at 512 tokens: one CU
// in four received only the last tiles - dead for most sequences - while others held
// three live ones of the longest sequences.  Here the live (pair, query tile) items of
// the XCD - (sequence, head) pairs p = x (mod 8) over the longest-first order, the tiles
// of a pair adjacent, so that one L2 serves a pair's K / V to all of them - are counted
// on the device, and slot s takes item j = s in even rounds of 32 and the mirrored
// position in odd rounds: a CU that drew a long item in one round draws a short one in
// the next.  Every lane of a wave holds one rank: lengths, tile counts and a wave prefix
// sum invert j -> (rank, head, tile) with the two dependent loads a plain look-up needs
// as well.  Args: a kernel argument struct with B, S, heads, nqb, padded_rows, batch_idx
// and seq_order.

struct AttWork {
  int b, head, qb, seq_start, len;
  bool exists;
};
// Shape of the balanced order of a streaming-attention launch over (B, S, heads): entries =
// workgroups of the launch (0: such a launch does not use the balanced order), bq = queries
// per tile (64 or 128), nqb = tile slots per sequence.  One function decides for the
// attention launcher and for whoever builds the list ahead of it.
struct AttListPlan {
  unsigned entries;
  int bq, nqb;
};
AttListPlan att_worklist_plan(int B, int S, int heads);
// Arguments of att_work_balanced when the offsets come from somewhere else than a kernel's
// own argument struct (the layer prologue builds the list from lengths it holds in LDS).
struct AttListArgs {
  int B, S, heads, nqb, padded_rows;
  const int *batch_idx, *seq_order;
};
template <int BQ, typename Args>
__device__ __forceinline__ AttWork att_work_balanced(const Args &p, unsigned int workgroup) {
  AttWork w{0, 0, 0, 0, 0, false};
  const int lane = thread_id() & 63;
  const int x = workgroup & 7, s = workgroup >> 3;
  const int round = s >> 5, pos = s & 31;
  const int j = (round << 5) + ((round & 1) ? 31 - pos : pos);
  int carry = 0;
  for (int base = 0; base < p.B; base += 64) {
    const int r = base + lane;
    const bool valid = r < p.B;
    const int seq = valid ? (p.seq_order ? p.seq_order[r] : r) : 0;
    const int start = p.batch_idx[seq];
    const int len = valid ? p.batch_idx[seq + 1] - start : 0;
    const int nq = p.padded_rows ? p.S : len;
    const int nqb = valid ? min((nq + BQ - 1) / BQ, p.nqb) : 0;
    const int first = r * p.heads;   // pairs [first, first + heads) belong to rank r
    const int cnt = ((first + p.heads + 7 - x) >> 3) - ((first + 7 - x) >> 3);
    const int mine = cnt * nqb;
    const int incl = wave_inclusive_sum(mine);
    const int lo = carry + incl - mine;   // first item of this rank
    const unsigned long long hit = __builtin_amdgcn_ballot_w64(mine > 0 && j >= lo && j < lo + mine);
    if (hit) {
      const int src = __builtin_ctzll(hit);
      const int jj = j - __builtin_amdgcn_readlane(lo, src);
      const int nqb_s = __builtin_amdgcn_readlane(nqb, src);
      const int first_s = (base + src) * p.heads;
      w.b = __builtin_amdgcn_readlane(seq, src);
      w.seq_start = __builtin_amdgcn_readlane(start, src);
      w.len = __builtin_amdgcn_readlane(len, src);
      w.qb = jj % nqb_s;
      // the (jj / nqb_s)-th head h of the rank with first_s + h = x (mod 8)
      w.head = ((x - first_s) & 7) + 8 * (jj / nqb_s);
      w.exists = true;
      return w;
    }
    carry += __builtin_amdgcn_readlane(incl, 63);
  }
  return w;
}

// Stores that write through the XCD's L2 instead of leaving the line dirty in it.  The L2s of the eight
// XCDs are not coherent, so a kernel ends by writing its dirty lines back, and the next one waits for
// that: 4 us behind a launch that stored 30 MB.  Written through, the lines leave while the other
// workgroups still compute (and stay in the memory-side cache, which a non-temporal store would pass by).
// FFN1 at 4800 rows 28.7 -> 26.3 us a launch, at 9830 rows 55.4 -> 52.1, projection at 4800 rows 9.8 ->
// 9.0, QKV at 911 rows 8.8 -> 8.3.
// The attention keeps ordinary stores: its rows leave in pieces of 32 bytes, which the L2 joins; written through
// they cost 0.3 to 1.4 % of a forward.
// (Stores that the compiler knows, agent scope being what writes through: it keeps them in order with other
// accesses to the same memory and waits for what a matrix instruction has yet to write into their registers.)
__device__ __forceinline__ void store_through(void *to, uint4_t v) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_global_store_b128((__attribute__((address_space(1))) uint4_t *)to, v, "agent");
#endif
}
__device__ __forceinline__ void store_through(void *to, uint2_t v) {
#if defined(__HIP_DEVICE_COMPILE__)
  __hip_atomic_store((__attribute__((address_space(1))) unsigned long long *)to, __builtin_bit_cast(unsigned long long, v),
                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#endif
}

}  // namespace bt
