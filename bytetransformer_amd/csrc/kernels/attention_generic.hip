// Fused multi-head attention on fp16 for any head size up to 128 (a multiple of 8), over
// token-major projections qkv [rows, 3 * hidden] (Q | K | V per row, bias already added).  Role of the
// reference's unfused path for head sizes other than 64 (attention_nofused.cu:27-114,
// softmax.h:25-60) without its logits buffer and its transposes.
//
// The structure is that of the streaming kernel for 64-wide heads (attention.hip): S^T = K.Q^T so
// that the accumulator already is the "B" operand of O^T = V^T.P^T, K and V tiles of 64 keys
// straight from memory into an LDS ring, V^T through the LDS transpose read, a lazy running maximum, row
// sums on an MFMA with an all-ones operand.  Two things differ: the head size is the kernel's D = 32 ND
// or less (columns past it stay zero in LDS and registers), and the probabilities enter the
// second product as the sum of two fp16 numbers, because this entry's probabilities have always been
// floats.  fp16 has few exponents, so they are computed 2^13 times as large as they are (the quotient O / l
// does not see it; the lazy maximum lets them grow to four times that): 23 bits from 2^-15 of the largest
// probability of a row on, and an absolute error of at most 2^-38 of it below.
//
// Before, this path ran on v_mfma_f32_32x32x2_f32 with every operand widened to float, at 1/16 of the
// fp16 rate, 128 queries per workgroup and 328 registers at head size 128: batch 8 x 300, six
// heads of 128, took 56 us; now 10.8.  It is bound by the dependency chain of a tile
// (products, maximum, exponentials, products) at one or two waves per SIMD.
#include "attention_common.h"

#include <type_traits>

namespace bt {
namespace {

constexpr int kGenThreads = 256;
constexpr int kGenKeys = 64;   // keys per tile
constexpr float kGenShift = 13.0f;   // probabilities are exp2(x - m + kGenShift), ...
constexpr float kGenLazy = 2.0f;     // ... where m lags behind the maximum by this much at most
static_assert(kGenShift + kGenLazy < 16.0f, "the leading fp16 of a probability overflows at 2^16");

struct GenericAttArgs {
  const half_t *qkv;      // [rows, 3H]
  half_t *out;            // [rows, H]
  const int *batch_idx;
  const int *seq_order;   // optional: rank -> sequence, longest first
  const half_t *mask;     // optional [B,S,S]
  const half_t *bias;     // optional [heads,S,S]
  int B, S, heads;
  float scale_log2e;
  int padded_rows;
  int nqb;                // query tiles per sequence
  int balanced;           // 1: the live query tiles are dealt evenly to the CUs (common.h)
  int d;                  // head size <= D
  int every_key;          // 1: all S keys of a sequence take part, whatever its length
  WarmDuty warm;          // ranges that the launches after this one will read (weights)
};

// 16-byte chunk swizzles of a [64][D] tile, D / 8 chunks per row (compare swz_k / swz_v of the
// 64-wide kernel).  K: 16 consecutive rows at one chunk on distinct banks; V: the 8 rows x 32 bytes
// of a transpose-read pass likewise.  Both repeat after 16 rows, so a lane's offset inside a
// tile is a constant plus a multiple of 16 rows.
template <int D>
__device__ __forceinline__ int gen_swz_k(int row) {
  return D == 128 ? row & 15 : D == 64 ? (row >> 1) & 7 : (row >> 2) & 3;
}
template <int D>
__device__ __forceinline__ int gen_swz_v(int row) {
  return D == 128 ? (row & 7) << 1 : D == 64 ? ((row >> 1) & 3) << 1 : ((row >> 2) & 1) << 1;
}

// QB 16-query blocks per wave, four waves.
template <int ND, int KIND, int QB>
__global__ __launch_bounds__(kGenThreads, 2) void attention_generic_kernel(GenericAttArgs p) {
  constexpr bool ADD = KIND != kAddNone;
  constexpr int D = 32 * ND, CPR = D / 8, DB = D / 16, BQ = 64 * QB;
  constexpr int kTile = kGenKeys * D;         // halfs of a K or V tile
  constexpr int NLD = CPR / 4;                // load instructions per wave for K, and as many for V
  __shared__ __attribute__((aligned(1024))) half_t ring[2 * 2 * kTile];

  if (workgroup_id() >= p.warm.grid_work) {
    warm_slice<kGenThreads>(p.warm);
    return;
  }
  int b, head, seq_start, seq_len, qb_index;
  if (p.balanced) {
    const AttWork w = att_work_balanced<BQ>(p, workgroup_id());
    if (!w.exists) {
      warm_slice<kGenThreads>(p.warm);
      return;
    }
    b = w.b, head = w.head, seq_start = w.seq_start, seq_len = w.len, qb_index = w.qb;
  } else {
    const unsigned lin = workgroup_id(), slot = lin >> 3;
    const unsigned pair = (slot / p.nqb) * 8 + (lin & 7);
    if (pair >= (unsigned)(p.B * p.heads)) {
      warm_slice<kGenThreads>(p.warm);
      return;
    }
    const int rank = pair / p.heads;
    head = pair % p.heads;
    b = p.seq_order ? p.seq_order[rank] : rank;
    seq_start = p.batch_idx[b];
    seq_len = p.batch_idx[b + 1] - seq_start;
    qb_index = (int)(slot % p.nqb);
  }
  const int klen = ((KIND & kAddMask) && p.padded_rows) || p.every_key ? p.S : seq_len;
  const int row_start = p.padded_rows ? b * p.S : seq_start;
  const int nq = p.padded_rows ? p.S : seq_len;
  const int q0 = qb_index * BQ;
  if (q0 >= nq) {
    warm_slice<kGenThreads>(p.warm);
    return;
  }

  const int tid = thread_id(), lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lq = lane & 15, lg = lane >> 4;
  const int d = p.d, dc = d >> 3;             // head size, in 16-byte chunks
  const int H = p.heads * d;
  const size_t ld = (size_t)3 * H;
  const half_t *Q = p.qkv + (size_t)row_start * ld + head * d;
  const half_t *K = Q + H, *V = K + H;

  if (d < D) {   // chunks past the head size are never fetched: they stay zero
    for (int i = tid; i < 2 * 2 * kTile / 8; i += kGenThreads) *(uint4_t *)(ring + 8 * i) = uint4_t{0u, 0u, 0u, 0u};
    __syncthreads();
  }

  half8_t qf[QB][ND];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const int q = q0 + (wave * QB + qb) * 16 + lq;
#pragma unroll
    for (int dh = 0; dh < ND; ++dh) {
      uint4_t v = {0u, 0u, 0u, 0u};
      if (q < nq && 4 * dh + lg < dc) v = *(const uint4_t *)(Q + (size_t)q * ld + 32 * dh + 8 * lg);
      qf[qb][dh] = __builtin_bit_cast(half8_t, v);
    }
  }

  int koff[ND];
  unsigned vaddr[DB];   // (bytes, from the ring's start in LDS)
#pragma unroll
  for (int dh = 0; dh < ND; ++dh) koff[dh] = lq * D + (((4 * dh + lg) ^ gen_swz_k<D>(lq)) << 3);
#pragma unroll
  for (int db = 0; db < DB; ++db) {
    const int row0 = 4 * lg + (lq >> 2), c = 2 * db + ((lq & 3) >> 1);
    vaddr[db] = lds_address(ring) + 2 * (row0 * D + ((c ^ gen_swz_v<D>(row0)) << 3) + 4 * (lq & 1));
  }

  // Tile copy: instruction i of a wave fills the 64 chunk slots from (i * 4 + wave) * 64 on; a
  // lane fetches the chunk that the swizzle puts in its slot.
  int ld_row[NLD], k_chunk[NLD], v_chunk[NLD];
#pragma unroll
  for (int i = 0; i < NLD; ++i) {
    const int slot = (i * 4 + wave) * 64 + lane, c = slot % CPR;
    ld_row[i] = slot / CPR;
    k_chunk[i] = c ^ gen_swz_k<D>(ld_row[i]);
    v_chunk[i] = c ^ gen_swz_v<D>(ld_row[i]);
  }
  auto issue_tile = [&](int t, int stage) {
    half_t *sK = ring + stage * 2 * kTile, *sV = sK + kTile;
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      const size_t row = (size_t)min(t * kGenKeys + ld_row[i], klen - 1) * ld;
      half_t *k_dst = sK + (i * 4 + wave) * 512, *v_dst = sV + (i * 4 + wave) * 512;
      if (d == D) {
        lds_dma16(K + row + 8 * k_chunk[i], k_dst);
        lds_dma16(V + row + 8 * v_chunk[i], v_dst);
      } else {
        if (k_chunk[i] < dc) lds_dma16(K + row + 8 * k_chunk[i], k_dst);
        if (v_chunk[i] < dc) lds_dma16(V + row + 8 * v_chunk[i], v_dst);
      }
    }
  };

  // the additive terms of a tile are requested one tile ahead
  uint2_t mask_raw[QB][4], bias_raw[QB][4];
  auto term_row = [&](const half_t *tensor, int plane, int planes, int qb) {
    return TermRow(tensor, (size_t)plane * p.S + min(q0 + (wave * QB + qb) * 16 + lq, p.S - 1), p.S,
                   (size_t)planes * p.S);
  };
  auto fetch_terms = [&](int t) {
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      const int key = t * kGenKeys + lg * 4;
      if (KIND & kAddMask) {
        const TermRow row = term_row(p.mask, b, p.B, qb);
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) mask_raw[qb][kb] = row.fetch<false>(key + kb * 16);
      }
      if (KIND & kAddBias) {
        const TermRow row = term_row(p.bias, head, p.heads, qb);
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) bias_raw[qb][kb] = row.fetch<false>(key + kb * 16);
      }
    }
  };

  float4_t o[DB + 1][QB];   // o[DB]: row sums (an all-ones V^T)
  float m_run[QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    m_run[qb] = kNegBig;
#pragma unroll
    for (int db = 0; db <= DB; ++db) o[db][qb] = float4_t{0.f, 0.f, 0.f, 0.f};
  }
  const half8_t ones = {1, 1, 1, 1, 1, 1, 1, 1};
  const float c = p.scale_log2e, cs = ADD ? 1.0f : c;
  const bool wave_live = q0 + wave * QB * 16 < nq;
  const int ntiles = (klen + kGenKeys - 1) / kGenKeys;
  if (ntiles > 0) {
    issue_tile(0, 0);
    if (ADD && wave_live) fetch_terms(0);
  }

  for (int t = 0; t < ntiles; ++t) {
    att_wait_vmcnt<0>();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (t + 1 < ntiles) issue_tile(t + 1, (t + 1) & 1);
    if (!wave_live) continue;   // such a wave only copies and keeps the barriers
    const half_t *sK = ring + (t & 1) * 2 * kTile, *sV = sK + kTile;
    const int k0 = t * kGenKeys;

    float4_t s[4][QB];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) s[kb][qb] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int dh = 0; dh < ND; ++dh) {
        const half8_t kf = *(const half8_t *)(sK + kb * 16 * D + koff[dh]);
#pragma unroll
        for (int qb = 0; qb < QB; ++qb)
          s[kb][qb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, qf[qb][dh], s[kb][qb], 0, 0, 0);
      }
    }
    if constexpr (ADD) {
#pragma unroll
      for (int qb = 0; qb < QB; ++qb)
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
          const int key = k0 + kb * 16 + lg * 4;
          uint2_t mv = mask_raw[qb][kb], bv = bias_raw[qb][kb];
          if (k0 + kGenKeys > klen) {   // (the last tile's may lie at the end of the tensor)
            if (KIND & kAddMask) mv = term_row(p.mask, b, p.B, qb).in_order(mv, key);
            if (KIND & kAddBias) bv = term_row(p.bias, head, p.heads, qb).in_order(bv, key);
          }
          s[kb][qb] = add_terms<KIND>(s[kb][qb], c, mv, bv);
        }
      if (t + 1 < ntiles) fetch_terms(t + 1);
    }
    if (k0 + kGenKeys > klen) {
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const bool dead = k0 + kb * 16 + lg * 4 + r >= klen;
#pragma unroll
          for (int qb = 0; qb < QB; ++qb) s[kb][qb][r] = dead ? kNegBig : s[kb][qb][r];
        }
    }

    half8_t pf[2][QB], pl[2][QB];   // probabilities: leading and trailing halfs
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      float mx = s[0][qb][0];
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[kb][qb][r]);
      mx = rows_max(mx);
      const float m_new = (mx - m_run[qb]) * cs > kGenLazy ? mx : m_run[qb];
      const float mc = __builtin_fmaf(m_new, cs, -kGenShift);
      if (__builtin_amdgcn_ballot_w64(m_new != m_run[qb]) != 0) {
        const float alpha = fast_exp2(__builtin_fmaf(m_run[qb], cs, -kGenShift) - mc);
#pragma unroll
        for (int db = 0; db <= DB; ++db) o[db][qb] *= alpha;
      }
      m_run[qb] = m_new;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int r = 0; r < 4; r += 2) {
          const float2_t e = {fast_exp2(__builtin_fmaf(s[kb][qb][r], cs, -mc)),
                              fast_exp2(__builtin_fmaf(s[kb][qb][r + 1], cs, -mc))};
          const half2_t h = __builtin_convertvector(e, half2_t);
          const half2_t l = __builtin_convertvector(float2_t{e[0] - (float)h[0], e[1] - (float)h[1]}, half2_t);
          pf[kb >> 1][qb][(kb & 1) * 4 + r] = h[0], pf[kb >> 1][qb][(kb & 1) * 4 + r + 1] = h[1];
          pl[kb >> 1][qb][(kb & 1) * 4 + r] = l[0], pl[kb >> 1][qb][(kb & 1) * 4 + r + 1] = l[1];
        }
    }

    // k-slot (lg, i) <-> key 32 kk + 16 (i >> 2) + 4 lg + (i & 3); four d-blocks of V^T at a time
    const unsigned v_tile = 2 * ((t & 1) * 2 * kTile + kTile);
    auto accumulate = [&](auto kk_tag) {
      constexpr int kk = decltype(kk_tag)::value, kRow = 2 * D;
#pragma unroll
      for (int d0 = 0; d0 < DB; d0 += 4) {
        constexpr int N = DB < 4 ? DB : 4;   // (D = 96 ends on two)
        uint2_t lo[4] = {}, hi[4] = {};
#pragma unroll
        for (int i = 0; i < N; ++i)
          if (d0 + i < DB) {
            lo[i] = lds_read_tr<32 * kk * kRow>(vaddr[d0 + i] + v_tile);
            hi[i] = lds_read_tr<(32 * kk + 16) * kRow>(vaddr[d0 + i] + v_tile);
          }
        lds_wait_tied<0>(lo, hi);
#pragma unroll
        for (int i = 0; i < N; ++i) {
          if (d0 + i >= DB) continue;
          const half8_t vf = __builtin_bit_cast(half8_t, uint4_t{lo[i][0], lo[i][1], hi[i][0], hi[i][1]});
#pragma unroll
          for (int qb = 0; qb < QB; ++qb) {
            o[d0 + i][qb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, pf[kk][qb], o[d0 + i][qb], 0, 0, 0);
            o[d0 + i][qb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, pl[kk][qb], o[d0 + i][qb], 0, 0, 0);
          }
        }
      }
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        o[DB][qb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, pf[kk][qb], o[DB][qb], 0, 0, 0);
        o[DB][qb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, pl[kk][qb], o[DB][qb], 0, 0, 0);
      }
    };
    accumulate(std::integral_constant<int, 0>{});
    accumulate(std::integral_constant<int, 1>{});
  }

#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const float inv = 1.0f / (o[DB][qb][0] + 1e-6f * 8192.0f);   // (2^kGenShift)
    const int q = q0 + (wave * QB + qb) * 16 + lq;
    if (q >= nq) continue;
    half_t *dst = p.out + (size_t)(row_start + q) * H + head * d + 4 * lg;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      if (16 * db + 4 * lg >= d) continue;
      const float4_t v = o[db][qb] * inv;
      *(half4_t *)(dst + 16 * db) = half4_t{(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]};
    }
  }
  warm_slice<kGenThreads>(p.warm);
}

template <int ND, int KIND>
int launch_generic_kind(const GenericAttArgs &p, bool wide, unsigned grid, hipStream_t s) {
  const char *who = "attention_generic_kernel";
  if constexpr (ND < 4 || KIND == kAddNone)
    if (wide) return Launch<attention_generic_kernel<ND, KIND, 2>>::on(s, who, grid, kGenThreads, 0, p);
  return Launch<attention_generic_kernel<ND, KIND, 1>>::on(s, who, grid, kGenThreads, 0, p);
}
template <int ND>
int launch_generic(const GenericAttArgs &p, int kind, bool wide, unsigned grid, hipStream_t s) {
  switch (kind) {
    case kAddNone: return launch_generic_kind<ND, kAddNone>(p, wide, grid, s);
    case kAddMask: return launch_generic_kind<ND, kAddMask>(p, wide, grid, s);
    case kAddBias: return launch_generic_kind<ND, kAddBias>(p, wide, grid, s);
    case kAddZero: return launch_generic_kind<ND, kAddZero>(p, wide, grid, s);
    default: return launch_generic_kind<ND, kAddBoth>(p, wide, grid, s);
  }
}

}  // namespace
}  // namespace bt

using namespace bt;

extern "C" int bt_attention_generic_f16_warm(const void *qkv, void *out, const int *batch_idx,
                                             const int *seq_order, const void *atten_mask,
                                             const void *attention_bias, int batch_size, int seq_len,
                                             int rows_cap, int head_num, int size_per_head,
                                             float scale, int padded_rows, const void *const *prefetch,
                                             const unsigned long long *prefetch_bytes,
                                             int prefetch_count, void *stream) {
  const char *who = "bt_attention_generic_f16";
  int rc = check_generic_attention(who, qkv, out, batch_idx, atten_mask, attention_bias, batch_size,
                                         seq_len, rows_cap, head_num, size_per_head, padded_rows);
  if (rc != BT_OK) return rc;
  GenericAttArgs p{(const half_t *)qkv, (half_t *)out, batch_idx, seq_order, (const half_t *)atten_mask,
                   (const half_t *)attention_bias, batch_size, seq_len, head_num, scale * kLog2e,
                   padded_rows ? 1 : 0};
  p.d = size_per_head;
  // (mask given but nothing to add: its meaning on padded rows stays)
  p.every_key = drop_terms_of_one_key(seq_len, p.mask, p.bias) && padded_rows;
  // 128-query tiles from 1300 of them on, the line of the 64-wide kernel: below it the launch is as
  // long as its longest chain of tiles and more, shorter workgroups fill the chip better
  const long long blocks128 = (long long)((seq_len + 127) / 128) * head_num * batch_size;
  // (heads beyond 96 with additive terms would not fit the registers two query blocks at a time)
  const int kind = add_kind(p.mask, p.bias, p.scale_log2e);
  const bool wide = blocks128 >= 1300 && !(size_per_head > 96 && kind != kAddNone);
  p.nqb = wide ? (seq_len + 127) / 128 : (seq_len + 63) / 64;
  // the balanced order from the third round of 32 workgroups per XCD on and up to 128 sequences, or
  // always / never by the option (the conditions of the 64-wide kernel)
  const unsigned per_xcd = ((unsigned)batch_size * head_num + 7) / 8 * p.nqb;
  const int order = option_attention_xcd_map();
  p.balanced = order == 3 || (order == 2 && per_xcd > 64 && batch_size <= 128);
  unsigned grid = p.balanced ? (per_xcd + 31) / 32 * 32 * 8 : per_xcd * 8;
  rc = plan_warm_duty(who, p.warm, grid, prefetch, prefetch_bytes, prefetch_count);
  if (rc != BT_OK) return rc;
  hipStream_t s = as_stream(stream);
  switch ((size_per_head + 31) / 32) {
    case 1: return launch_generic<1>(p, kind, wide, grid, s);
    case 2: return launch_generic<2>(p, kind, wide, grid, s);
    case 3: return launch_generic<3>(p, kind, wide, grid, s);
    default: return launch_generic<4>(p, kind, wide, grid, s);
  }
}

extern "C" int bt_attention_generic_f16(const void *qkv, void *out, const int *batch_idx,
                                        const int *seq_order, const void *atten_mask,
                                        const void *attention_bias, int batch_size, int seq_len,
                                        int rows_cap, int head_num, int size_per_head,
                                        float scale, int padded_rows, void *stream) {
  return bt_attention_generic_f16_warm(qkv, out, batch_idx, seq_order, atten_mask, attention_bias,
                                       batch_size, seq_len, rows_cap, head_num, size_per_head, scale,
                                       padded_rows, nullptr, nullptr, 0, stream);
}
