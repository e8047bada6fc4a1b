// Fused multi-head attention for gfx950 over head-major Q/K/V
// ([3][heads][rows_cap][64], fp16), one workgroup per (query tile, head,
// sequence), wave64 + v_mfma_f32_16x16x32_f16.
//
// Both kernels compute the logits TRANSPOSED, S^T = K.Q^T, so that the MFMA
// accumulator of a 16-key block (lane = query, 4 consecutive keys per lane) is
// already laid out as the "B" operand of the second product O^T = V^T.P^T: the
// probabilities never leave registers.  K and V rows travel global -> LDS with
// direct-to-LDS 16-byte loads (no staging registers) into XOR-swizzled
// row-major tiles; the "A" operand of the second product, V^T, is fetched with
// the LDS transpose read (ds_read_b64_tr_b16), so V is never transposed in
// memory.
//
//   attention_short_kernel    whole K / V of the sequence resident in LDS,
//                             all logits of a query tile in registers, exact
//                             two-pass softmax: P = exp(s-max)/(sum+1e-6) is
//                             rounded to fp16 before P.V exactly as
//                             attention_fused.cu:348-381 does.
//   attention_grouped_kernel  K / V streamed in 64-key tiles through a 2- or 3-stage
//                             LDS ring with an online softmax; handles any
//                             length; the [S, S] logits never exist.
//
// Keys at or past the sequence length are excluded by index (the mask tensor is
// not read), the convention of the reference's remove-padding kernels
// (attention_fused.cu:359, attention_fused_long.cu:254).  Tile rows past the
// length are fetched from the last valid row (finite data, never out of
// bounds) and their probabilities are forced to zero.
#include "attention_common.h"

#include <type_traits>

namespace bt {

constexpr int kAttThreads = 256;
constexpr int kHeadDim = 64;
struct AttArgs {
  const half_t *qkv;   // [3][heads][rows_cap][64]
  half_t *out;         // [rows, heads*64]
  const int *batch_idx;
  const int *seq_order;   // optional: grid z -> sequence, longest first (null = identity)
  const half_t *mask;     // optional [B,S,S] 0/1 mask, padded rows only: every key of the
                          // sequence's S rows takes part, shifted by (mask-1)*10000
  const half_t *bias;     // optional [heads,S,S] term added to the scaled logits
  WarmDuty warm;          // ranges that the NEXT kernels will read (weights)
  int B, S, rows_cap, heads;
  float scale_log2e;   // scale * log2(e)
  int padded_rows;
  int nqb;             // query tiles per sequence (set by the launcher)
  unsigned per_nqb, per_heads;   // floor(2^32 / nqb), floor(2^32 / heads) (set by the launcher)
  unsigned nqb_grid;   // host only: workgroups of the launch
  int xcd_map;         // 0: plain (tile, head, sequence) order, 1: XCD-aware, 2: XCD-aware and balanced over the CUs
  const int *mask_ok;  // optional int[256] from bt_mask_prefix_slots: all non-zero = the mask
                       // is the plain prefix mask of the lengths, and is then ignored
  int every_key;       // 1: all S keys of a sequence take part, whatever its length
  const int4 *work_list;   // optional: entry w of bt_attention_worklist = what workgroup w of the
                           // balanced order works on {sequence or -1, head | tile << 16, first row, length}
};

// Which (sequence rank, head, query tile) a workgroup of the 1-D grid works on.  The
// hardware deals consecutive workgroup ids round-robin to the 8 XCDs.  In a plain
// (tile fastest) order the XCD of a workgroup is a function of its query-tile index, and
// with ragged lengths the high tiles are mostly dead: some XCDs get a fraction of the
// work of others.  The XCD-aware order gives XCD x the (sequence, head) pairs
// p = x (mod 8) - pairs counted sequence-major over the longest-first order, so every
// XCD sees the same mix of lengths - and runs the query tiles of one pair back to back
// on that XCD, whose L2 then serves the pair's K / V to all of them.
struct AttItem {
  int rank, head, qb;
  bool exists;
};
__device__ __forceinline__ AttItem att_item(const AttArgs &p) {
  AttItem it;
  const unsigned lin = workgroup_id();
  const unsigned slot = p.xcd_map ? lin >> 3 : lin;
  unsigned pair = divide(slot, p.nqb, p.per_nqb);
  it.qb = slot - pair * p.nqb;
  if (p.xcd_map) pair = pair * 8 + (lin & 7);
  it.exists = pair < (unsigned)(p.B * p.heads);
  it.rank = divide(pair, p.heads, p.per_heads);
  it.head = pair - it.rank * p.heads;
  return it;
}

// What the streaming kernel needs to find its work, as leading kernel arguments of their own: those are in
// scalar registers when a wave starts, where the struct's fields are memory reads.
struct AttFirst {
  const half_t *qkv;
  const int *batch_idx, *order;   // order: seq_order, or the work list (kAttList)
  unsigned batch_heads;           // B | heads << 16
  int S, rows_cap;
  unsigned grid_work, nqb, per_nqb, per_heads, flags;
};
constexpr unsigned kAttMap = 3, kAttList = 4, kAttPadded = 8, kAttEveryKey = 16;   // flags (kAttMap: xcd_map)
#define BT_ATT_FIRST                                                                                   \
  const half_t *qkv, const int *batch_idx, const int *order, unsigned batch_heads, int S, int rows_cap, \
      unsigned grid_work, unsigned nqb, unsigned per_nqb, unsigned per_heads, unsigned flags
#define BT_ATT_FIRST_NAMES \
  qkv, batch_idx, order, batch_heads, S, rows_cap, grid_work, nqb, per_nqb, per_heads, flags
#define BT_ATT_FIRST_OF(f) \
  f.qkv, f.batch_idx, f.order, f.batch_heads, f.S, f.rows_cap, f.grid_work, f.nqb, f.per_nqb, f.per_heads, f.flags
inline AttFirst att_first(const AttArgs &a) {
  const bool list = a.xcd_map == 2 && a.work_list;
  return AttFirst{a.qkv, a.batch_idx, list ? (const int *)a.work_list : a.seq_order,
                  (unsigned)a.B | (unsigned)a.heads << 16, a.S, a.rows_cap, a.warm.grid_work, (unsigned)a.nqb, a.per_nqb,
                  a.per_heads, (unsigned)a.xcd_map | (list ? kAttList : 0) | (a.padded_rows ? kAttPadded : 0) |
                                   (a.every_key ? kAttEveryKey : 0)};
}
// ... and what it needs later: every argument byte costs the host (4.6 us to issue a launch with the whole of AttArgs
// here, 4.3 with this), so the additive terms travel with the kernels that apply them.
struct AttTerms {
  const half_t *mask, *bias;
  const int *mask_ok;
};
struct AttNoTerms {};
template <int KIND>
struct AttTail : std::conditional_t<(KIND & kAddBoth) != 0, AttTerms, AttNoTerms> {
  half_t *out;
  float scale_log2e;
  unsigned warm_first, warm_ends, warm_forms_turns;
  unsigned warm_shape[kWarmRanges];
  const char *warm_base[kWarmRanges];
};
template <int KIND>
static AttTail<KIND> att_tail(const AttArgs &a) {
  AttTail<KIND> t{};
  if constexpr ((KIND & kAddBoth) != 0) t.mask = a.mask, t.bias = a.bias, t.mask_ok = a.mask_ok;
  t.out = a.out, t.scale_log2e = a.scale_log2e, t.warm_first = a.warm.first, t.warm_ends = a.warm.ends;
  t.warm_forms_turns = a.warm.forms_turns;
  for (int r = 0; r < kWarmRanges; ++r) t.warm_shape[r] = a.warm.shape[r], t.warm_base[r] = a.warm.base[r];
  return t;
}
template <int KIND>
__device__ __forceinline__ AttArgs att_args(BT_ATT_FIRST, const AttTail<KIND> &tail) {
  AttArgs p{};
  if constexpr ((KIND & kAddBoth) != 0) p.mask = tail.mask, p.bias = tail.bias, p.mask_ok = tail.mask_ok;
  p.out = tail.out, p.scale_log2e = tail.scale_log2e, p.warm.first = tail.warm_first;
  p.warm.ends = tail.warm_ends, p.warm.forms_turns = tail.warm_forms_turns;
#pragma unroll
  for (int r = 0; r < kWarmRanges; ++r) p.warm.shape[r] = tail.warm_shape[r], p.warm.base[r] = tail.warm_base[r];
  p.qkv = qkv, p.batch_idx = batch_idx;
  p.seq_order = flags & kAttList ? nullptr : order;
  p.work_list = flags & kAttList ? (const int4 *)order : nullptr;
  p.B = batch_heads & 0xffff, p.heads = batch_heads >> 16, p.S = S, p.rows_cap = rows_cap;
  p.warm.grid_work = grid_work, p.nqb = nqb, p.per_nqb = per_nqb, p.per_heads = per_heads;
  p.xcd_map = flags & kAttMap, p.padded_rows = (flags & kAttPadded) != 0, p.every_key = (flags & kAttEveryKey) != 0;
  return p;
}

// What a workgroup of the streaming kernel works on, all of it in scalar registers.
struct AttTile {
  int b, head, qb, seq_start, seq_len;
};
// (Found by scalar loads.  With the work in scalar registers
// 12 layers take, before -> after: 4 x 96 443 -> 437 us, 7 x 217 627 -> 620, 100 x 120 1696 -> 1677.)
template <int BQ>
__device__ __forceinline__ bool att_tile(const AttArgs &p, AttTile &t) {
  if (workgroup_id() >= p.warm.grid_work) return false;
  if (p.work_list) {
    // the balanced order, looked up by an earlier launch: one scalar load
    typedef int entry_t __attribute__((ext_vector_type(4)));
    const entry_t w = scalar_load((const entry_t *)p.work_list + workgroup_id());
    t = AttTile{w[0], w[1] & 0xffff, w[1] >> 16, w[2], w[3]};
    return w[0] >= 0;
  }
  if (p.xcd_map == 2) {
    const AttWork w = att_work_balanced<BQ>(p, workgroup_id());
    t = AttTile{w.b, w.head, w.qb, w.seq_start, w.len};
    return w.exists;
  }
  const AttItem item = att_item(p);
  if (!item.exists) return false;
  const int b = p.seq_order ? scalar_load(p.seq_order + item.rank) : item.rank;
  // (no offsets: padded rows under a mask tensor, which says everything)
  const int start = p.batch_idx ? scalar_load(p.batch_idx + b) : b * p.S;
  const int len = p.batch_idx ? scalar_load(p.batch_idx + b + 1) - start : p.S;
  t = AttTile{b, item.head, item.qb, start, len};
  return true;
}

// 16-byte chunk swizzles of a [rows][64] fp16 tile (8 chunks per 128-byte row).
// K is read with ds_read_b128 by 16 consecutive rows at one chunk: slot =
// chunk ^ (row>>1 & 7) spreads them over all 64 banks.  V is read with the
// transpose read, 4 consecutive rows x 32 bytes per 16 lanes: slot =
// chunk ^ 2*(row>>1 & 3) puts those four rows on distinct banks.
__device__ __forceinline__ int swz_k(int row) { return (row >> 1) & 7; }
__device__ __forceinline__ int swz_v(int row) { return ((row >> 1) & 3) << 1; }

// V^T fragment for d-block db and key pair-block kk of a [keys][64] swizzled V
// tile: 8 keys {32kk+4g+r, 32kk+16+4g+r} for d = 16db + (lane&15), g = lane>>4.
__device__ __forceinline__ half8_t load_vt_frag(const half_t *sV, int kk, int db, int lq, int lg) {
  const int row0 = 32 * kk + 4 * lg + (lq >> 2);
  const int c = 2 * db + ((lq & 3) >> 1), sub = 4 * (lq & 1);
  const half_t *p0 = sV + row0 * kHeadDim + ((c ^ swz_v(row0)) << 3) + sub;
  const int row1 = row0 + 16;
  const half_t *p1 = sV + row1 * kHeadDim + ((c ^ swz_v(row1)) << 3) + sub;
  const fp16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4f16(
      (__attribute__((address_space(3))) fp16x4_t *)p0);
  const fp16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4f16(
      (__attribute__((address_space(3))) fp16x4_t *)p1);
  const half4_t l4 = __builtin_bit_cast(half4_t, lo), h4 = __builtin_bit_cast(half4_t, hi);
  return half8_t{l4[0], l4[1], l4[2], l4[3], h4[0], h4[1], h4[2], h4[3]};
}

__device__ __forceinline__ half8_t load_k_frag(const half_t *sK, int kb, int dh, int lq, int lg) {
  const int row = 16 * kb + lq;
  return *(const half8_t *)(sK + row * kHeadDim + (((4 * dh + lg) ^ swz_k(row)) << 3));
}

// ---------------------------------------------------------------------------
// grouped / streaming kernel
// ---------------------------------------------------------------------------
constexpr int kKT = 64;                          // keys per streamed tile
constexpr int kTileHalfs = kKT * kHeadDim;       // one K or V tile

// QB 16-query blocks per wave; workgroup covers 4*QB*16 queries.  KIND: a mask tensor and / or an
// attention bias contribute additive terms to the logits.
// KS = 2 (key split): eight waves; waves 4-7 work on the same queries as waves 0-3 but on
// the other 64-key half of every 128-key ring slot, with their own running maximum, sum
// and output, and the two halves are merged through LDS at the end.  The dependency chain
// of a query tile - what bounds a launch of a few workgroups per CU, where the longest
// sequence's workgroups finish last - is half as long, and twice the waves hide it.
// WQ = 1, KS = 4, one stage: 16 queries per workgroup, whose four waves take a 64-key tile each.  For a launch that
// leaves most CUs idle: up to 256 keys are one step instead of four in a row (12 layers at 1 x 256 under a mask,
// 192 workgroups instead of 48: 429 -> 409 us; at 1 x 128 392 -> 388, at 2 x 120 410 -> 408.  With a second
// stage for longer sequences a workgroup fills the CU, and those of the warm-up wait for it: 436 -> 454).
template <int QB, int KIND, int STAGES, int KS, int WQ>
__device__ __forceinline__ void attention_tile(const AttArgs &p, const AttTile &item, half_t *ring) {
  constexpr bool ADD = KIND != kAddNone;
  constexpr int BQ = WQ * QB * 16, kWaves = WQ * KS;
  constexpr int AHEAD = STAGES > 1 ? STAGES - 1 : 1;     // tiles in flight beyond the one being consumed
  constexpr int kSlotKeys = kKT * KS;   // keys per ring slot
  constexpr int kSlotHalfs = KS * 2 * kTileHalfs;
  static_assert(STAGES <= 2 || (STAGES == 3 && !ADD), "ring depth (one: all keys fit a slot); the additive terms alternate between two register sets");
  const int b = item.b, head = item.head, seq_start = item.seq_start, seq_len = item.seq_len, qb_index = item.qb;
  // A mask tensor that the device-side check found to be the plain prefix mask adds 0 to
  // the logits of the sequence's keys and removes the others: the lengths say the same.
  const half_t *mask = KIND & kAddMask ? p.mask : nullptr;
  if ((KIND & kAddMask) && p.mask_ok) {
    const int l = thread_id() & 63;
    const int ok = p.mask_ok[l] & p.mask_ok[l + 64] & p.mask_ok[l + 128] & p.mask_ok[l + 192];
    if (__builtin_amdgcn_ballot_w64(ok == 0) == 0) mask = nullptr;
  }
  // with a mask tensor every one of the S key rows takes part
  int klen = mask || p.every_key ? p.S : seq_len;
  const int row_start = p.padded_rows ? b * p.S : seq_start;
  const int nq = p.padded_rows ? p.S : klen;
  const int q0 = qb_index * BQ;
  if (q0 >= nq) return;
  // (as a vector value: with a scalar length the compiler reshapes the loop over the key tiles, copies the
  // running output in every tile and needs 132 registers instead of 116, three waves per SIMD instead of four)
  asm("" : "+v"(klen));

  const int tid = thread_id(), lane = tid & 63;
  const int wave_all = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave = wave_all % WQ;       // which 16-query blocks
  const int grp = KS > 1 ? wave_all / WQ : 0;   // which 64 keys of a ring slot
  const int lq = lane & 15, lg = lane >> 4;

  const size_t head_stride = (size_t)p.rows_cap * kHeadDim;
  const half_t *Q = p.qkv + (size_t)head * head_stride + (size_t)row_start * kHeadDim;
  const half_t *K = Q + (size_t)p.heads * head_stride;
  const half_t *V = K + (size_t)p.heads * head_stride;

  // Q fragments: "B" operand, lane (query lq, k-group lg) holds d = 32*dh + 8*lg .. +8
  half8_t qf[QB][2];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const int q = q0 + (wave * QB + qb) * 16 + lq;
#pragma unroll
    for (int dh = 0; dh < 2; ++dh) {
      uint4_t v = {0u, 0u, 0u, 0u};
      if (q < nq) v = *(const uint4_t *)(Q + (size_t)q * kHeadDim + 32 * dh + 8 * lg);
      qf[qb][dh] = __builtin_bit_cast(half8_t, v);
    }
  }

  // Where this lane's operand fragments sit inside a K or V tile, in halfs: the swizzle
  // term of a fragment's row does not depend on the key block (K: row = 16 kb + lq, V: row
  // = 32 kk + 4 lg + (lq >> 2); the block index drops out of swz_k / swz_v), so the whole
  // address is one of these six lane constants plus a compile-time offset - ring stage,
  // key block - that fits the instruction's immediate field: no address arithmetic is
  // left in the loop over the key tiles (it was a quarter of its vector instructions).
  int koff[2];
  unsigned vaddr[4];   // (bytes, from the ring's start in LDS)
#pragma unroll
  for (int dh = 0; dh < 2; ++dh) koff[dh] = lq * kHeadDim + (((4 * dh + lg) ^ swz_k(lq)) << 3);
#pragma unroll
  for (int db = 0; db < 4; ++db) {
    const int row0 = 4 * lg + (lq >> 2);
    const int c = 2 * db + ((lq & 3) >> 1);
    vaddr[db] = lds_address(ring) +
                2 * (row0 * kHeadDim + ((c ^ swz_v(row0)) << 3) + 4 * (lq & 1) + grp * 2 * kTileHalfs);
  }

  // Slot copy: 16 load instructions per 64-key tile (8 rows each; 0-7 = K, 8-15 = V),
  // 16 / WQ per wave.  Lane -> (row, slot) and fetches the chunk the swizzle puts
  // in that slot.
  const int ld_row = lane >> 3, ld_slot = lane & 7;
  auto issue_tile = [&](int t, int stage) {
    half_t *sbase = ring + stage * kSlotHalfs;
    const int k0 = t * kSlotKeys;
#pragma unroll
    for (int i = 0; i < 16 / WQ; ++i) {
      const int id_all = i * kWaves + wave_all;   // 0 .. 16 KS - 1
      const int sub = id_all >> 4, id = id_all & 15;
      const int row = (id & 7) * 8 + ld_row;
      const int key = min(k0 + sub * kKT + row, klen - 1);
      if (id < 8)
        lds_dma16(K + (size_t)key * kHeadDim + ((ld_slot ^ swz_k(row)) << 3),
                  sbase + sub * 2 * kTileHalfs + (id & 7) * 8 * kHeadDim);
      else
        lds_dma16(V + (size_t)key * kHeadDim + ((ld_slot ^ swz_v(row)) << 3),
                  sbase + sub * 2 * kTileHalfs + kTileHalfs + (id & 7) * 8 * kHeadDim);
    }
  };

  // o[4] is a fifth "d block" fed with an all-ones V^T fragment: the MFMA then
  // accumulates the row sums of the (fp16-rounded) probabilities, already
  // reduced over the wave, in the same rescaled form as O.
  float4_t o[5][QB];
  float m_run[QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    m_run[qb] = kNegBig;
#pragma unroll
    for (int db = 0; db < 5; ++db) o[db][qb] = float4_t{0.f, 0.f, 0.f, 0.f};
  }
  const half8_t ones = {1, 1, 1, 1, 1, 1, 1, 1};

  const bool wave_live = q0 + wave * QB * 16 < nq;
  const int ntiles = (klen + kSlotKeys - 1) / kSlotKeys;

  const float c = p.scale_log2e;
  // after the mask term is folded in, the logits already are in the exp2 domain
  const float cs = ADD ? 1.0f : c;
  // The additive terms of a tile are requested one whole tile ahead, in front of that tile's K and V,
  // into the register set that its parity names; fetched where they are used, every tile waited for
  // memory a second time.  Batch 1 x 256 under its mask: 9.8 -> 7.6 us a launch, 6 x 250 (rows that
  // start anywhere) 17.3 -> 10.5, 12 x 380 with a bias 31.9 -> 22.6.
  const bool with_mask = (KIND & kAddMask) && mask;   // (the verdict may have dropped it)
  uint2_t mask_raw[2][QB][4], bias_raw[2][QB][4];
  auto term_row = [&](const half_t *tensor, int plane, int planes, int qb) {
    return TermRow(tensor, (size_t)plane * p.S + min(q0 + (wave * QB + qb) * 16 + lq, p.S - 1), p.S,
                   (size_t)planes * p.S);
  };
  const bool ragged_end = klen % kSlotKeys != 0;   // every tile but the last is full
  [[maybe_unused]] const int masked_tile = ragged_end ? ntiles - 1 : -1;
  auto fetch_terms = [&](int t, auto set_tag) {
    constexpr int SET = decltype(set_tag)::value;
    const int key = t * kSlotKeys + grp * kKT + lg * 4;
    auto fetch = [&](auto inside_tag) {
      constexpr bool INSIDE = decltype(inside_tag)::value;
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        if (with_mask) {
          const TermRow row = term_row(mask, b, p.B, qb);
#pragma unroll
          for (int kb = 0; kb < 4; ++kb) mask_raw[SET][qb][kb] = row.template fetch<INSIDE>(key + kb * 16);
        }
        if (KIND & kAddBias) {
          const TermRow row = term_row(p.bias, head, p.heads, qb);
#pragma unroll
          for (int kb = 0; kb < 4; ++kb) bias_raw[SET][qb][kb] = row.template fetch<INSIDE>(key + kb * 16);
        }
      }
    };
    if (ragged_end && t == ntiles - 1)
      fetch(std::false_type{});
    else
      fetch(std::true_type{});
  };
  // (two query blocks with both kinds of terms: one set of registers, requested at the top of the tile)
  constexpr bool kTermsAhead = ADD && !(QB == 2 && KIND == kAddBoth);
  if (kTermsAhead && ntiles > 0) fetch_terms(0, std::integral_constant<int, 0>{});
#pragma unroll
  for (int t = 0; t < AHEAD; ++t)
    if (t < ntiles) issue_tile(t, t);

  // ST: the ring stage of tile t, a compile-time constant (the loop below is unrolled over
  // the stages)
  auto process_tile = [&](int t, auto masked_tag, auto stage_tag) {
    constexpr bool MASKED = decltype(masked_tag)::value;
    constexpr int ST = decltype(stage_tag)::value;
    // This wave's share of tile t has landed once only what was requested after it is outstanding: the
    // four loads of the next tile in a three-deep ring, nothing in a two-deep one, which requests a tile
    // (and its terms before it) last of all.
    if (AHEAD > 1 && t + 1 < ntiles)
      att_wait_vmcnt<4>();
    else
      att_wait_vmcnt<0>();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (kTermsAhead && t + 1 < ntiles) fetch_terms(t + 1, std::integral_constant<int, (ST + 1) & 1>{});
    if (ADD && !kTermsAhead) fetch_terms(t, std::integral_constant<int, ST & 1>{});
    if (STAGES > 1 && t + AHEAD < ntiles) issue_tile(t + AHEAD, (ST + AHEAD) % STAGES);
    // a wave whose queries all lie past the sequence, or whose half of the slot lies past
    // the last key, only copies and keeps the barriers
    const int k0 = t * kSlotKeys + grp * kKT;
    if (!wave_live || (KS > 1 && k0 >= klen)) return;
    const half_t *sK = ring + ST * kSlotHalfs + grp * 2 * kTileHalfs;

    // S^T = K . Q^T for this tile: 4 key blocks x QB query blocks
    float4_t s[4][QB];
    const float4_t zero4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const half8_t kf0 = *(const half8_t *)(sK + kb * 16 * kHeadDim + koff[0]);
      const half8_t kf1 = *(const half8_t *)(sK + kb * 16 * kHeadDim + koff[1]);
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        s[kb][qb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf0, qf[qb][0], zero4, 0, 0, 0);
        s[kb][qb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf1, qf[qb][1], s[kb][qb], 0, 0, 0);
      }
    }
    if constexpr (ADD) {
      auto apply = [&](auto kind_tag) {
        constexpr int K = decltype(kind_tag)::value;
#pragma unroll
        for (int qb = 0; qb < QB; ++qb)
#pragma unroll
          for (int kb = 0; kb < 4; ++kb) {
            uint2_t mv = mask_raw[ST & 1][qb][kb], bv = bias_raw[ST & 1][qb][kb];
            if (MASKED) {
              const int key = k0 + kb * 16 + lg * 4;
              if (K & kAddMask) mv = term_row(mask, b, p.B, qb).in_order(mv, key);
              if (K & kAddBias) bv = term_row(p.bias, head, p.heads, qb).in_order(bv, key);
            }
            s[kb][qb] = add_terms<K>(s[kb][qb], c, mv, bv);
          }
      };
      if (with_mask || !(KIND & kAddMask))
        apply(std::integral_constant<int, KIND>{});
      else
        apply(std::integral_constant<int, KIND & kAddBias>{});
    }
    if (MASKED) {
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const bool dead = k0 + kb * 16 + lg * 4 + r >= klen;
#pragma unroll
          for (int qb = 0; qb < QB; ++qb) s[kb][qb][r] = dead ? kNegBig : s[kb][qb][r];
        }
    }

    // the V^T fragments of the tile: keys 32 kk + 4 lg + .. (lo) and 16 rows further on (hi), on their
    // way while the probabilities are computed
    constexpr int kV = 2 * (ST * kSlotHalfs + kTileHalfs), kRow = 2 * kHeadDim;
    uint2_t v_lo[2][4], v_hi[2][4];
#pragma unroll
    for (int db = 0; db < 4; ++db) {
      v_lo[0][db] = lds_read_tr<kV>(vaddr[db]);
      v_hi[0][db] = lds_read_tr<kV + 16 * kRow>(vaddr[db]);
    }
#pragma unroll
    for (int db = 0; db < 4; ++db) {
      v_lo[1][db] = lds_read_tr<kV + 32 * kRow>(vaddr[db]);
      v_hi[1][db] = lds_read_tr<kV + 48 * kRow>(vaddr[db]);
    }

    // The reference point of a query's exponentials follows its maximum lazily: it moves
    // only when the maximum has grown by more than kLazyMax binary orders (the first tile
    // always does).  Probabilities then reach at most 2^kLazyMax - far inside fp16, the
    // sums are fp32 - and the quotient O / l does not depend on the reference point, while
    // the rescaling of the running output, a quarter of the vector work of a tile, is
    // left to the few tiles where a maximum jumps.  Whether one has is asked of each lane's own
    // keys: a row's maximum has grown if one of its four lanes' has, so the rows are folded, and
    // the exponentials wait for it, only then (with the order of the two halves below, us:
    // 16 x 1024 full 68.9 -> 66.6, ragged 43.5 -> 41.9; 16 x 512 14.5 -> 14.3; 16 heads, 32 x 384, 25.1 -> 24.3).
    float mx[QB];
    bool grown = false;
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      mx[qb] = fmaxf(s[0][qb][0], s[0][qb][1]);
      mx[qb] = fmaxf(fmaxf(mx[qb], s[0][qb][2]), s[0][qb][3]);
#pragma unroll
      for (int kb = 1; kb < 4; ++kb) {
        mx[qb] = fmaxf(fmaxf(mx[qb], s[kb][qb][0]), s[kb][qb][1]);
        mx[qb] = fmaxf(fmaxf(mx[qb], s[kb][qb][2]), s[kb][qb][3]);
      }
      grown |= (mx[qb] - m_run[qb]) * cs > kLazyMax;
    }
    if (__builtin_amdgcn_ballot_w64(grown) != 0) {
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        const float m_row = rows_max(mx[qb]);
        const float m_new = (m_row - m_run[qb]) * cs > kLazyMax ? m_row : m_run[qb];
        const float alpha = fast_exp2(m_run[qb] * cs - m_new * cs);
#pragma unroll
        for (int db = 0; db < 5; ++db) o[db][qb] *= alpha;
        m_run[qb] = m_new;
      }
    }
    half8_t pf[2][QB];
    auto probs = [&](auto kk_tag) {
      constexpr int kk = decltype(kk_tag)::value;
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        const float mc = m_run[qb] * cs;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int kb = 2 * kk + h;
          float e[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) e[r] = fast_exp2(__builtin_fmaf(s[kb][qb][r], cs, -mc));
          const half2_t h01 = __builtin_convertvector(float2_t{e[0], e[1]}, half2_t);
          const half2_t h23 = __builtin_convertvector(float2_t{e[2], e[3]}, half2_t);
          pf[kk][qb][h * 4 + 0] = h01[0];
          pf[kk][qb][h * 4 + 1] = h01[1];
          pf[kk][qb][h * 4 + 2] = h23[0];
          pf[kk][qb][h * 4 + 3] = h23[1];
        }
      }
    };
    // O^T += V^T . P^T ; k-slot (lg, s) <-> key 32*kk + 16*(s>>2) + 4*lg + (s&3)
    auto product = [&](auto kk_tag) {
      constexpr int kk = decltype(kk_tag)::value;
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        const half8_t vf = __builtin_bit_cast(
            half8_t, uint4_t{v_lo[kk][db][0], v_lo[kk][db][1], v_hi[kk][db][0], v_hi[kk][db][1]});
#pragma unroll
        for (int qb = 0; qb < QB; ++qb)
          o[db][qb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, pf[kk][qb], o[db][qb], 0, 0, 0);
      }
#pragma unroll
      for (int qb = 0; qb < QB; ++qb)
        o[4][qb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, pf[kk][qb], o[4][qb], 0, 0, 0);
    };
    using kk0 = std::integral_constant<int, 0>;
    using kk1 = std::integral_constant<int, 1>;
    // (the second half's exponentials behind the first half's products: the matrix pipe works beside them)
    probs(kk0{});
    lds_wait_tied<8>(v_lo[0], v_hi[0]);
    product(kk0{});
    probs(kk1{});
    lds_wait_tied<0>(v_lo[1], v_hi[1]);
    product(kk1{});
  };
  // No masking code on the steady-state path.  The kernels with terms compare with the number of the tile:
  // asked the other way the compiler kept a loop of its own for sequences that end with a tile, and the
  // wide kernel under mask and bias spilled 66 registers (32 x 500: 97 -> 74.7 us; 32 x 512: 134 -> 114).  The
  // wide kernel without terms is faster the other way (32 x 512: 42.4 against 47 us).
  auto step = [&](int t, auto stage_tag) {
    bool masked;
    if constexpr (ADD)
      masked = t == masked_tile;
    else
      masked = ragged_end && t == ntiles - 1;
    if (masked)
      process_tile(t, std::true_type{}, stage_tag);
    else
      process_tile(t, std::false_type{}, stage_tag);
  };
  // one turn of the ring per iteration: tile t sits in stage t % STAGES
  for (int t = 0; t < ntiles; t += STAGES) {
    step(t, std::integral_constant<int, 0>{});
    if constexpr (STAGES >= 2) {
      if (t + 1 < ntiles) step(t + 1, std::integral_constant<int, 1>{});
    }
    if constexpr (STAGES == 3) {
      if (t + 2 < ntiles) step(t + 2, std::integral_constant<int, 2>{});
    }
  }

  if (KS > 1) {
    // fold the other keys into the first group's: its waves get maximum, sum and output handed over
    // through the ring (lane-major, one word per lane and item: no bank conflicts)
    float *xch = (float *)ring + (size_t)wave * (21 * QB) * 64 + lane;
    constexpr int kGroup = WQ * 21 * QB * 64;   // words of one group
    static_assert((KS - 1) * kGroup * sizeof(float) <= STAGES * kSlotHalfs * sizeof(half_t), "the groups fit the ring");
    __syncthreads();           // every wave is done reading the ring
    if (grp > 0) {
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        float *to = xch + (grp - 1) * kGroup + qb * 21 * 64;
        to[20 * 64] = m_run[qb];
#pragma unroll
        for (int db = 0; db < 5; ++db)
#pragma unroll
          for (int r = 0; r < 4; ++r) to[(db * 4 + r) * 64] = o[db][qb][r];
      }
    }
    __syncthreads();
    if (grp > 0) return;
#pragma unroll
    for (int g = 0; g < KS - 1; ++g)
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        const float *from = xch + g * kGroup + qb * 21 * 64;
        const float m_other = from[20 * 64];
        const float m_new = fmaxf(m_run[qb], m_other);
        const float a_mine = fast_exp2((m_run[qb] - m_new) * cs);
        const float a_other = fast_exp2((m_other - m_new) * cs);
        m_run[qb] = m_new;
#pragma unroll
        for (int db = 0; db < 5; ++db)
#pragma unroll
          for (int r = 0; r < 4; ++r) o[db][qb][r] = o[db][qb][r] * a_mine + from[(db * 4 + r) * 64] * a_other;
      }
  }

  // O / (l + 1e-6) -> fp16, token-major [row][head*64 + d]
  const int H = p.heads * kHeadDim;
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const float inv = __builtin_amdgcn_rcpf(o[4][qb][0] + 1e-6f);
    const int q = q0 + (wave * QB + qb) * 16 + lq;
    if (q >= nq) continue;
    half_t *dst = p.out + (size_t)(row_start + q) * H + head * kHeadDim + 4 * lg;
#pragma unroll
    for (int db = 0; db < 4; ++db) {
      const float4_t v = o[db][qb] * inv;
      *(half4_t *)(dst + 16 * db) = half4_t{(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]};
    }
  }
}

template <int QB, int KIND, int STAGES, int KS = 1, int WQ = 4>
__global__ __launch_bounds__(64 * WQ * KS, KS == 2 && !KIND ? 4 : 2) void attention_grouped_kernel(BT_ATT_FIRST, AttTail<KIND> tail) {
  const AttArgs p = att_args<KIND>(BT_ATT_FIRST_NAMES, tail);
  __shared__ __attribute__((aligned(1024))) half_t ring[STAGES * KS * 2 * kTileHalfs];
  AttTile item;
  if (att_tile<16 * WQ * QB>(p, item)) attention_tile<QB, KIND, STAGES, KS, WQ>(p, item, ring);
  warm_slice<64 * WQ * KS>(p.warm);
}

// The balanced order of a launch of `entries` workgroups as a list: one wave per entry.
template <int BQ>
__global__ __launch_bounds__(kAttThreads) void attention_worklist_kernel(AttArgs p, int4 *list,
                                                                        unsigned entries) {
  const unsigned e = workgroup_id() * (kAttThreads / 64) + (thread_id() >> 6);
  if (e >= entries) return;
  const AttWork w = att_work_balanced<BQ>(p, e);
  if ((thread_id() & 63) == 0)
    list[e] = w.exists ? int4{w.b, w.head | (w.qb << 16), w.seq_start, w.len} : int4{-1, 0, 0, 0};
}

// ---------------------------------------------------------------------------
// short kernel: K, V resident in LDS, logits of the query tile in registers
// ---------------------------------------------------------------------------
template <int NKB, int KIND>  // capacity in 16-key blocks (keys <= 16*NKB), NKB even; KIND as above
__global__ __launch_bounds__(kAttThreads) void attention_short_kernel(AttArgs p) {
  constexpr bool ADD = KIND != kAddNone;
  constexpr int KEYS = NKB * 16;
  constexpr int BQ = 64;  // 4 waves x 16 queries
  extern __shared__ __attribute__((aligned(1024))) half_t att_smem[];
  half_t *sK = att_smem;                      // [KEYS][64] swizzled
  half_t *sV = att_smem + KEYS * kHeadDim;    // [KEYS][64] swizzled

  if (workgroup_id() >= p.warm.grid_work) {
    warm_slice<kAttThreads>(p.warm);
    return;
  }
  const AttItem item = att_item(p);
  if (!item.exists) {
    warm_slice<kAttThreads>(p.warm);
    return;
  }
  const int b = p.seq_order ? p.seq_order[item.rank] : item.rank, head = item.head;
  const int seq_start = p.batch_idx[b];
  const int klen = (KIND & kAddMask) || p.every_key ? p.S : p.batch_idx[b + 1] - seq_start;
  const int row_start = p.padded_rows ? b * p.S : seq_start;
  const int nq = p.padded_rows ? p.S : klen;
  const int q0 = item.qb * BQ;
  if (q0 >= nq) {
    warm_slice<kAttThreads>(p.warm);
    return;
  }

  const int tid = thread_id(), lane = tid & 63, wave = tid >> 6;
  const int lq = lane & 15, lg = lane >> 4;
  const int H = p.heads * kHeadDim;
  const int q = q0 + wave * 16 + lq;

  const size_t head_stride = (size_t)p.rows_cap * kHeadDim;
  const half_t *Q = p.qkv + (size_t)head * head_stride + (size_t)row_start * kHeadDim;
  const half_t *K = Q + (size_t)p.heads * head_stride;
  const half_t *V = K + (size_t)p.heads * head_stride;

  // copy K and V rows [0, keys32) into LDS, 8 rows per wave instruction
  const int keys32 = min(((klen + 31) >> 5) << 5, KEYS);
  if (klen > 0) {
    const int ld_row = lane >> 3, ld_slot = lane & 7;
    for (int g8 = wave; g8 < keys32 / 8; g8 += 4) {
      const int row = g8 * 8 + ld_row;
      const int key = min(row, klen - 1);
      lds_dma16(K + (size_t)key * kHeadDim + ((ld_slot ^ swz_k(row)) << 3),
                sK + g8 * 8 * kHeadDim);
      lds_dma16(V + (size_t)key * kHeadDim + ((ld_slot ^ swz_v(row)) << 3),
                sV + g8 * 8 * kHeadDim);
    }
  }
  half8_t qf[2];
#pragma unroll
  for (int dh = 0; dh < 2; ++dh) {
    uint4_t v = {0u, 0u, 0u, 0u};
    if (q < nq) v = *(const uint4_t *)(Q + (size_t)q * kHeadDim + 32 * dh + 8 * lg);
    qf[dh] = __builtin_bit_cast(half8_t, v);
  }
  att_wait_vmcnt<0>();
  asm volatile("" ::: "memory");
  __syncthreads();
  // no barrier follows: a wave whose 16 queries all lie past the sequence is done
  if (q0 + wave * 16 >= nq) {
    warm_slice<kAttThreads>(p.warm);
    return;
  }

  const int nkb = keys32 >> 4;  // even
  float4_t s[NKB];
#pragma unroll
  for (int kb = 0; kb < NKB; ++kb) {
    s[kb] = float4_t{0.f, 0.f, 0.f, 0.f};
    if (kb < nkb) {
#pragma unroll
      for (int dh = 0; dh < 2; ++dh)
        s[kb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(load_k_frag(sK, kb, dh, lq, lg), qf[dh],
                                                       s[kb], 0, 0, 0);
    }
  }

  const float c = p.scale_log2e;
  const float cs = ADD ? 1.0f : c;
  if (ADD) {
    const int qc = min(q, p.S - 1);
    const TermRow mrow(p.mask, (size_t)b * p.S + qc, p.S, (size_t)p.B * p.S);
    const TermRow brow(p.bias, (size_t)head * p.S + qc, p.S, (size_t)p.heads * p.S);
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) {
      const int key = kb * 16 + lg * 4;
      uint2_t mv = {0u, 0u}, bv = {0u, 0u};
      if (KIND & kAddMask) mv = mrow.in_order(mrow.fetch<false>(key), key);
      if (KIND & kAddBias) bv = brow.in_order(brow.fetch<false>(key), key);
      s[kb] = add_terms<KIND>(s[kb], c, mv, bv);
    }
  }
  // exact softmax over the row: mask by index, max, exp, sum, normalise, round
  float mx = kNegBig;
#pragma unroll
  for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (kb * 16 + lg * 4 + r >= klen) s[kb][r] = kNegBig;
      mx = fmaxf(mx, s[kb][r]);
    }
  mx = rows_max(mx);
  const float mc = mx * cs;
  float sum = 0.f;
#pragma unroll
  for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      s[kb][r] = fast_exp2(__builtin_fmaf(s[kb][r], cs, -mc));
      sum += s[kb][r];
    }
  sum = rows_sum(sum);
  const float inv = 1.0f / (sum + 1e-6f);

  float4_t o[4];
#pragma unroll
  for (int db = 0; db < 4; ++db) o[db] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kk = 0; kk < NKB / 2; ++kk) {
    if (2 * kk < nkb) {
      half8_t pf;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        pf[r] = (half_t)(s[2 * kk][r] * inv);
        pf[4 + r] = (half_t)(s[2 * kk + 1][r] * inv);
      }
#pragma unroll
      for (int db = 0; db < 4; ++db)
        o[db] = __builtin_amdgcn_mfma_f32_16x16x32_f16(load_vt_frag(sV, kk, db, lq, lg), pf, o[db],
                                                       0, 0, 0);
    }
  }

  if (q < nq) {
    half_t *dst_row = p.out + (size_t)(row_start + q) * H + head * kHeadDim + 4 * lg;
#pragma unroll
    for (int db = 0; db < 4; ++db)
      *(half4_t *)(dst_row + 16 * db) =
          half4_t{(half_t)o[db][0], (half_t)o[db][1], (half_t)o[db][2], (half_t)o[db][3]};
  }
  warm_slice<kAttThreads>(p.warm);
}

// Size of the 1-D grid for `nqb` query tiles per sequence; fills the mapping fields.
static unsigned att_grid(AttArgs &a, int nqb, bool streaming = false) {
  a.nqb = nqb;
  a.per_nqb = inverse_of(nqb), a.per_heads = inverse_of(a.heads);
  a.xcd_map = option_attention_xcd_map();
  const unsigned pairs = (unsigned)a.B * a.heads;
  // The balanced list is the streaming kernel's, and pays from the third round of 32
  // workgroups per XCD on: up to two rounds its look-up (vector loads and a wave scan
  // where the plain order needs three scalar loads) cost 0.3-1.5 % per forward.
  // Its look-up takes one pass (two dependent loads) per 64 sequences: beyond 128 the
  // plain order stays, and so many sequences even out by themselves.
  if (a.xcd_map == 2 && ((pairs + 7) / 8 * nqb <= 64 || a.B > 128)) a.xcd_map = 1;
  if (a.xcd_map == 3) a.xcd_map = 2;   // option value 3: the balanced list at any size
  if (a.xcd_map == 2 && !streaming) a.xcd_map = 1;
  if (a.xcd_map == 2) return ((pairs + 7) / 8 * nqb + 31) / 32 * 32 * 8;   // whole rounds of 32 per XCD
  return a.xcd_map ? (pairs + 7) / 8 * 8 * nqb : pairs * nqb;
}

static int check_att_args(const char *who, const void *qkv, const void *out, const int *batch_idx,
                          const void *mask, int padded_rows, int B, int S, int rows_cap,
                          int heads, int d) {
  BT_REQUIRE(!mask || padded_rows, BT_ERR_INVALID_ARGUMENT,
             "%s: atten_mask is only applied on padded rows (padded_rows != 0)", who);
  BT_REQUIRE(qkv && out && batch_idx, BT_ERR_INVALID_ARGUMENT, "%s: null pointer argument", who);
  BT_REQUIRE(aligned16({qkv, out, mask}), BT_ERR_INVALID_ARGUMENT,
             "%s: tensor pointers must be 16-byte aligned", who);
  BT_REQUIRE(B > 0 && S > 0 && heads > 0 && rows_cap > 0, BT_ERR_INVALID_ARGUMENT,
             "%s: batch_size=%d seq_len=%d head_num=%d rows_cap=%d must be positive", who, B, S,
             heads, rows_cap);
  BT_REQUIRE(d == kHeadDim, BT_ERR_UNSUPPORTED, "%s: size_per_head=%d, only 64 is supported", who,
             d);
  BT_REQUIRE(B <= 65535 && heads <= 65535, BT_ERR_UNSUPPORTED, "%s: grid too large", who);
  return BT_OK;
}

template <int NKB, int KIND>
static int launch_short_impl(const AttArgs &a, hipStream_t s) {
  constexpr size_t smem = (size_t)2 * NKB * 16 * kHeadDim * sizeof(half_t);
  static_assert(smem <= kMostLds, "LDS budget");
  return Launch<attention_short_kernel<NKB, KIND>>::on(s, "attention_short_kernel", a.nqb_grid, kAttThreads, smem, a);
}

template <int NKB>
static int launch_short(const AttArgs &a, hipStream_t s) {
  switch (add_kind(a.mask, a.bias, a.scale_log2e)) {
    case kAddNone: return launch_short_impl<NKB, kAddNone>(a, s);
    case kAddMask: return launch_short_impl<NKB, kAddMask>(a, s);
    case kAddBias: return launch_short_impl<NKB, kAddBias>(a, s);
    case kAddZero: return launch_short_impl<NKB, kAddZero>(a, s);
    default: return launch_short_impl<NKB, kAddBoth>(a, s);
  }
}

}  // namespace bt

using namespace bt;

extern "C" int bt_attention_short(const void *qkv_heads, void *attention_output,
                                  const int *batch_idx, const int *seq_order,
                                  const void *atten_mask, const void *attention_bias,
                                  int batch_size, int seq_len, int rows_cap, int head_num,
                                  int size_per_head, float scale, int padded_rows,
                                  const void *const *prefetch,
                                  const unsigned long long *prefetch_bytes, int prefetch_count,
                                  void *stream) {
  int rc = check_att_args("bt_attention_short", qkv_heads, attention_output, batch_idx, atten_mask,
                          padded_rows, batch_size, seq_len, rows_cap, head_num, size_per_head);
  if (rc) return rc;
  BT_REQUIRE(seq_len <= 512, BT_ERR_UNSUPPORTED,
             "bt_attention_short: seq_len=%d exceeds 512, use bt_attention_grouped", seq_len);
  AttArgs a{(const half_t *)qkv_heads, (half_t *)attention_output, batch_idx, seq_order,
            (const half_t *)atten_mask, (const half_t *)attention_bias,
            {}, batch_size, seq_len,
            rows_cap, head_num, scale * kLog2e, padded_rows};
  a.every_key = drop_terms_of_one_key(seq_len, a.mask, a.bias);
  hipStream_t s = as_stream(stream);
  a.nqb_grid = att_grid(a, (seq_len + 63) / 64);
  rc = plan_warm_duty("bt_attention_short", a.warm, a.nqb_grid, prefetch, prefetch_bytes, prefetch_count);
  if (rc) return rc;
  if (seq_len <= 64) return launch_short<4>(a, s);
  if (seq_len <= 128) return launch_short<8>(a, s);
  if (seq_len <= 256) return launch_short<16>(a, s);
  if (seq_len <= 384) return launch_short<24>(a, s);
  return launch_short<32>(a, s);
}

namespace bt {
// Shape of a streaming-attention launch: 128-query tiles with a three-deep ring once there
// is plenty of work (three workgroups per CU); else 64-query tiles with a two-deep ring: 32 KB
// of LDS and ~100 registers let four workgroups share a CU (a build held to 84 registers fits
// five and measures the same), which hides more of the per-tile dependency chain than the
// third stage did (-0.1 to -2.8 % per forward from batch 1 x 256 to batch 16 x 384; with the
// balanced work list also -0.8 to -1.9 % at batch 32 x 256 / 384 and 16 x 768, so the switch
// sits at 1300 workgroups of 128 queries; batch 16 x 512 is within 0.3 % either way).
// 16-query tiles whose waves share the keys for sequences of 65 to 256 tokens, while a launch of them leaves
// CUs to the warm-up.
struct GroupedPlan {
  bool wide;        // 128-query tiles
  bool narrow;      // 16-query tiles
  unsigned grid;
};
constexpr long long kNarrowBlocks = 208;
// Two or three key tiles leave waves without keys and fewer turns to save, so it has to be fewer workgroups there; so it
// has where the three weights to warm up fill the 12 MB that a launch takes on (hidden 816 and more), since every
// workgroup beyond 160 takes one from the warm-up.  Whole forwards, 64-query against 16-query tiles, us, operator /
// graph (full, 60 % full): 12 heads, 12 layers, at 1 x 128 (96 workgroups of 16 queries) 378 374 / 368 368, 369 367;
// 2 x 96 (144) 387 381; 1 x 180 (144) 398 387 / 394 386, 385 387; 2 x 120 (192) 393 392; 1 x 256 (192) 414 395 / 413 396,
// 405 396; 16 heads, 24 layers, at 1 x 128 (128) 938 929; 1 x 160 (160) 995 968; 2 x 96 (192) 1030 1073 / 920 951, 904 949;
// 1 x 190 (192) 1060 1083 / 934 955, 917 953; 1 x 200 (208) 1035 1041 / 951 955, 916 951; 1 x 256 (256) 1094 1103.
constexpr long long kNarrowBlocksFew = 160;
constexpr int kNarrowHidden = 816;
static GroupedPlan plan_grouped(AttArgs &a, int batch_size, int seq_len, int head_num) {
  const long long blocks128 = (long long)((seq_len + 127) / 128) * head_num * batch_size;
  const int qb = option_attention_qb();
  GroupedPlan plan;
  plan.wide = qb == 2 || (qb < 0 && blocks128 >= 1300);
  const long long blocks16 = (long long)((seq_len + 15) / 16) * head_num * batch_size;
  const long long most = seq_len > 3 * kKT && head_num * kHeadDim < kNarrowHidden ? kNarrowBlocks : kNarrowBlocksFew;
  plan.narrow = qb < 0 && option_attention_key_split() < 0 && option_attention_xcd_map() != 3 && seq_len > kKT &&
                seq_len <= 4 * kKT && blocks16 <= most && cu_count() == 256;
  plan.grid = att_grid(a, plan.wide ? (seq_len + 127) / 128 : plan.narrow ? (seq_len + 15) / 16 : (seq_len + 63) / 64,
                       true);
  return plan;
}
template <int KIND>
static int launch_grouped(const AttArgs &a, const GroupedPlan &plan, int seq_len, unsigned grid, hipStream_t s) {
  // (the additive terms alternate between two register sets, so their kernels take an even ring)
  constexpr int kWideStages = KIND == kAddNone ? 3 : 2;
  // eight waves over two key halves: pays for a few long sequences that leave most CUs
  // with one workgroup or none (batch 1 x 1024: 9.9 -> 8.7 us); with several workgroups
  // per CU the four-wave form is faster (batch 16 x 512: 16.3 against 19.6 us).  Decided by the
  // workgroups of the attention itself: those that a warm-up hint adds leave the sums as they are.
  const int ks = option_attention_key_split();
  const AttFirst f = att_first(a);
  const AttTail<KIND> t = att_tail<KIND>(a);
  const char *who = "attention_grouped_kernel";
  if (plan.narrow)
    return Launch<attention_grouped_kernel<1, KIND, 1, 4, 1>>::on(s, who, grid, kAttThreads, 0, BT_ATT_FIRST_OF(f), t);
  if (plan.wide)
    return Launch<attention_grouped_kernel<2, KIND, kWideStages, 1, 4>>::on(s, who, grid, kAttThreads, 0, BT_ATT_FIRST_OF(f), t);
  if (ks == 1 || (ks < 0 && seq_len >= 512 && a.warm.grid_work <= 256))
    return Launch<attention_grouped_kernel<1, KIND, 2, 2, 4>>::on(s, who, grid, 2 * kAttThreads, 0, BT_ATT_FIRST_OF(f), t);
  return Launch<attention_grouped_kernel<1, KIND, 2, 1, 4>>::on(s, who, grid, kAttThreads, 0, BT_ATT_FIRST_OF(f), t);
}
AttListPlan att_worklist_plan(int B, int S, int heads) {
  AttListPlan out{0, 64, 0};
  if (B <= 0 || S <= 0 || heads <= 0) return out;
  AttArgs a{};
  a.B = B, a.S = S, a.heads = heads;
  const GroupedPlan plan = plan_grouped(a, B, S, heads);
  out.bq = plan.wide ? 128 : 64;
  out.nqb = a.nqb;
  out.entries = a.xcd_map == 2 ? plan.grid : 0;
  return out;
}
}  // namespace bt

extern "C" unsigned long long bt_attention_worklist_bytes(int batch_size, int seq_len,
                                                          int head_num) {
  return (unsigned long long)att_worklist_plan(batch_size, seq_len, head_num).entries *
         sizeof(int4);
}

extern "C" int bt_attention_worklist(const int *batch_idx, const int *seq_order, int batch_size,
                                     int seq_len, int head_num, int padded_rows, void *work_list,
                                     void *stream) {
  BT_REQUIRE(batch_idx && work_list, BT_ERR_INVALID_ARGUMENT,
             "bt_attention_worklist: null pointer argument");
  BT_REQUIRE(batch_size > 0 && seq_len > 0 && head_num > 0, BT_ERR_INVALID_ARGUMENT,
             "bt_attention_worklist: sizes must be positive");
  BT_REQUIRE(aligned16({work_list}), BT_ERR_INVALID_ARGUMENT,
             "bt_attention_worklist: work_list must be 16-byte aligned");
  AttArgs a{};
  a.batch_idx = batch_idx, a.seq_order = seq_order;
  a.B = batch_size, a.S = seq_len, a.heads = head_num, a.padded_rows = padded_rows;
  const GroupedPlan plan = plan_grouped(a, batch_size, seq_len, head_num);
  BT_REQUIRE(a.xcd_map == 2, BT_ERR_INVALID_ARGUMENT,
             "bt_attention_worklist: launches of this shape take no work list "
             "(bt_attention_worklist_bytes is 0)");
  const unsigned blocks = (plan.grid + kAttThreads / 64 - 1) / (kAttThreads / 64);
  if (plan.wide)
    attention_worklist_kernel<128><<<blocks, kAttThreads, 0, as_stream(stream)>>>(
        a, (int4 *)work_list, plan.grid);
  else
    attention_worklist_kernel<64><<<blocks, kAttThreads, 0, as_stream(stream)>>>(
        a, (int4 *)work_list, plan.grid);
  BT_CHECK_LAUNCH("attention_worklist_kernel");
  return BT_OK;
}

extern "C" int bt_attention_grouped(const void *qkv_heads, void *attention_output,
                                    const int *batch_idx, const int *seq_order,
                                    const void *atten_mask, const void *attention_bias,
                                    int batch_size, int seq_len, int rows_cap, int head_num,
                                    int size_per_head, float scale, int padded_rows,
                                    const void *const *prefetch,
                                    const unsigned long long *prefetch_bytes, int prefetch_count,
                                    const int *mask_prefix_slots, const void *work_list,
                                    void *stream) {
  // without offsets: only where nothing would read them (padded rows, the mask tensor
  // applied element by element, no verdict that could drop it, no balanced order)
  const bool no_offsets = !batch_idx && padded_rows && atten_mask && !mask_prefix_slots;
  int rc = check_att_args("bt_attention_grouped", qkv_heads, attention_output,
                          no_offsets ? (const int *)qkv_heads : batch_idx, atten_mask,
                          padded_rows, batch_size, seq_len, rows_cap, head_num, size_per_head);
  if (rc) return rc;
  BT_REQUIRE(aligned16({work_list}), BT_ERR_INVALID_ARGUMENT,
             "bt_attention_grouped: work_list must be 16-byte aligned");
  if (no_offsets) seq_order = nullptr;
  AttArgs a{(const half_t *)qkv_heads, (half_t *)attention_output, batch_idx, seq_order,
            (const half_t *)atten_mask, (const half_t *)attention_bias,
            {}, batch_size, seq_len,
            rows_cap, head_num, scale * kLog2e, padded_rows};
  a.every_key = drop_terms_of_one_key(seq_len, a.mask, a.bias);
  a.mask_ok = a.mask ? mask_prefix_slots : nullptr;
  a.work_list = (const int4 *)work_list;   // read only when the launch uses the balanced order
  hipStream_t s = as_stream(stream);
  GroupedPlan plan = plan_grouped(a, batch_size, seq_len, head_num);
  if (no_offsets && a.xcd_map == 2) {   // the balanced order ranks the sequences by length
    a.xcd_map = 1;
    plan.grid = ((unsigned)batch_size * head_num + 7) / 8 * 8 * a.nqb;
  }
  unsigned grid = plan.grid;
  rc = plan_warm_duty("bt_attention_grouped", a.warm, grid, prefetch, prefetch_bytes, prefetch_count);
  if (rc) return rc;
  switch (add_kind(a.mask, a.bias, a.scale_log2e)) {
    case kAddNone: return launch_grouped<kAddNone>(a, plan, seq_len, grid, s);
    case kAddMask: return launch_grouped<kAddMask>(a, plan, seq_len, grid, s);
    case kAddBias: return launch_grouped<kAddBias>(a, plan, seq_len, grid, s);
    case kAddZero: return launch_grouped<kAddZero>(a, plan, seq_len, grid, s);
    default: return launch_grouped<kAddBoth>(a, plan, seq_len, grid, s);
  }
}
