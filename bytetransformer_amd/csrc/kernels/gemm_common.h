// What the products of both precisions share: the LDS image of a k-step, counted waits, buffer descriptors.
#pragma once
#include "common.h"

namespace bt {

constexpr int kBK = 64;   // k extent of one LDS tile (halfs) = 8 chunks of 16 bytes
constexpr int kSchedMfma = 0x008, kSchedLdsRead = 0x100;   // instruction classes of sched_group_barrier

// XOR swizzle of the 16-byte chunk slot inside a 128-byte tile row: rows r and r+1
// differ by half of the 256-byte bank window, so 16 consecutive rows need 8 distinct
// slots.  The 16 lanes that one ds_read_b128 pass serves then touch every bank once.
__device__ __forceinline__ int swz(int row) { return (row >> 1) & 7; }

__device__ __forceinline__ float gelu_tanh_f32(float x) {
  // 0.5 x (1 + tanh(u)) == x / (1 + exp(-2u)),  u = 0.79788456 (x + 0.044715 x^3)
  // exponent folded into one polynomial: -2 u log2(e) = x (c1 + c3 x^2)
  constexpr float c1 = -2.0f * 0.7978845608028654f * 1.4426950408889634f;
  constexpr float c3 = c1 * 0.044715f;
  const float e = __builtin_amdgcn_exp2f(x * (c1 + c3 * x * x));
  return x * __builtin_amdgcn_rcpf(1.0f + e);
}

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  // s_waitcnt immediate on gfx9: vmcnt[3:0], expcnt[6:4], lgkmcnt[11:8], vmcnt[5:4] in [15:14]
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0F70);
}

// Wait until at most `younger` whole stages (NI loads each) are still in flight.
template <int NI, int MAXY>
__device__ __forceinline__ void wait_stages(int younger) {
  if constexpr (MAXY == 0) {
    wait_vmcnt<0>();
  } else {
    if (younger >= MAXY)
      wait_vmcnt<MAXY * NI>();
    else
      wait_stages<NI, MAXY - 1>(younger);
  }
}

// A [K, N] weight tile sits in LDS as 64 k-rows of BN halfs and is read with the LDS
// transpose read: the 32 lanes of one pass fetch 32 bytes of each of the k-rows r .. r + 3 and
// r + 8 .. r + 11.  Rows are BN / 32 segments of 64 bytes long; with a multiple of four segments
// per row the four rows start on the same bank and the segment is XORed with row & 3, with an odd
// multiple of two (BN = 64, 192) rows r and r + 2 do and bit 0 of the segment is XORed with bit 1 of
// the row; bit 3 of the row picks the half of the segment, which parts row r from row r + 8.
// Returned in 16-byte chunks (the unit a loading lane moves).
template <int BN>
__device__ __forceinline__ int swz_kn(int k_row) {
  static_assert(BN == 32 || BN % 64 == 0, "whole 64-byte segment pairs");
  if (BN == 32) return 0;   // gemm_wave_k: four k-rows are 256 contiguous bytes
  const int half = ((k_row >> 3) & 1) << 1;
  return ((BN / 32) % 4 == 0 ? (k_row & 3) << 2 : ((k_row >> 1) & 1) << 2) | half;
}

// The buffer-descriptor type exists in the device pass only; the host pass sees the
// kernel as an empty stub.
#if defined(__HIP_DEVICE_COMPILE__)
// Untyped buffer descriptor (stride 0) over [base, base + bytes): loads past the end
// return 0.
typedef __amdgpu_buffer_rsrc_t rsrc_t;
__device__ __forceinline__ rsrc_t make_rsrc(const void *base, size_t bytes) {
  const int recs = bytes > 0x7fffffffull ? 0x7fffffff : (int)bytes;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, recs, 0x00020000);
}

// Byte offset, from the first element of a [K, N] weight tile (k-step 0, first column of
// the tile), of the 16 bytes that a loading lane moves with the load that fills bytes
// [1024 g, 1024 g + 1024) of the tile's LDS image; the tile has `cols` columns inside the
// matrix, and chunks past them get an offset outside every descriptor (they read as zero).
template <int BN>
__device__ __forceinline__ int kn_load_offset(int g, int lane, int N, int cols) {
  constexpr int CPR = BN / 8;                       // 16-byte chunks per k-row
  const int slot = g * 64 + lane;
  const int k_row = slot / CPR, c = (slot % CPR) ^ swz_kn<BN>(k_row);
  return c * 8 < cols ? (k_row * N + c * 8) * (int)sizeof(half_t) : 0x7ffffff0;
}

// Weight operand of one 16x16x32 MFMA (16 columns from n_base, 32 k-rows from k_base) out
// of the LDS image of a [K, N] tile: lane l holds column n_base + (l & 15) at k-rows
// k_base + 8 (l >> 4) .. + 7, gathered by two transpose reads of 4 k-rows x 16 columns per
// 16 lanes.
template <int BN>
__device__ __forceinline__ half8_t load_kn_frag(const half_t *sW, int n_base, int k_base, int lane) {
  const int lq = lane & 15;
  const int k_row = k_base + 8 * (lane >> 4) + (lq >> 2);
  const int col = n_base + 4 * (lq & 3);
  const half_t *p0 = sW + k_row * BN + (((col >> 3) ^ swz_kn<BN>(k_row)) << 3) + (col & 7);
  const fp16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4f16(
      (__attribute__((address_space(3))) fp16x4_t *)p0);
  const fp16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4f16(
      (__attribute__((address_space(3))) fp16x4_t *)(p0 + 4 * BN));   // rows + 4: same swizzle term
  const half4_t l4 = __builtin_bit_cast(half4_t, lo), h4 = __builtin_bit_cast(half4_t, hi);
  return half8_t{l4[0], l4[1], l4[2], l4[3], h4[0], h4[1], h4[2], h4[3]};
}
#endif  // __HIP_DEVICE_COMPILE__

// Whether a product of these sizes, other than a plain one, adds up as tile 14 does (gemm_wave_k), or in one chain over k.
bool product_takes_wave_k(int rows_cap, int n, int k);

}  // namespace bt
