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

#endif  // __HIP_DEVICE_COMPILE__

}  // namespace bt
