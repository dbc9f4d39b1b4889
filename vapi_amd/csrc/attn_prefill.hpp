// Pieces shared by the prefill kernels that stage K and V in LDS by direct
// global-to-LDS loads (attn_prefill.hip, attn_prefill_f32.hip).
#pragma once

#include "attn_common.hpp"

namespace vk {

using LdsVoid = __attribute__((address_space(3))) void;


// The XOR swizzle of key row r's 16-byte chunks. D = 128 (16 chunks, a row
// is 256 bytes: every row starts at bank 0): the row index rotated left by
// one bit, a bijection on 0..15, so the 16 rows a K fragment read touches
// use 16 distinct chunk positions for any chunk, and the 8 rows of one
// half-wave of a transposing V read (rows 0..7 or 8..15, chunks 2t, 2t + 1)
// use 8 distinct chunk pairs (XOR with r alone puts rows 2m and 2m + 1 on
// the same pair). Measured 0.5-1% faster than XOR with r; the bank-conflict
// counter reads the same either way (2 cycles per transposing read).
// D = 256 (32 chunks, 512-byte rows): the same rotation, XORed into the
// low four bits of the chunk index (chunks p and p ^ 16 share banks).
// D = 64: r mod 8.
template <int D>
__device__ __forceinline__ uint32_t pf_swz(uint32_t r) {
  if constexpr (D >= 128) {
    const uint32_t x = r & 15;
    return ((x << 1) | (x >> 3)) & 15;
  } else {
    return r & (D / 8 - 1);
  }
}

// Element offset of 16-byte chunk p of key row r (0..31) in a step buffer.
template <int D>
__device__ __forceinline__ uint32_t pf_chunk(uint32_t r, uint32_t p) {
  constexpr uint32_t CPR = D / 8;  // chunks per row
  return (r * CPR + (p ^ pf_swz<D>(r))) * 8;
}

// Waits until at most n of this wave's vector memory loads are in flight
// (s_waitcnt: vmcnt in bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8). The
// ring's waits count only its own direct loads, which holds while the
// kernel uses no scratch (vapi_amd/build.py refuses a build where it does).
template <int n>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(n >= 0 && n < 16, "vmcnt immediate");
  __builtin_amdgcn_s_waitcnt(n | (0x7 << 4) | (0xF << 8));
}

// The workgroup barrier of the ring: this wave's loads of the next step
// have landed (the caller's wait_vmcnt), then s_barrier alone. A
// __syncthreads() would add a release fence, which waits for every load
// in flight into LDS, including the step issued two ahead.
__device__ __forceinline__ void ring_barrier() {
  __asm__ volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  __asm__ volatile("" ::: "memory");
}

__device__ __forceinline__ uint32_t lds_addr(const uint16_t* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint16_t*)p;
}

}  // namespace vk
