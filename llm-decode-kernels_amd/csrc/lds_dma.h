// 16-byte buffer loads straight to LDS and the explicit waits and barriers that order them, shared
// by the kernels that keep a ring of LDS stages in flight (prefill.hip, attention.hip).
#pragma once

#include "ldk_common.h"

namespace ldk {

// s_waitcnt vmcnt(N): at most N vector-memory loads of this wave still outstanding. Loads complete
// in issue order for this count, so it waits for every load issued before the last N. The builtin
// (gfx9 encoding: vmcnt in bits 3:0 and 15:14, expcnt and lgkmcnt left open) is what the
// compiler's own wait insertion reads, so it knows the older stages are complete and adds no wait
// of its own before their LDS reads; the empty asm with a memory clobber on each side keeps the
// compiler from moving any load or LDS access across it, which the count relies on.
template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("" : : : "memory");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
  asm volatile("" : : : "memory");
}

// Workgroup barrier that is also a compiler memory barrier, without the vmcnt(0) a C++ fence adds
// (the ring keeps later stages' loads in flight across it).
__device__ __forceinline__ void ring_barrier() {
  asm volatile("" : : : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" : : : "memory");
}

// 16-byte buffer loads to LDS (lane i writes lds_base + 16 i), issued as inline asm: the
// compiler's wait insertion then does not track them, so it adds no conservative vmcnt wait before
// the LDS reads of other stages (it would after the loop's back edge, where it no longer knows
// which LDS array each pending load writes); the ring's own vmcnt waits order them. M0 holds the
// LDS base for the load; the asm restores M0's previous value itself (M0 is reserved to the
// compiler, which does not save a clobbered M0). An LDS DMA that reads M0 right after an SALU
// write of it needs one wait state on gfx9-family chips (gfx950 included); the compiler's hazard
// recognizer inserts it for its own M0 writes but cannot see inside this asm string, so the string
// carries its own s_nop 0. The address is base + voffset + soffset; only
// voffset is checked against the
// resource's size, so every load that relies on the check (x rows past M, scales past N) keeps
// its whole offset in voffset, and soffset carries only the uniform K-step offset of loads that
// stay inside their arrays.
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}
__device__ __forceinline__ void dma_buffer16(u32x4 rsrc, uint32_t voffset, uint32_t soffset, uint32_t lds_base) {
  uint32_t saved;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %4 offen lds\n\ts_mov_b32 m0, %0"
               : "=&s"(saved)
               : "v"(voffset), "s"(rsrc), "s"(lds_base), "s"(soffset)
               : "memory");
}
// The same with 4 bytes per lane (lane i writes lds_base + 4 i), for rows only 4-byte aligned.
__device__ __forceinline__ void dma_buffer4(u32x4 rsrc, uint32_t voffset, uint32_t soffset, uint32_t lds_base) {
  uint32_t saved;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %4 offen lds\n\ts_mov_b32 m0, %0"
               : "=&s"(saved)
               : "v"(voffset), "s"(rsrc), "s"(lds_base), "s"(soffset)
               : "memory");
}
// Raw buffer descriptor over [p, p + bytes): a load at an offset past it returns zeros (and, to
// LDS, writes zeros).
__device__ __forceinline__ u32x4 raw_rsrc(const void* p, uint32_t bytes) {
  const uint64_t a = (uint64_t)(uintptr_t)p;
  return u32x4{(uint32_t)a, (uint32_t)(a >> 32) & 0xffffu, bytes, 0x00020000u};
}
// The same from a uniform address the compiler may have formed in vector registers.
__device__ __forceinline__ u32x4 raw_rsrc_uniform(const void* p, uint32_t bytes) {
  u32x4 r = raw_rsrc(p, bytes);
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = __builtin_amdgcn_readfirstlane(r[i]);
  return r;
}

}  // namespace ldk
