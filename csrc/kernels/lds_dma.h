// LDS-DMA of 1-KiB pieces, for kernels that count what is in flight themselves; through descriptors in scalar registers
// nothing of an address is left to the lanes but a constant offset each, and what is out of a descriptor's range lands as
// zeros. The requests are inline asm: behind the builtins hipcc waits for every LDS-DMA in flight ahead of a transposing LDS
// read, the youngest tile's among them (s_waitcnt vmcnt(0) in the middle of a tile). They have no result; what they have written is
// read behind counted waits and a barrier.
#pragma once
#include "common.h"

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;

// a value that is the same in all lanes, in a scalar register
__device__ __forceinline__ uint32_t scalar(uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); }

// the descriptor of `bytes` bytes from `first` on
__device__ __forceinline__ u32x4 bytes_at(uintptr_t first, int bytes) {
  return {scalar((uint32_t)first), scalar((uint32_t)(first >> 32) & 0xffff), scalar((uint32_t)bytes), 0x00020000};
}
__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return (uint32_t)(uintptr_t)(lds_void*)const_cast<void*>(p);
}
// 16 bytes a lane to the 1 KiB at `to`. The wait states are those of a vector instruction that wrote a scalar
__device__ __forceinline__ void dma_piece(uint32_t to, int voff, const u32x4 rsrc) {
  const uint32_t m = scalar(to);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
               :: "s"(m), "v"(voff), "s"(rsrc) : "memory", "m0");
}
// the same from an address of each lane's own
__device__ __forceinline__ void dma_lanes(uint32_t to, const void* from) {
  const uint32_t m = scalar(to);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" :: "s"(m), "v"(from) : "memory", "m0");
}
