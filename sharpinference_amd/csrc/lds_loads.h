// Loads from memory straight into LDS, 16 bytes a lane, for kernels that stage tiles without holding them in registers.
// The compiler does not know of them: it neither waits for them nor counts them.  A kernel waits with lds_loads_wait, by the
// number of the wave's own loads that may still be under way (loads return in order; loads of the compiler's own in between only
// make such a wait longer), and makes the data everyone's with a barrier behind it.  Loads of the compiler's own whose first
// use lies among these are to be forced beforehand (an empty asm statement that takes the value), or their wait would
// take in these as well.
#pragma once
#include "common.h"

typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

// Operands of such loads begin at 16-byte addresses; of others the pieces go through registers (DIRECT false), by kernels compiled apart:
// a branch at the loads made the products 4 to 6 % slower and prompt attention 7.
inline bool whole_pieces(const void* a, const void* b) { return (((uintptr_t)a | (uintptr_t)b) & 15) == 0; }
// `bytes` of memory from `base` on, as the descriptor buffer loads take: lanes whose offset lies at or beyond them read zeros.
__device__ __forceinline__ u32x4 buffer_of(const void* base, uint32_t bytes) {
  const uint64_t a = (uint64_t)base;
  return u32x4{(uint32_t)a, (uint32_t)(a >> 32) & 0xffffu, bytes, 0x00020000u};
}
__device__ __forceinline__ uint32_t lds_address(const char* p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)p;
}
// Lane l's 16 bytes at offset + step (step and lds the same for all lanes) go to LDS byte lds + 16 l (the instruction takes the LDS
// address from m0: an operand, so that the compiler knows what m0 holds).  STREAM: with the streaming hint, for data that nobody else
// reads.  The compiler keeps dependent instructions apart where the hardware does not, but does not look inside the statement.  Two
// such distances end at this load: five wait states from a vector instruction that writes a scalar register (readfirstlane, or a
// spilled scalar read back from a lane) to a memory instruction that reads it as descriptor or step, and one from a write of m0.
// s_nop 4 is five.
template <bool STREAM = false>
__device__ __forceinline__ void load_to_lds(u32x4 rsrc, uint32_t offset, uint32_t step, uint32_t lds) {
  lds = __builtin_amdgcn_readfirstlane(lds);
  step = __builtin_amdgcn_readfirstlane(step);
  if constexpr (STREAM)
    asm volatile("s_nop 4\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds" ::"{m0}"(lds), "v"(offset), "s"(rsrc), "s"(step) : "memory");
  else
    asm volatile("s_nop 4\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"{m0}"(lds), "v"(offset), "s"(rsrc), "s"(step) : "memory");
}
// The same bytes by way of registers, from any address.
__device__ __forceinline__ void copy_to_lds(u32x4 rsrc, uint32_t offset, uint32_t step, uint32_t lds) {
  const char* base = (const char*)((uint64_t)rsrc[0] | (uint64_t)rsrc[1] << 32);
  u32x4 piece;
  __builtin_memcpy(&piece, base + (size_t)step + offset, 16);
  *(__attribute__((address_space(3))) u32x4*)(uintptr_t)(lds + (threadIdx.x & (kWave - 1)) * 16) = piece;
}
template <bool DIRECT> __device__ __forceinline__ void bring_to_lds(u32x4 rsrc, uint32_t offset, uint32_t step, uint32_t lds) {
  if constexpr (DIRECT) load_to_lds(rsrc, offset, step, lds);
  else copy_to_lds(rsrc, offset, step, lds);
}
template <int LEFT = 0> __device__ __forceinline__ void lds_loads_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LEFT) : "memory");
}
