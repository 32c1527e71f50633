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
// Two such loads by one descriptor and step, to two places: the wait states ahead of both once, and between them m0 written and the one
// state behind that.  m0 is written before the second load reads step, descriptor and offset: early (&), or a step that equals lds0 is read
// out of it.  us of products, a load at a time and in pairs: 64 experts of 2,816 x 2,048, six picks, 1,664 tokens 197 -> 192; 28 of 2,048 x
// 4,096, 2,048 tokens 216 -> 211; 16 of 5,120 x 8,192, 8,192 tokens 671 -> 666.  Prompt attention is as fast either way (128 wide, 2,048 tokens
// 100.2 and 100.6, 4,096 behind 4,096 875 and 877, 1,900 in a window 60.1 and 60.7; 192 wide 122.5 and 121.1; 64 wide 95.0 and 94.4).
template <bool STREAM = false>
__device__ __forceinline__ void load_two_to_lds(u32x4 rsrc, uint32_t offset0, uint32_t offset1, uint32_t step, uint32_t lds0, uint32_t lds1) {
  lds0 = __builtin_amdgcn_readfirstlane(lds0);
  lds1 = __builtin_amdgcn_readfirstlane(lds1);
  step = __builtin_amdgcn_readfirstlane(step);
  if constexpr (STREAM)
    asm volatile("s_nop 4\n\tbuffer_load_dwordx4 %1, %3, %4 offen nt lds\n\ts_mov_b32 m0, %5\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, %4 offen nt lds"
                 : "+&{m0}"(lds0) : "v"(offset0), "v"(offset1), "s"(rsrc), "s"(step), "s"(lds1) : "memory");
  else
    asm volatile("s_nop 4\n\tbuffer_load_dwordx4 %1, %3, %4 offen lds\n\ts_mov_b32 m0, %5\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, %4 offen lds"
                 : "+&{m0}"(lds0) : "v"(offset0), "v"(offset1), "s"(rsrc), "s"(step), "s"(lds1) : "memory");
}
// The same bytes by way of registers, from any address.
__device__ __forceinline__ void copy_to_lds(u32x4 rsrc, uint32_t offset, uint32_t step, uint32_t lds) {
  const char* base = (const char*)((uint64_t)rsrc[0] | (uint64_t)rsrc[1] << 32);
  u32x4 piece;
  __builtin_memcpy(&piece, base + (size_t)step + offset, 16);
  *(__attribute__((address_space(3))) u32x4*)(uintptr_t)(lds + (threadIdx.x & (kWave - 1)) * 16) = piece;
}
// Loads 0 .. N - 1 of one descriptor and step, in pairs.
template <bool DIRECT, int N, bool STREAM = false>
__device__ __forceinline__ void bring_all_to_lds(u32x4 rsrc, const uint32_t (&offset)[N], uint32_t step, const uint32_t (&lds)[N]) {
#pragma unroll
  for (int i = 0; i < N; i += 2) {
    const int j = i + 1 < N ? i + 1 : i;
    if (DIRECT && j > i) load_two_to_lds<STREAM>(rsrc, offset[i], offset[j], step, lds[i], lds[j]);
    else {
      if constexpr (DIRECT) load_to_lds<STREAM>(rsrc, offset[i], step, lds[i]);
      else {
        copy_to_lds(rsrc, offset[i], step, lds[i]);
        if (j > i) copy_to_lds(rsrc, offset[j], step, lds[j]);
      }
    }
  }
}
template <int LEFT = 0> __device__ __forceinline__ void lds_loads_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LEFT) : "memory");
}
