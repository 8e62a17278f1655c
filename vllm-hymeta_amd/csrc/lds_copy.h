// Copies from global memory into LDS that do not pass registers.
#pragma once

#include "common.h"

namespace hymeta {
namespace {

// 16 bytes per lane from global memory into LDS at (wave-uniform) dst + 16 lane, without passing registers.  asm
// statements, their completion counted by hand: the compiler books such a load on the LDS counter as well and would turn
// every wait for a fragment read into a wait for all of them.
__device__ __forceinline__ uint32_t lds_address(char* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)p));
}
__device__ __forceinline__ void copy16_to_lds(const char* src, char* dst) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds_address(dst)), "v"(src) : "memory");
}
// The same from a wave-uniform base and a 32-bit offset per lane.
__device__ __forceinline__ void copy16_to_lds(const char* base, uint32_t offset, char* dst) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_address(dst)), "v"(offset), "s"(base) : "memory");
}
// Until everything this wave has asked for has landed and every wave of the workgroup has got here with its reads and
// writes of LDS done.
__device__ __forceinline__ void copies_landed_barrier() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

}  // namespace
}  // namespace hymeta
