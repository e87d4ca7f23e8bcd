// Loads from memory straight to LDS, and the waits of a ring of LDS buffers filled by them.
#pragma once
#include "common.h"

namespace adamah {

// 16 bytes a lane from memory straight to LDS, lane l's to byte `lds` + 16 l.  Written out because the compiler, which
// cannot tell the buffers of a ring apart, waits for every such load in flight before it reads LDS (two buffers then hide
// nothing: 2048 x 28672 x 4096 took 600 us).  No register is loaded, so there is none to wait for: `ring_wait` stands
// ahead of the reads of the bytes.  M0 is set by every such load and declared overwritten (the warning that the compiler
// reserves it is off: nothing relies on its being kept).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void load_to_lds(const void* p, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(p) : "memory", "m0");
}
// the same of bytes that are read once: first to leave the L2 again
__device__ __forceinline__ void load_to_lds_once(const void* p, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt" ::"s"(lds), "v"(p) : "memory", "m0");
}
// the same from a base all lanes share and an offset of each; 4 bytes a lane
__device__ __forceinline__ void load_to_lds(const void* base, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory", "m0");
}
// the same, or nothing (the same for all lanes)
__device__ __forceinline__ void load_to_lds_unless(uint32_t skip, const void* base, uint32_t off, uint32_t lds) {
  asm volatile("s_cmp_lg_u32 %3, 0\n\ts_cbranch_scc1 .Lskip%=\n\ts_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n.Lskip%=:"
               ::"s"(lds), "v"(off), "s"(base), "s"(__builtin_amdgcn_readfirstlane((int)skip)) : "memory", "m0", "scc");
}
__device__ __forceinline__ void load4_to_lds(const void* base, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory", "m0");
}
#pragma clang diagnostic pop
__device__ __forceinline__ uint32_t lds_byte(const void* p) { return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p; }
// all but the last N loads of this wave have arrived and its reads of LDS are done; then every wave's
template <int N>
__device__ __forceinline__ void ring_wait() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory"); }

}  // namespace adamah
