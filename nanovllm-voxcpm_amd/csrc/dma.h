// Direct loads from global memory to LDS and the waits for them.  The loads are inline assembly, which the
// compiler does not count among the loads in flight: whoever uses them writes every wait himself.
#pragma once
#include "common.h"

namespace mlora {

namespace {

template <int N> __device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) char*)(p)));
}
__device__ __forceinline__ const char* uniform(const char* p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v)), hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
  return reinterpret_cast<const char*>((static_cast<uint64_t>(hi) << 32) | lo);
}

// One 1 KB direct load: lane i's 16 bytes at base + voff go to LDS byte lds + 16 i.  The load takes the LDS address from
// m0, which the compiler itself puts there for the asm (an asm that wrote it could not say so: m0 is a reserved
// register and has no place among the clobbers); between that write and the load lies one wait state.
__device__ __forceinline__ void dma16(const void* base, uint32_t voff, uint32_t lds) {
#ifdef MLORA_TRACE
  base = uniform(static_cast<const char*>(base));  // (the branches around the stamps cost the compiler its proof of that)
#endif
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"{m0}"(lds), "v"(voff), "s"(base) : "memory");
}

// The same with the non-temporal hint, for lines that no other workgroup asks for.
__device__ __forceinline__ void dma16_once(const void* base, uint32_t voff, uint32_t lds) {
#ifdef MLORA_TRACE
  base = uniform(static_cast<const char*>(base));
#endif
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"{m0}"(lds), "v"(voff), "s"(base) : "memory");
}

// From a lane's own 64-bit address (rows of x and y lie anywhere).
__device__ __forceinline__ void dma16v(const char* p, uint32_t lds) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"{m0}"(lds), "v"(p) : "memory");
}

// Waits until no more than `younger` (at most MOST) stages of PER loads each are on their way.
template <int PER, int MOST> __device__ __forceinline__ void wait_stages(int younger) {
  if (younger >= MOST) wait_loads<MOST * PER>();
  else if (MOST > 1 && younger == MOST - 1) wait_loads<(MOST > 1 ? MOST - 1 : 0) * PER>();
  else if (MOST > 2 && younger == MOST - 2) wait_loads<(MOST > 2 ? MOST - 2 : 0) * PER>();
  else if (MOST > 3 && younger == MOST - 3) wait_loads<(MOST > 3 ? MOST - 3 : 0) * PER>();
  else if (MOST > 4 && younger == MOST - 4) wait_loads<(MOST > 4 ? MOST - 4 : 0) * PER>();
  else wait_loads<0>();
}

// A barrier that waits for no load.
__device__ __forceinline__ void stage_barrier() { asm volatile("s_barrier" ::: "memory"); }

}  // namespace

}  // namespace mlora
