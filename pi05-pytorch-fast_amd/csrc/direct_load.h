// Direct global-to-LDS loads and the waits that order them, for kernels that keep such loads in
// flight across barriers.  They are inline asm (the loads write LDS only, no register), because
// the compiler puts a wait for every earlier direct load that it knows of before an LDS read.
// It does not count them: a wait that has to cover one is wait_vm, and the compiler's own waits
// for register loads only wait for more.
#pragma once

#include "w4a4_internal.h"

namespace w4a4 {
namespace {

// One 1 KB piece from global memory (uniform base + per-lane byte offset) to LDS address
// `dst` (lane L writes bytes 16 L ..).
__device__ __forceinline__ void load_lds_1k(const char* base, uint32_t voff, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               ::"v"(voff), "s"(base), "s"(__builtin_amdgcn_readfirstlane(dst)) : "memory", "m0");
}

// An ordinary 16-byte load to registers, named because the wait counts include it.
typedef int load_16_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ load_16_t load_16(const char* p) { return *reinterpret_cast<const load_16_t*>(p); }

// Waits until at most N of this wave's vector memory operations are under way.
template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// This wave's LDS operations are done, and every wave of the workgroup has come here.
__device__ __forceinline__ void lds_done_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// A copy that the compiler cannot know to equal v: what is computed from it inside a loop stays
// there, and takes no register across the loop's other parts.
__device__ __forceinline__ int opaque_copy(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

}  // namespace
}  // namespace w4a4
