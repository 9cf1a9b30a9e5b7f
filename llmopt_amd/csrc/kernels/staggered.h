// Barriers and waits of kernels whose waves multiply and read at different times (dense_gemm.hip, w4a16_gemm.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace llmopt {

// A barrier that nothing moves across.
__device__ __forceinline__ void meet() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
}
template <int COUNT>
__device__ __forceinline__ void copies_landed() {  // all but the last COUNT
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(COUNT) : "memory");
}
__device__ __forceinline__ void lds_read() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

}  // namespace llmopt
