// Workgroup barrier for data in LDS.
#pragma once
#include <hip/hip_runtime.h>

namespace hpq {

// Barrier of a workgroup whose wavefronts exchange data through LDS alone: unlike
// __syncthreads it does not wait for global loads, which stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

}  // namespace hpq
