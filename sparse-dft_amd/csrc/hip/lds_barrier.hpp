// Workgroup barrier over LDS data only: global loads in flight stay in flight
// (__syncthreads waits for them).
#pragma once
#include <hip/hip_runtime.h>

namespace sdft_hip {

__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0), the other counters free
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

}  // namespace sdft_hip
