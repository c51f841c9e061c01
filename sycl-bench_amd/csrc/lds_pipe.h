// Waits and the barrier of the LDS pipelines that global-to-LDS copies feed.
#pragma once

#include "mfx_internal.h"

namespace mfx {

// Waits until at most n of this wave's vector memory operations are
// outstanding (s_waitcnt vmcnt(n), n <= 63; expcnt and lgkmcnt left alone).
template <int n>
__device__ __forceinline__ void vm_wait() {
  static_assert(n >= 0 && n < 64, "vmcnt holds 6 bits");
  __builtin_amdgcn_s_waitcnt((n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8));
}

// Waits for this wave's outstanding LDS operations only.
__device__ __forceinline__ void lds_wait() { __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4)); }

// s_barrier alone, with memory accesses kept on their side of it: the caller
// has waited for what the other waves may read or overwrite.  (__syncthreads
// would also wait for the global-to-LDS copies still in flight.)
__device__ __forceinline__ void bare_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

}  // namespace mfx
