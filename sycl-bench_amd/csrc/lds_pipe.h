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

// LDS layout of 32 rows x 16 k of a k-contiguous FP32 operand: 128 16-byte
// chunks, chunk c holding row c / 4, k = 4 * kq .. +3.  The four lanes of a
// copy that share a row read its 64 bytes, so one copy of a wave touches 16
// cache lines (rows across the lanes instead: 64, and the address path, not
// the data, bounds the copy).  The order of a row's four chunks is permuted by
// (row / 4) % 4, so that 16 consecutive rows' chunks of one kq fall in
// different banks.  Measured on MI355X against the 64-line order: single BF16
// direct tile, both operands k-contiguous, 4096^3 290 -> 222 us; FP32 64x64
// tile 18.2 -> 17.5 ns per k.
__device__ __forceinline__ int kchunk_row(int c) { return c >> 2; }
__device__ __forceinline__ int kchunk_kq(int c) { return (c & 3) ^ ((c >> 4) & 3); }
__device__ __forceinline__ int kchunk_at(int row, int kq) { return row * 4 + (kq ^ ((row >> 2) & 3)); }

}  // namespace mfx
