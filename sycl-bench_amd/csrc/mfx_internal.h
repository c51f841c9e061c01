// Internal declarations shared by the libmfx translation units: the handle,
// launch bookkeeping, number formats (BF16 / OCP e4m3 / keyed RNG) and the
// tile-scheduling helpers used by every kernel family.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstring>
#include <mutex>
#include <string>
#include <type_traits>
#include <utility>
#include <vector>

#include "../../include/mfx.h"

namespace mfx {

// ---------------------------------------------------------------------------
// Error plumbing
// ---------------------------------------------------------------------------
void set_last_error(const std::string& msg);
mfx_status hip_fail(hipError_t e, const char* what);

#define MFX_HIP(expr)                                                   \
  do {                                                                  \
    hipError_t _e = (expr);                                             \
    if(_e != hipSuccess) return ::mfx::hip_fail(_e, #expr);             \
  } while(0)

#define MFX_CHECK(expr)                                                 \
  do {                                                                  \
    mfx_status _s = (expr);                                             \
    if(_s != MFX_SUCCESS) return _s;                                    \
  } while(0)

mfx_status invalid(const std::string& msg);
mfx_status unsupported(const std::string& msg);

// ---------------------------------------------------------------------------
// Handle
// ---------------------------------------------------------------------------
struct TimingRecord {
  const char* name;
  hipEvent_t start;
  hipEvent_t stop;
};

struct Handle {
  int device = 0;
  int cu_count = 0;
  std::string device_name;
  void* workspace = nullptr;
  size_t workspace_bytes = 0;
  bool timing = false;
  std::vector<TimingRecord> records;
  std::vector<hipEvent_t> free_events;
  int forced_config[5] = {-1, -1, -1, -1, -1};
  bool capturing = false;  // set while a grouped launch is being captured
  // Grouped launches: spin limit of the in-kernel dependency waits (env
  // MFX_SPIN_LIMIT overrides), pinned staging for the work tables and the
  // event that marks their upload, and the error flag of the last launch.
  int spin_limit = 1 << 22;
  int grouped_policy = -1;  // forced grouped tile policy (-1: tuned / estimated)
  void* staging = nullptr;
  size_t staging_bytes = 0;
  hipEvent_t staging_ready = nullptr;
  int* error_flag = nullptr;
  bool grouped_waits = true;  // the last grouped call launched kernels that can time out
  int forced_splits = -1;  // split-K: -1 automatic, 1 never, >= 2 that many slices
  // split-K partial tiles, one buffer of kMaxPartialBytes per stream (stream_partials)
  static constexpr int kPartialStreams = 8;
  struct {
    hipStream_t stream;
    void* p;
  } partials[kPartialStreams] = {};
  int partial_streams = 0;
  // packed operands of lists that run as dense launches (list_workspace)
  void* list_memory = nullptr;
  size_t list_bytes = 0;
};

inline int cus_of(const Handle* h) { return h->cu_count > 0 ? h->cu_count : 256; }

// Looks up the device's fixed no-allocation scratch array (mfx_create calls
// it with the device current).
mfx_status noalloc_init(int device);

// Returns a workspace pointer of at least `bytes` (grows the arena; growing
// synchronises the device, so it must not happen under graph capture).
mfx_status workspace(Handle* h, size_t bytes, void** out);
// The same in memory of its own, which no caller's graph holds: a list that runs
// as dense launches needs more than its tables, and must not regrow the
// workspace that a captured call points into.
mfx_status list_workspace(Handle* h, size_t bytes, void** out);

// Stream s's own buffer of kMaxPartialBytes for split-K partial tiles, allocated
// at its first use and kept until mfx_destroy, so that two streams' calls on one
// handle do not meet in it and no later call moves it (a stream whose value an
// ended one had before finds it idle: hipStreamDestroy waits for the work). Null where there is none
// (the caller then runs unsplit): the stream is being captured, whose graph may
// replay beside anything; it is hipStreamPerThread, one value for several
// streams; kPartialStreams others hold one; or the memory is not to be had.
void* stream_partials(Handle* h, hipStream_t s);

// Memory of a packed call: *ws for its packed operands, *partials for its
// partial tiles, behind them where the workspace already holds both, else the
// stream's buffer, else null (none, or not to be had: the caller runs unsplit).
// Partial tiles never regrow the workspace, so one that holds the packed operands
// stays where a captured call found it.
mfx_status packed_workspace(Handle* h, size_t packed, size_t partial, hipStream_t s, void** ws, void** partials);

// Whether a call on s is being captured into a caller's or the library's graph.
bool is_capturing(const Handle* h, hipStream_t s);

// Records an event pair around `launch()` when timing is on, and converts a
// launch error into MFX_ERROR_HIP.
template <class F>
mfx_status timed_launch(Handle* h, const char* name, hipStream_t s, F&& launch);

hipEvent_t take_event(Handle* h);

template <class F>
mfx_status timed_launch(Handle* h, const char* name, hipStream_t s, F&& launch) {
  hipEvent_t a = nullptr, b = nullptr;
  if(h->timing) {
    a = take_event(h);
    b = take_event(h);
    if(!a || !b) return hip_fail(hipErrorOutOfMemory, "hipEventCreate");
    MFX_HIP(hipEventRecord(a, s));
  }
  launch();
  hipError_t e = hipGetLastError();
  if(e != hipSuccess) return hip_fail(e, name);
  if(h->timing) {
    MFX_HIP(hipEventRecord(b, s));
    h->records.push_back({name, a, b});
  }
  return MFX_SUCCESS;
}

inline int64_t round_up(int64_t x, int64_t m) { return (x + m - 1) / m * m; }
inline int64_t ceil_div(int64_t x, int64_t m) { return (x + m - 1) / m; }

// ---------------------------------------------------------------------------
// Number formats (host + device, bit-exact on both sides)
// ---------------------------------------------------------------------------
__host__ __device__ inline uint32_t f32_bits(float x) {
  uint32_t u;
  memcpy(&u, &x, 4);
  return u;
}
__host__ __device__ inline float bits_f32(uint32_t u) {
  float x;
  memcpy(&x, &u, 4);
  return x;
}

// Round-to-nearest-even FP32 -> BF16 (NaN stays NaN, quiet).
__host__ __device__ inline uint16_t bf16_rne(float x) {
  uint32_t u = f32_bits(x);
  if((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__host__ __device__ inline float bf16_to_f32(uint16_t h) { return bits_f32((uint32_t)h << 16); }

// OCP e4m3 (E4M3FN: bias 7, max 448, no infinities, S.1111.111 = NaN),
// round-to-nearest-even, saturating to +-448.
__host__ __device__ inline uint8_t e4m3_rne_sat(float x) {
  uint32_t u = f32_bits(x);
  uint8_t sign = (uint8_t)((u >> 24) & 0x80u);
  uint32_t au = u & 0x7fffffffu;
  if(au > 0x7f800000u) return (uint8_t)(sign | 0x7f);
  float a = bits_f32(au);
  if(a > 448.0f) return (uint8_t)(sign | 0x7e);
  if(a < 0.015625f) {  // below the smallest normal 2^-6: multiples of 2^-9
    float s = a * 512.0f;  // exact
    // round half to even on an exact value in [0, 8)
    uint32_t i = (uint32_t)s;
    float frac = s - (float)i;
    if(frac > 0.5f || (frac == 0.5f && (i & 1u))) ++i;
    return (uint8_t)(sign | i);  // i == 8 encodes the smallest normal
  }
  int e = (int)((au >> 23) & 0xffu) - 127;  // -6 .. 8
  uint32_t m = au & 0x7fffffu;
  uint32_t r = (m + 0x7ffffu + ((m >> 20) & 1u)) >> 20;  // 0 .. 8
  uint32_t code = ((uint32_t)(e + 7) << 3) + r;
  if(code > 0x7eu) code = 0x7eu;
  return (uint8_t)(sign | code);
}
__host__ __device__ inline float e4m3_to_f32(uint8_t q) {
  uint32_t s = q & 0x80u, e = (q >> 3) & 0xfu, m = q & 7u;
  float v;
  if(e == 15 && m == 7) return bits_f32(0x7fc00000u | (s << 24));
  if(e == 0)
    v = (float)m * 0.001953125f;  // m * 2^-9
  else
    v = bits_f32(((e + 120u) << 23) | (m << 20));
  return s ? -v : v;
}

// Smallest e with amax <= 448 * 2^e (0 for amax == 0), clamped to the E8M0
// range usable as an MFMA scale.
__host__ __device__ inline int fp8_block_exponent(float amax) {
  if(!(amax > 0.0f)) return 0;
  int e = (int)((f32_bits(amax) >> 23) & 0xffu) - 127 - 8;
  if(((f32_bits(amax) >> 23) & 0xffu) == 0) e = -126 - 8;
  // adjust so that 448*2^(e-1) < amax <= 448*2^e, using exact power-of-two scaling
  for(int it = 0; it < 4; ++it) {
    if(amax > ldexpf(448.0f, e)) ++e;
    else if(amax <= ldexpf(448.0f, e - 1)) --e;
    else break;
  }
  if(e < -127) e = -127;
  if(e > 127) e = 127;
  return e;
}

// Keyed SplitMix64: the value for (seed, matrix, index) is independent of
// launch shape, so host and device generate bit-identical inputs.
__host__ __device__ inline uint64_t mix64(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}
__host__ __device__ inline uint64_t keyed_hash(uint64_t seed, uint32_t matrix, uint64_t index) {
  uint64_t base = mix64(seed ^ (0x9e3779b97f4a7c15ull * ((uint64_t)matrix + 1ull)));
  return mix64(base + 0x9e3779b97f4a7c15ull * (index + 1ull));
}
// 2 * (h >> 40) * 2^-24 - 1: a 24-bit grid on [-1, 1), exact in FP32.
__host__ __device__ inline float uniform_pm1(uint64_t h) {
  return (float)(uint32_t)(h >> 40) * 1.1920928955078125e-07f - 1.0f;
}

// ---------------------------------------------------------------------------
// Tile scheduling
// ---------------------------------------------------------------------------
// Workgroups are dispatched round-robin over the 8 XCDs (wg i -> XCD i % 8).
// This renumbers them so each XCD owns one contiguous range of tile ids, which
// keeps the A/B panels a tile needs in that XCD's L2.
__device__ __forceinline__ int xcd_remap(int bid, int nblocks) {
  const int xcd = bid & 7, local = bid >> 3;
  const int per = nblocks >> 3, rem = nblocks & 7;
  return xcd < rem ? xcd * (per + 1) + local : rem * (per + 1) + (xcd - rem) * per + local;
}

// Grouped ordering: GROUP consecutive tile rows are walked column by column.
__host__ __device__ __forceinline__ void grouped_tile(int pid, int tiles_m, int tiles_n, int group, int& tm, int& tn) {
  const int in_group = group * tiles_n;
  const int gid = pid / in_group;
  const int first_m = gid * group;
  const int gsize = tiles_m - first_m < group ? tiles_m - first_m : group;
  const int r = pid - gid * in_group;
  tm = first_m + r % gsize;
  tn = r / gsize;
}

// The lower triangle of a T x T tile grid in bands of `group` tile rows, each
// band walked column by column (its full-width part, then its own triangle),
// so consecutive ids -- one XCD's workgroups after xcd_remap -- cover a
// compact block of tiles that shares A and B panels in L2, as grouped_tile
// does for a full grid.  A plain row-by-row order gives each round of an
// XCD's workgroups one or two tile rows and as many distinct B panels as
// tiles.  Every (ti, tj) with tj <= ti < T once for
// p < T (T + 1) / 2.
__host__ __device__ inline void grouped_lower_tile(int p, int T, int group, int& ti, int& tj) {
  int r0 = 0, rows = group < T ? group : T;
  for(;;) {
    const int in_band = rows * r0 + rows * (rows + 1) / 2;
    if(p < in_band || r0 + rows >= T) break;
    p -= in_band;
    r0 += rows;
    rows = group < T - r0 ? group : T - r0;
  }
  if(p < rows * r0) {
    tj = p / rows;
    ti = r0 + p % rows;
    return;
  }
  p -= rows * r0;
  int c = 0;
  while(p >= rows - c) {
    p -= rows - c;
    ++c;
  }
  tj = r0 + c;
  ti = r0 + c + p;
}

// A triangular launch's tile (ti, tj) for id p: the triangle order of the
// T x T grid, or -- when `tail_first` >= 0, the re-tiled last round of a
// bigger tile's triangle (tri_tail) -- sub-tile p % r^2 of big tile
// tail_first + p / r^2 of the big_T x big_T triangle.  False for a sub-tile
// with nothing of the triangle in it (above a diagonal big tile's diagonal,
// or past the matrix), which the workgroup skips.
__host__ __device__ inline bool triangle_tile(int p, int T, int group, int tail_first, int r, int big_T, int& ti,
    int& tj) {
  if(tail_first < 0) {
    grouped_lower_tile(p, T, group, ti, tj);
    return true;
  }
  int bi, bj;
  grouped_lower_tile(tail_first + p / (r * r), big_T, group, bi, bj);
  const int s = p % (r * r);
  ti = bi * r + s / r;
  tj = bj * r + s % r;
  return tj <= ti && ti < T;
}

// Scheduling modes shared by the FP32 and BF16 kernel families.
enum TileMode : int { TILES_FULL = 0, TILES_LOWER = 1, TILES_UPPER = 2 };

// Tile `id` of a full grid, or of a triangle (tiles_m == tiles_n).
__host__ __device__ inline void tile_of(int mode, int id, int tiles_m, int tiles_n, int group, int& tm, int& tn) {
  if(mode == TILES_FULL) {
    grouped_tile(id, tiles_m, tiles_n, group, tm, tn);
  } else {
    int ti, tj;
    grouped_lower_tile(id, tiles_m, group, ti, tj);
    tm = mode == TILES_LOWER ? ti : tj;
    tn = mode == TILES_LOWER ? tj : ti;
  }
}

// Split-K of a tiled launch: tiles [0, head) run whole; each tile from `head`
// on runs as `splits` slices of its k stages, which write partial tiles
// (tile - head) * splits + slice of bm x bn floats, summed in slice order by
// splitk_reduce (splitk.hip).  splits == 1: no tile is split (head = tiles).
struct SplitPlan {
  int head = 0, splits = 1;
};

// Epilogue parameters common to all families.
struct Epilogue {
  float* C;
  int64_t ldc;
  float alpha, beta;
  int M, N;
  int uplo;    // TILES_FULL: write everything; LOWER/UPPER: that triangle only
  int mirror;  // also write the opposite triangle from the transposed value
};

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

// One 16-byte chunk per lane from global memory straight into LDS
// (global_load_lds_dwordx4): lane l's chunk lands at lds_wave_base + l.  The
// LDS base must be the same for the whole wave.
template <class T>
__device__ __forceinline__ void lds_dma16(const T* src, T* lds_wave_base) {
  static_assert(sizeof(T) == 16, "one 16-byte chunk per lane");
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
      (__attribute__((address_space(3))) void*)lds_wave_base, 16, 0, 0);
}

// The same with one 4-byte value per lane (global_load_lds_dword).
template <class T>
__device__ __forceinline__ void lds_dma4(const T* src, T* lds_wave_base) {
  static_assert(sizeof(T) == 4, "one 4-byte value per lane");
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
      (__attribute__((address_space(3))) void*)lds_wave_base, 4, 0, 0);
}

// Waits for this wave's outstanding memory operations, LDS transfers included.
__device__ __forceinline__ void lds_dma_wait() { __builtin_amdgcn_s_waitcnt(0); }

// Compile-time loop: f(std::integral_constant<int, I>) for I in [0, N).  Used
// where an index selects an accumulator block, so the index stays a constant
// and the accumulators stay in registers (a runtime index, or a loop the
// unroller gives up on, moves the whole array to scratch memory).
template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// alpha * acc + beta * old, rounded the same way wherever it is written: the two
// halves of a mirrored square have to agree to the last bit, and left to itself
// the compiler fuses either product into the sum.
__device__ __forceinline__ float scaled(const Epilogue& ep, float acc, float old) {
  return fmaf(ep.alpha, acc, ep.beta * old);
}

// Writes one 32x32 MFMA accumulator block whose top-left corner is (r0, c0).
// v_mfma_f32_32x32x* layout: lane l, register q holds
// row 8*(q/4) + 4*(l/32) + q%4, column l%32.
// Always inlined and taking the block by value: a call would force the whole
// accumulator array into scratch memory.
// All old values of a block are loaded, and all new ones computed, before its
// first store, which the compiler may not do by itself (C may alias C): with one
// load, wait and store per element the triangle blocks of a 1024 x 1024 FP32 syrk
// took 7 us of its 29. The value is chosen by beta first and stored by position
// afterwards: a predicated store that chose it itself waited, even without beta,
// for every memory operation before it, the previous store among them, which cost
// a block at the matrix's edge 2.4 us. A mirrored block's transposed value is four
// consecutive floats of a row in each lane, written 16 bytes wide where C's rows
// are aligned for it.
__device__ __forceinline__ void store_block32(const Epilogue& ep, floatx16 acc, int r0, int c0, int lane) {
  const int col = c0 + (lane & 31);
  const int rbase = r0 + 4 * (lane >> 5);
  const bool inside = ep.uplo == TILES_FULL || (ep.uplo == TILES_LOWER ? r0 >= c0 + 32 : c0 >= r0 + 32);
  float* const direct = ep.C + (int64_t)rbase * ep.ldc + col;
  float* const mirrored = ep.C + (int64_t)col * ep.ldc + rbase;
  float v[16];
  if(inside && r0 + 32 <= ep.M && c0 + 32 <= ep.N) {
    // Interior block: each register q is one 32-float row segment per half wave.
    if(ep.beta != 0.0f) {
      float old[16];
#pragma unroll
      for(int q = 0; q < 16; ++q) old[q] = direct[(int64_t)(8 * (q >> 2) + (q & 3)) * ep.ldc];
#pragma unroll
      for(int q = 0; q < 16; ++q) direct[(int64_t)(8 * (q >> 2) + (q & 3)) * ep.ldc] = scaled(ep, acc[q], old[q]);
    } else {
#pragma unroll
      for(int q = 0; q < 16; ++q) direct[(int64_t)(8 * (q >> 2) + (q & 3)) * ep.ldc] = ep.alpha * acc[q];
    }
    if(ep.uplo == TILES_FULL || !ep.mirror) return;
    const bool wide = ep.ldc % 4 == 0 && (reinterpret_cast<uintptr_t>(ep.C) & 15u) == 0;
    if(ep.beta != 0.0f) {
      float old[16];
      if(wide) {
#pragma unroll
        for(int g = 0; g < 4; ++g) {
          const floatx4 was = *reinterpret_cast<const floatx4*>(mirrored + 8 * g);
#pragma unroll
          for(int u = 0; u < 4; ++u) old[4 * g + u] = was[u];
        }
      } else {
#pragma unroll
        for(int q = 0; q < 16; ++q) old[q] = mirrored[8 * (q >> 2) + (q & 3)];
      }
#pragma unroll
      for(int q = 0; q < 16; ++q) v[q] = scaled(ep, acc[q], old[q]);
    } else {
#pragma unroll
      for(int q = 0; q < 16; ++q) v[q] = ep.alpha * acc[q];
    }
    if(wide) {
#pragma unroll
      for(int g = 0; g < 4; ++g)
        *reinterpret_cast<floatx4*>(mirrored + 8 * g) = (floatx4){v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]};
    } else {
#pragma unroll
      for(int q = 0; q < 16; ++q) mirrored[8 * (q >> 2) + (q & 3)] = v[q];
    }
    return;
  }
  // nothing of the block is wanted: a small problem's tile has many of these
  if(r0 >= ep.M || c0 >= ep.N || (ep.uplo == TILES_LOWER && r0 + 31 < c0) || (ep.uplo == TILES_UPPER && c0 + 31 < r0)) return;
  // A block at the matrix's edge or across the diagonal: old values come from
  // clamped positions without a branch (those of elements that are not written
  // are not used), so that only the stores are predicated, by the rows [lo, hi)
  // that this lane's column has (a test of uplo for each element was five
  // branches).
  const int last_row = ep.M - 1, near_col = min(col, ep.N - 1);
  const int lo = ep.uplo == TILES_LOWER ? col : 0;
  const int hi = col >= ep.N ? 0 : ep.uplo == TILES_UPPER ? min(col + 1, ep.M) : ep.M;
  auto row_of = [&](int q) { return rbase + 8 * (q >> 2) + (q & 3); };
  if(ep.beta != 0.0f) {
    float old[16];
#pragma unroll
    for(int q = 0; q < 16; ++q) old[q] = ep.C[(int64_t)min(row_of(q), last_row) * ep.ldc + near_col];
#pragma unroll
    for(int q = 0; q < 16; ++q) v[q] = scaled(ep, acc[q], old[q]);
  } else {
#pragma unroll
    for(int q = 0; q < 16; ++q) v[q] = ep.alpha * acc[q];
  }
#pragma unroll
  for(int q = 0; q < 16; ++q)
    if(row_of(q) >= lo && row_of(q) < hi) direct[(int64_t)(8 * (q >> 2) + (q & 3)) * ep.ldc] = v[q];
  if(ep.uplo == TILES_FULL || !ep.mirror) return;
  // C is square; the diagonal has no mirror
  const int mlo = ep.uplo == TILES_LOWER ? col + 1 : 0, mhi = ep.uplo == TILES_UPPER ? min(col, hi) : hi;
  if(ep.beta != 0.0f) {  // without it the transposed value is the same
    float old[16];
#pragma unroll
    for(int q = 0; q < 16; ++q) old[q] = ep.C[(int64_t)near_col * ep.ldc + min(row_of(q), last_row)];
#pragma unroll
    for(int q = 0; q < 16; ++q) v[q] = scaled(ep, acc[q], old[q]);
  }
#pragma unroll
  for(int q = 0; q < 16; ++q)
    if(row_of(q) >= mlo && row_of(q) < mhi) mirrored[8 * (q >> 2) + (q & 3)] = v[q];
}

// ---------------------------------------------------------------------------
// Launchers implemented by the kernel translation units
// ---------------------------------------------------------------------------
struct DenseOp {
  // C = alpha * sum_p opA_p * opB_p + beta * C, with p over one or two products
  // (two for syr2k: A*B^T then B*A^T).
  int M, N, K;
  const float* A; int64_t lda; bool a_kmajor;  // element (m,k) at A[m*lda+k] if kmajor else A[k*lda+m]
  const float* B; int64_t ldb; bool b_kmajor;  // element (k,n) at B[n*ldb+k] if kmajor else B[k*ldb+n]
  int nprod;                                    // 1, or 2 with operands swapped for the second
  Epilogue ep;
  int tiles;                                    // TILES_FULL / LOWER / UPPER
};

// FP32 triangular schedules whose last round of tiles leaves most CUs idle: the
// full rounds run on the chosen square tile, and the big tiles of the last
// round are re-tiled `ratio` x `ratio` into a smaller square configuration
// in a second launch, when that is estimated faster than one more round of
// big tiles (small == -1: no re-tiling).
struct TriTail {
  int head = 0;     // big tiles of the first launch (all of them without re-tiling)
  int small = -1;   // configuration of the second launch
  int ratio = 1;    // big tile side / small tile side
  double us = 0.0;  // estimated microseconds of both
};
TriTail tri_tail(mfx_precision p, int config, int64_t tiles_per_side, int cus, int64_t k = 4096);
// How an FP32 triangle runs on `config`: its k slices or its re-tiled last round,
// whichever is estimated shorter, and that estimate. The one place that decides,
// for the choice of the configuration, the memory and the launch.
double plan_f32_triangle(int config, int64_t tiles_per_side, int64_t k, int cus, int64_t max_partial, SplitPlan* plan,
    TriTail* tail);

mfx_status launch_dense_f32(Handle* h, const DenseOp& op, int config, hipStream_t s);
// The same with split-K partial tiles in `ws` (ws_bytes long) instead of the
// stream's buffer; fails if a split this call makes needs more.
mfx_status launch_dense_f32_ws(Handle* h, const DenseOp& op, int config, void* ws, size_t ws_bytes, hipStream_t s);
size_t dense_f32_workspace(const DenseOp& op, int config, int cus, int forced_splits);
mfx_status launch_dense_bf16x(Handle* h, const DenseOp& op, bool split, int config, hipStream_t s);
// The same on a caller-provided workspace of dense_bf16x_workspace() bytes, or
// with its partial tiles in `partials` and the packed operands alone in ws.
mfx_status launch_dense_bf16x_ws(Handle* h, const DenseOp& op, bool split, int config, void* ws, hipStream_t s,
    void* partials = nullptr);

// Sums the partial tiles of a split launch and applies op's epilogue.
struct SplitReduceArgs {
  const float* partial;
  int bm, bn, splits;
  int head, tiles;  // split tiles are [head, tiles)
  int mode, tiles_m, tiles_n, group;
  Epilogue ep;
};
mfx_status launch_splitk_reduce(Handle* h, const SplitReduceArgs& a, hipStream_t s);
constexpr int64_t kMaxPartialBytes = (int64_t)32 << 20;
// The configuration for `op` without k slices, in place of `config` (chosen with
// them): `config` itself where it was forced or tuned.
int whole_config(Handle* h, mfx_precision p, const DenseOp& op, int config);
// Estimated microseconds of `count` workgroups of `len` k each (no split).
double tile_span(mfx_precision p, int config, int64_t count, double len, int cus);
bool bf16_two_per_cu(mfx_precision p, int config, int64_t tiles, int64_t k, int cus);
// Estimated microseconds of a dense launch on `config` (tile_span's model)
// and the split plan behind it; partial tiles take at most max_partial bytes.
double plan_splits(mfx_precision p, int config, int64_t tiles, int64_t k, int cus, int64_t max_partial, SplitPlan* plan);
mfx_status launch_dense_fp8(Handle* h, const DenseOp& op, bool two_term, int config, hipStream_t s);
// Packed operands and split-K partial tiles (*partial of them, at the end).
size_t dense_bf16x_workspace(const DenseOp& op, bool split, int config, int cus, int forced_splits,
    size_t* partial = nullptr);
size_t dense_fp8_workspace(const DenseOp& op, bool two_term, int config, int cus);

int config_count(mfx_precision p);
bool config_info(mfx_precision p, int c, int* bm, int* bn, int* bk, int* waves);
int choose_config(Handle* h, mfx_precision p, int64_t m, int64_t n, int64_t k);

}  // namespace mfx

struct mfx_handle_s {
  mfx::Handle h;
};
