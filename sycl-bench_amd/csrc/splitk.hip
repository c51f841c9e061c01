// Split-K plans and the reduction behind them, shared by the kernel families.
//
// A schedule whose tiles do not fill whole rounds of the CUs runs the tiles
// of its last, partial round (all of them, when there are fewer tiles than
// CUs) as k slices in separate workgroups.  Each slice writes its partial
// tile to the workspace; splitk_reduce, in a launch of its own, sums the
// partials of every output element in slice order (the same result on every
// run) and applies alpha / beta.  The kernel boundary orders the two, so no
// workgroup waits for another: a form that summed in the last-arriving
// workgroup had every workgroup write back its XCD's whole L2 and took twice
// the time of the unsplit kernel.
#include <algorithm>

#include "mfx_internal.h"

namespace mfx {
namespace {

// One 32 x 32 sub-block of a split tile per workgroup, four consecutive
// columns per thread: 16-byte loads of the partials (four slices in flight),
// 16-byte accesses to C where its alignment allows.  A mirrored block is
// transposed through LDS, so its stores are row segments too.  HBM-bound:
// splits * bm * bn * 4 bytes per tile, which the slices have just written.
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const SplitReduceArgs p) {
  const int sub_n = p.bn / 32, subs = p.bm / 32 * sub_n;
  const int t = blockIdx.x / subs, sub = blockIdx.x - t * subs;
  int tm, tn;
  tile_of(p.mode, p.head + t, p.tiles_m, p.tiles_n, p.group, tm, tn);
  const int lr0 = sub / sub_n * 32, lc0 = sub % sub_n * 32;  // within the tile
  const int r0 = tm * p.bm + lr0, c0 = tn * p.bn + lc0;
  const Epilogue& ep = p.ep;
  if(r0 >= ep.M || c0 >= ep.N) return;
  if(ep.uplo == TILES_LOWER && r0 + 31 < c0) return;
  if(ep.uplo == TILES_UPPER && c0 + 31 < r0) return;
  const int lr = threadIdx.x >> 3, lc = (threadIdx.x & 7) * 4;
  const int64_t area4 = (int64_t)p.bm * p.bn / 4;
  const floatx4* src = reinterpret_cast<const floatx4*>(p.partial) + (int64_t)t * p.splits * area4 +
                       ((lr0 + lr) * p.bn + lc0 + lc) / 4;
  floatx4 v = src[0];
  int s = 1;
  for(; s + 4 <= p.splits; s += 4) {
    floatx4 w[4];
#pragma unroll
    for(int u = 0; u < 4; ++u) w[u] = src[(s + u) * area4];
#pragma unroll
    for(int u = 0; u < 4; ++u) v += w[u];
  }
  for(; s < p.splits; ++s) v += src[s * area4];

  const int row = r0 + lr, col = c0 + lc;
  const bool vec = (reinterpret_cast<uintptr_t>(ep.C) & 15u) == 0 && ep.ldc % 4 == 0;
  const bool inside = r0 + 32 <= ep.M && c0 + 32 <= ep.N;
  if(ep.uplo == TILES_FULL && inside && vec) {
    floatx4* c = reinterpret_cast<floatx4*>(ep.C + (int64_t)row * ep.ldc + col);
    const floatx4 old = ep.beta != 0.0f ? *c : v;
#pragma unroll
    for(int e = 0; e < 4; ++e) v[e] = ep.beta != 0.0f ? scaled(ep, v[e], old[e]) : ep.alpha * v[e];
    *c = v;
    return;
  }
  auto wanted = [&](int r, int c) {
    return r < ep.M && c < ep.N && (ep.uplo == TILES_FULL || (ep.uplo == TILES_LOWER ? r >= c : r <= c));
  };
#pragma unroll
  for(int e = 0; e < 4; ++e)
    if(wanted(row, col + e)) {
      float* c = ep.C + (int64_t)row * ep.ldc + col + e;
      *c = ep.beta != 0.0f ? scaled(ep, v[e], *c) : ep.alpha * v[e];
    }
  if(ep.uplo == TILES_FULL || !ep.mirror) return;
  // element (row, col) of the triangle also gives (col, row), from its own C
  __shared__ float tr[32][33];
#pragma unroll
  for(int e = 0; e < 4; ++e) tr[lr][lc + e] = v[e];
  __syncthreads();
#pragma unroll
  for(int e = 0; e < 4; ++e) {
    const int r = r0 + lc + e, cc = c0 + lr;  // source element; its mirror is (cc, r)
    if(r != cc && wanted(r, cc)) {
      float* c = ep.C + (int64_t)cc * ep.ldc + r;
      const float x = tr[lc + e][lr];
      *c = ep.beta != 0.0f ? scaled(ep, x, *c) : ep.alpha * x;
    }
  }
}

// Time of one tile, microseconds: `fixed` for its launch, first loads and
// epilogue, and nanoseconds per k with at most a third of the CUs busy
// (latency and LDS bound), with all of them busy (power, L2 and fabric shared
// by every CU) and, for tiles small enough in LDS, with two on every CU.
// Measured on MI355X at K = 1024 and 4096.
struct TileCost {
  double fixed, idle, full, twice;  // twice == 0: one tile per CU
};
constexpr TileCost kF32Cost[] = {
    {25.0, 231.0, 228.0, 0.0},  // 256x256, four waves
    {8.0, 65.0, 64.0, 122.0},   // 128x128, four waves
    {8.0, 20.3, 21.1, 35.0},    // 64x64 in many short slices by a rule of its own: priced out of the choice
    {18.0, 120.0, 115.0, 0.0},  // 256x128, four waves
    {25.0, 226.0, 220.0, 0.0},  // 256x256, eight waves
    {18.0, 116.0, 112.0, 0.0},  // 256x128, eight waves
    {8.0, 59.4, 62.0, 123.0},   // 128x128, eight waves
    {4.0, 16.4, 18.2, 34.5},    // 64x64, two k-groups
};
constexpr TileCost kSplitCost[] = {
    {12.0, 44.0, 64.0, 0.0}, // 256x256, four waves: one wave per SIMD stores the tile
    {5.8, 12.4, 18.0, 0.0},  // 128x128, four waves
    {4.0, 6.7, 6.8, 13.0},   // 64x64
    {7.0, 22.5, 33.0, 0.0},  // 256x128, four waves
    {6.0, 43.6, 65.0, 0.0},  // 256x256, eight waves
    {6.5, 22.6, 34.0, 0.0},  // 256x128, eight waves
    {4.9, 13.3, 19.0, 0.0},  // 128x128, eight waves
};
constexpr TileCost kBf16Cost[] = {
    {13.5, 16.0, 24.5, 0.0}, {4.5, 6.2, 8.2, 0.0},  {3.4, 3.87, 3.9, 5.5}, {5.5, 9.7, 14.0, 0.0},
    {6.0, 15.4, 24.5, 0.0}, {5.3, 9.5, 13.8, 0.0}, {4.0, 6.1, 8.3, 0.0},
};
constexpr TileCost kFp8Cost[] = {
    {16.0, 7.7, 10.8, 0.0},  // 256x256, four waves
    {6.5, 2.8, 3.5, 0.0},    // 128x128
    {10.0, 7.8, 10.9, 0.0},  // 256x256, eight waves
    {3.0, 1.6, 1.9, 2.86},   // 64x64
};
constexpr TileCost kFp8TwoCost[] = {
    {14.0, 22.5, 30.6, 0.0}, {6.0, 7.7, 9.7, 0.0}, {9.0, 22.7, 32.0, 0.0}, {3.0, 3.9, 4.3, 6.57}};

// Reading the partials back and the launch that does it.  Below kSplitFromUs
// a call is bound by its launches on the host (about 10 us for the first, 3.5
// for each further one, from Python), which a split adds to.
constexpr double kReduceFixedUs = 3.5, kReduceBytesPerUs = 4.0e6, kSplitFromUs = 11.0;

bool tile_cost(mfx_precision p, int c, TileCost* out) {
  if(c < 0 || c >= config_count(p)) return false;
  switch(p) {
    case MFX_PREC_FP32: *out = kF32Cost[c]; return true;
    case MFX_PREC_SPLIT_BF16: *out = kSplitCost[c]; return true;
    case MFX_PREC_BF16: *out = kBf16Cost[c]; return true;
    case MFX_PREC_FP8_BLOCK: *out = kFp8Cost[c]; return true;
    case MFX_PREC_FP8_BLOCK2: *out = kFp8TwoCost[c]; return true;
    default: return false;
  }
}

}  // namespace

mfx_status launch_splitk_reduce(Handle* h, const SplitReduceArgs& a, hipStream_t s) {
  const int64_t grid = (int64_t)(a.tiles - a.head) * (a.bm / 32) * (a.bn / 32);
  if(grid == 0) return MFX_SUCCESS;
  return timed_launch(h, "splitk_reduce", s, [&] { splitk_reduce_kernel<<<(unsigned)grid, 256, 0, s>>>(a); });
}

// `count` workgroups of `len` k each cost fixed + len * (ns per k at the load
// they put on the CUs) per round.
double tile_span(mfx_precision p, int config, int64_t count, double len, int cus) {
  TileCost tc;
  if(count <= 0 || !tile_cost(p, config, &tc)) return 0.0;
  const int64_t slots = tc.twice > 0.0 ? 2 * (int64_t)cus : cus;
  const int64_t rounds = count / slots, rest = count - rounds * slots;
  auto round = [&](double load) {  // load: workgroups per CU
    const double ns = load > 1.0 ? tc.twice  // the CUs that got two set the pace
                                 : tc.idle + (tc.full - tc.idle) * std::max(0.0, (load - 0.33) / 0.67);
    return tc.fixed + 1e-3 * ns * len;
  };
  return (double)rounds * round((double)slots / cus) + (rest ? round((double)rest / cus) : 0.0);
}

// Whether the eight-wave 128x128 BF16 tile runs with two LDS buffers instead of
// four, which lets two workgroups share a CU: sums of at most four stages (128
// k split, 256 single) have nothing for the third and fourth buffer, and more
// tiles than CUs are bound by storing C, which one workgroup does while the
// other loads and multiplies.  5524 x 7793 x 79, the
// call: split BF16 62.6 -> 48.0 us (61.0 on the best other tile), single BF16
// 53.6 -> 39.0 (52.4).
bool bf16_two_per_cu(mfx_precision p, int config, int64_t tiles, int64_t k, int cus) {
  const int64_t most = p == MFX_PREC_SPLIT_BF16 ? 128 : p == MFX_PREC_BF16 ? 256 : 0;
  return config == 6 && k <= most && tiles > cus;
}

// The tiles that do not fill a round of the CUs -- all of them, or those past
// the whole rounds -- run whole or in up to 64 slices of at least two stages,
// whichever this model makes shorter: tile_span, and for a split the
// reduction.
double plan_splits(mfx_precision p, int config, int64_t tiles, int64_t k, int cus, int64_t max_partial,
    SplitPlan* plan) {
  int bm, bn, bk, w;
  if(plan) *plan = SplitPlan{(int)tiles, 1};
  if(!config_info(p, config, &bm, &bn, &bk, &w) || tiles <= 0) return 0.0;
  // two tiles per CU and round, which take turns storing: 2.5 us on the scale of
  // the other tiles' `fixed`, which does not hold the stores of round after round
  if(bf16_two_per_cu(p, config, tiles, k, cus))
    return (double)ceil_div(tiles, 2 * (int64_t)cus) * (2.5 + 1e-3 * (p == MFX_PREC_SPLIT_BF16 ? 26.0 : 13.0) * (double)k);
  auto span = [&](int64_t count, double len) { return tile_span(p, config, count, len, cus); };
  double best = span(tiles, (double)k);
  const int64_t steps = ceil_div(k, bk);
  const double tile_bytes = 4.0 * bm * bn;
  auto try_split = [&](int64_t head) {
    const int64_t rest = tiles - head;
    const double whole = head ? span(head, (double)k) : 0.0;
    // few, widening candidates: this runs in every call
    for(int64_t s = 2; s <= 64 && 2 * s <= steps && whole < best; s += s < 8 ? 1 : s / 4) {
      const double bytes = (double)(rest * s) * tile_bytes;
      if(bytes > (double)max_partial) break;
      const double t = whole + span(rest * s, (double)(ceil_div(steps, s) * bk)) + kReduceFixedUs + bytes / kReduceBytesPerUs;
      if(t < best * 0.98) {  // a split has to be clearly ahead
        best = t;
        if(plan) *plan = SplitPlan{(int)head, (int)s};
      }
    }
  };
  if(best < kSplitFromUs) return best;
  if(tiles % cus) try_split(tiles / cus * cus);
  if(tiles > cus && tiles < 3 * cus) try_split(0);
  return best;
}

}  // namespace mfx
