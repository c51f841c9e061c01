// Host side of the persistent grouped launch (queue layout and protocol in
// grouped.h): planning, workspace binding, the tile policy, chains, the
// hipGraph form and the C entry points.
#include <algorithm>
#include <array>
#include <cmath>
#include <cstdlib>
#include <memory>
#include <numeric>
#include <optional>
#include <queue>

#include "grouped.h"

namespace mfx {

std::string tune_key(mfx_precision p, int64_t m, int64_t n, int64_t k);
int tuned_lookup(const std::string& key);
bool tuned_any();

namespace {

// Tile policies: (large, small, bound) -- a problem takes the large tile when
// that pads its output area by at most `bound` (0: always), else the small
// one.  The FP32 grouped kernels do not compile the 256x256 configuration (0)
// and run 256x128 (3) in its place.
struct GroupedPolicy {
  int big, small;
  double bound;
  // 0: one persistent kernel, in-kernel dependency waits; 1: one pre-pass +
  // persistent launch per dependency level, no in-kernel waits; 2:
  // pipelined segments -- like 1, with the independent problems spread over
  // at least three segments and each launch packing the next segment's
  // independent operands in pre-pack items beside its own tiles.
  int per_level;
  // BF16: problems whose operands allow it (K % 16 == 0, aligned rows) run
  // bf16_tile_direct on their FP32 operands instead of being packed.
  int direct;
};
constexpr GroupedPolicy kPolicies[] = {
    {0, 0, 0.0},   // 0
    {0, 1, 1.34},  // 1
    {0, 2, 1.34},  // 2
    {3, 3, 0.0},   // 3
    {3, 1, 1.34},  // 4
    {3, 1, 2.0},   // 5
    {3, 2, 1.34},  // 6
    {1, 1, 0.0},   // 7
    {1, 2, 1.34},  // 8
    {2, 2, 0.0},   // 9
    {4, 4, 0.0},   // 10: eight-wave tiles from here on
    {4, 6, 1.34},  // 11
    {4, 5, 1.34},  // 12
    {5, 5, 0.0},   // 13
    {5, 6, 1.34},  // 14
    {6, 6, 0.0},   // 15
    {4, 4, 0.0, 1},   // 16: one launch per dependency level from here on
    {4, 6, 1.34, 1},  // 17
    {4, 5, 1.34, 1},  // 18
    {3, 1, 1.34, 1},  // 19
    {6, 6, 0.0, 1},   // 20
    {4, 4, 0.0, 2},   // 21: pipelined segments from here on
    {4, 5, 1.34, 2},  // 22
    {4, 6, 1.34, 2},  // 23
    {3, 1, 1.34, 2},  // 24
    {4, 4, 0.0, 1, 1},   // 25: FP32 operands read directly (BF16) from here on
    {4, 5, 1.34, 1, 1},  // 26
    {4, 6, 1.34, 1, 1},  // 27
    {3, 1, 1.34, 1, 1},  // 28
    {4, 4, 0.0, 0, 1},   // 29: in-kernel waits
    {4, 5, 1.34, 0, 1},  // 30
    {4, 4, 0.0, 2, 1},   // 31: pipelined segments
    {4, 6, 1.34, 2, 1},  // 32
    {4, 5, 1.34, 2, 1},  // 33
    {4, 6, 0.0, 2, 1},   // 34: independent problems on the large tile, problems with
    {4, 5, 0.0, 2, 1},   // 35:   producers (a chain's later levels) on the small one
    {2, 2, 0.0, 0, 1},   // 36: small tiles for lists that would leave CUs idle on large ones,
    {6, 6, 0.0, 0, 1},   // 37:   in one kernel
    {2, 2, 0.0, 1, 1},   // 38:   and one launch per level
    {6, 6, 0.0, 1, 1},   // 39
};
constexpr int kPolicyCount = sizeof(kPolicies) / sizeof(kPolicies[0]);

// Relative per-CU contraction rate of each tile configuration on large
// problems (larger tiles reuse each loaded panel more), used by the list
// schedule's tile times (tile_ms).
constexpr double kTileRate[7] = {1.0, 0.6, 0.2, 0.85, 1.15, 0.95, 0.65};

// The configuration a grouped launch of `prec` runs for configuration c.
int grouped_config(mfx_precision prec, int c) { return prec == MFX_PREC_FP32 && c == 0 ? 3 : c; }

int problem_config(const GroupedPolicy& pol, mfx_precision prec, int64_t m, int64_t n) {
  const int big = grouped_config(prec, pol.big), small = grouped_config(prec, pol.small);
  if(big == small || pol.bound <= 0.0) return big;
  const double padded = (double)round_up(m, cfg_bm(big)) * (double)round_up(n, cfg_bn(big));
  return padded <= pol.bound * (double)m * (double)n ? big : small;
}

// Topological level of every problem. Producers come first in `problems`, so one
// pass in consumer order; the pairs are sorted only where the caller's are not.
std::vector<int> problem_levels(int count, const mfx_dep* deps, int ndeps) {
  std::vector<int> level(count, 0);
  auto by_consumer = [](const mfx_dep& a, const mfx_dep& b) { return a.consumer < b.consumer; };
  std::vector<mfx_dep> sorted;
  if(!std::is_sorted(deps, deps + ndeps, by_consumer)) {
    sorted.assign(deps, deps + ndeps);
    std::sort(sorted.begin(), sorted.end(), by_consumer);
    deps = sorted.data();
  }
  for(int d = 0; d < ndeps; ++d) level[deps[d].consumer] = std::max(level[deps[d].consumer], level[deps[d].producer] + 1);
  return level;
}

// Tile configuration of every problem under a policy: the padding rule,
// then, on a dependency level whose tiles would not give every CU one, the
// small tile for all of the level's problems (a chain's later levels hold
// few problems, and a level cannot overlap the next).
std::vector<int> assign_configs(const GroupedPolicy& pol, mfx_precision prec, const mfx_gemm_problem* problems,
    int count, const std::vector<int>& level, int cus) {
  std::vector<int> cfg(count);
  for(int i = 0; i < count; ++i) cfg[i] = problem_config(pol, prec, problems[i].m, problems[i].n);
  const int small = grouped_config(prec, pol.small);
  if(grouped_config(prec, pol.big) == small) return cfg;
  const int levels = count ? *std::max_element(level.begin(), level.end()) + 1 : 0;
  std::vector<int64_t> tiles(levels, 0);
  for(int i = 0; i < count; ++i)
    if(problems[i].m > 0 && problems[i].n > 0)
      tiles[level[i]] += ceil_div(problems[i].m, cfg_bm(cfg[i])) * ceil_div(problems[i].n, cfg_bn(cfg[i]));
  for(int i = 0; i < count; ++i)
    if(level[i] > 0 && tiles[level[i]] < cus) cfg[i] = small;
  return cfg;
}

// Microseconds of one tile of a grouped kernel: fixed + K * ns per k, the
// latter between `idle` (a quarter of the CUs busy) and `full` (all of them),
// by precision and configuration, measured on MI355X at K = 512 and 2048.
// `full` lies between one-tile problems, whose panels all come from HBM (split
// BF16 256x256: 165, 128x128: 60), and the tiles of one large problem, which
// share them in L2 (110, 36).
struct GroupedTileCost {
  double fixed, idle, full;
};
constexpr GroupedTileCost kGroupedF32[7] = {{10.0, 228.0, 240.0}, {6.0, 71.0, 80.0},    {4.0, 23.3, 23.5}, {8.0, 120.0, 138.0},
                                            {10.0, 228.0, 240.0}, {8.0, 117.0, 135.0}, {6.0, 68.0, 78.0}};
constexpr GroupedTileCost kGroupedSplit[7] = {{10.0, 100.0, 160.0}, {6.0, 38.0, 48.0},  {5.0, 27.0, 27.0}, {8.0, 62.0, 90.0},
                                              {10.0, 84.0, 140.0}, {8.0, 60.0, 85.0}, {4.0, 35.5, 46.0}};
constexpr GroupedTileCost kGroupedBf16[7] = {{10.0, 70.0, 95.0}, {6.0, 27.0, 40.0}, {5.0, 17.0, 17.5}, {8.0, 42.0, 62.0},
                                             {10.0, 55.0, 80.0}, {8.0, 40.0, 58.0}, {4.0, 25.0, 38.0}};

double ns_per_k(const GroupedTileCost& t, double busy) {  // busy: tiles per CU
  return t.idle + (t.full - t.idle) * std::min(1.0, std::max(0.0, (busy - 0.25) / 0.75));
}
const GroupedTileCost& tile_cost(mfx_precision prec, int c) {
  return prec == MFX_PREC_FP32 ? kGroupedF32[c] : prec == MFX_PREC_SPLIT_BF16 ? kGroupedSplit[c] : kGroupedBf16[c];
}
// Single BF16 64x64 tiles of packed problems fall behind 128x128 ones from
// about K = 256 on: in one kernel eight chained products of 200 take 52 and 51
// us, of 363 87 and 73.
constexpr double kPackedSmallUs = 5.0;
bool packed_small(mfx_precision prec, int64_t k) { return prec == MFX_PREC_BF16 && k % 16 != 0 && k >= 256; }

// The tiles that some problems take on one configuration: what their estimate
// needs of them, so that no estimate walks the problems again.
struct TileSums {
  int64_t tiles = 0, packed = 0;  // packed: of problems with packed_small
  double tiles_k = 0.0;           // K summed over the tiles
  double kmin[2], kmax[2] = {-1.0, -1.0};  // of problems without and with packed_small
  void add(int64_t n, double k, bool slow) {
    kmin[slow] = kmax[slow] < 0.0 ? k : std::min(kmin[slow], k);
    kmax[slow] = std::max(kmax[slow], k);
    tiles += n;
    packed += slow ? n : 0;
    tiles_k += k * (double)n;
  }
  void add(const TileSums& o) {
    for(int s = 0; s < 2; ++s) {
      if(o.kmax[s] < 0.0) continue;
      kmin[s] = kmax[s] < 0.0 ? o.kmin[s] : std::min(kmin[s], o.kmin[s]);
      kmax[s] = std::max(kmax[s], o.kmax[s]);
    }
    tiles += o.tiles;
    packed += o.packed;
    tiles_k += o.tiles_k;
  }
};

// Microseconds of all of these tiles on one CU, and of the longest and shortest
// one (kept where `longest` / `shortest` are beyond it already).
double sum_us(mfx_precision prec, int c, const TileSums& t, double busy, double* longest, double* shortest) {
  if(t.tiles == 0) return 0.0;
  const GroupedTileCost& cost = tile_cost(prec, c);
  const double ns = ns_per_k(cost, busy), slow = c == 2 ? kPackedSmallUs : 0.0;
  for(int s = 0; s < 2; ++s) {
    if(t.kmax[s] < 0.0) continue;
    const double fixed = cost.fixed + (s ? slow : 0.0);
    *longest = std::max(*longest, fixed + 1e-3 * ns * t.kmax[s]);
    *shortest = *shortest < 0.0 ? fixed + 1e-3 * ns * t.kmin[s] : std::min(*shortest, fixed + 1e-3 * ns * t.kmin[s]);
  }
  return cost.fixed * (double)t.tiles + slow * (double)t.packed + 1e-3 * ns * t.tiles_k;
}

// Estimated microseconds of one level's tiles on configuration a, and b: whole
// rounds over the CUs where all tiles are alike, else the work spread over the
// CUs plus a quarter of the longest tile.
double level_estimate(mfx_precision prec, int a, const TileSums& ta, int b, const TileSums& tb, int cus) {
  const int64_t tiles = ta.tiles + tb.tiles;
  if(tiles == 0) return 0.0;
  double longest = 0.0, shortest = -1.0;
  const double busy = (double)tiles / cus;
  const double work = sum_us(prec, a, ta, busy, &longest, &shortest) + sum_us(prec, b, tb, busy, &longest, &shortest);
  if(longest <= shortest * 1.001) return (double)ceil_div(tiles, cus) * longest;
  return std::max(longest, work / cus + 0.25 * longest);
}

// Tile shapes, and the shape of each configuration.
constexpr int kShapes = 4, kShapeBm[kShapes] = {256, 128, 64, 256}, kShapeBn[kShapes] = {256, 128, 64, 128};
constexpr int kShapeOf[7] = {0, 1, 2, 3, 0, 3, 1};

// A problem list as the estimates see it, gathered in one pass: choosing among
// the policies of a list took four times as long as planning the chosen one
// while each walked the problems for every level and configuration (519
// problems, FP32: 1.07 ms, against 0.26 for the whole plan now; 1000 problems
// in a row 65 ms).
struct ListSummary {
  mfx_precision prec;
  const mfx_gemm_problem* problems;
  int count, levels = 0, cus;
  std::vector<int> level;
  bool lone = false;      // problems with producers or consumers hold more than half of the work
  bool slow_wait = false; // a problem with producers or consumers has its operands packed
  double first_k = 0.0;   // longest K of the first level's problems with consumers
  std::vector<std::array<TileSums, kShapes>> all;  // per level: every problem on one shape
  std::vector<int> best;        // per level: the configuration estimated shortest for all of its problems
  std::vector<double> best_us;  // and that estimate

  ListSummary(mfx_precision p, const mfx_gemm_problem* q, int n, const mfx_dep* deps, int ndeps, int cu)
      : prec(p), problems(q), count(n), cus(cu), level(problem_levels(n, deps, ndeps)) {
    if(count > 0) levels = *std::max_element(level.begin(), level.end()) + 1;
  }

  // the sum of the levels is part of one kernel's estimate
  bool summed() const { return lone && levels > 1 && prec != MFX_PREC_FP32; }

  void gather(const mfx_dep* deps, int ndeps) {
    std::vector<char> linked(count, 0);
    for(int d = 0; d < ndeps; ++d) linked[deps[d].consumer] = linked[deps[d].producer] = 1;
    double free_work = 0.0, all_work = 0.0;
    all.resize(levels);
    for(int i = 0; i < count; ++i) {
      const mfx_gemm_problem& q = problems[i];
      const double w = (double)q.m * q.n * q.k;
      all_work += w;
      if(!linked[i]) free_work += w;
      slow_wait = slow_wait || (linked[i] && prec != MFX_PREC_FP32 && q.k % 16 != 0);
      if(q.m <= 0 || q.n <= 0) continue;
      const double k = (double)std::max<int64_t>(q.k, 1);
      if(linked[i] && level[i] == 0) first_k = std::max(first_k, k);
      const bool slow = packed_small(prec, q.k);
      for(int s = 0; s < kShapes; ++s) all[level[i]][s].add(tiles(i, s), k, slow);
    }
    lone = free_work < 0.5 * all_work;
    best.assign(levels, -1);
    best_us.assign(levels, 0.0);
    for(int l = 0; l < levels; ++l)
      for(int c = 0; c < 7; ++c) {
        if(grouped_config(prec, c) != c) continue;
        const double t = uniform(l, c);
        if(best[l] < 0 || t < best_us[l]) {
          best[l] = c;
          best_us[l] = t;
        }
      }
  }

  int64_t tiles(int i, int shape) const {  // the sides are powers of two
    const mfx_gemm_problem& q = problems[i];
    const int bm = kShapeBm[shape] == 256 ? 8 : kShapeBm[shape] == 128 ? 7 : 6;
    const int bn = kShapeBn[shape] == 256 ? 8 : kShapeBn[shape] == 128 ? 7 : 6;
    return ((q.m + kShapeBm[shape] - 1) >> bm) * ((q.n + kShapeBn[shape] - 1) >> bn);
  }

  double uniform(int l, int c) const { return level_estimate(prec, c, all[l][kShapeOf[c]], c, TileSums{}, cus); }

  // The tiles of each level on the large and the small configuration of `pol`,
  // as assign_configs gives them out: one pass for all policies of the same
  // shapes and bound.
  using Assigned = std::vector<std::array<TileSums, 2>>;
  struct Sharing {
    int sb, ss;
    double bound;
    Assigned sums;
  };
  std::vector<std::unique_ptr<Sharing>> known;

  const Assigned& assigned(const GroupedPolicy& pol) {
    const int sb = kShapeOf[grouped_config(prec, pol.big)], ss = kShapeOf[grouped_config(prec, pol.small)];
    for(const auto& k : known)
      if(k->sb == sb && k->ss == ss && (k->bound == pol.bound || sb == ss)) return k->sums;
    known.emplace_back(new Sharing{sb, ss, pol.bound, Assigned(levels)});
    Assigned& sums = known.back()->sums;
    if(sb == ss || pol.bound <= 0.0) {
      for(int l = 0; l < levels; ++l) sums[l][0] = all[l][sb];
    } else {
      const double area = (double)kShapeBm[sb] * kShapeBn[sb];
      for(int i = 0; i < count; ++i) {
        const mfx_gemm_problem& q = problems[i];
        if(q.m <= 0 || q.n <= 0) continue;
        const int64_t n = tiles(i, sb);
        const bool is_big = area * (double)n <= pol.bound * (double)q.m * (double)q.n;
        sums[level[i]][is_big ? 0 : 1].add(is_big ? n : tiles(i, ss), (double)std::max<int64_t>(q.k, 1),
            packed_small(prec, q.k));
      }
    }
    if(sb != ss)
      for(int l = 1; l < levels; ++l)
        if(sums[l][0].tiles + sums[l][1].tiles < cus) {
          sums[l][0] = TileSums{};
          sums[l][1] = all[l][ss];
        }
    return sums;
  }
};

// What a further dependency level costs beyond its tiles: a launch of its own
// (item fetches from cold queues, a drained pipeline), or in one kernel the
// publication and the wait. In a chain without other problems to fill the wait
// it depends on the tile and on packing: nearly nothing beyond the publication
// on 128x128 tiles read directly, but 12 us on 64x64 tiles, whose second
// workgroup per CU polls beside the first, and more where a level packs its
// operands first (split BF16, eight chained products of 512: 87 us on 128x128
// tiles in one kernel, 100 in a launch per level, 111 on 64x64 tiles in one kernel).
constexpr double kLevelLaunchUs = 16.0, kLevelWaitUs = 8.0, kLoneLevelWaitUs = 6.0, kSlowLevelWaitUs = 20.0;

// Estimated microseconds of a launch under a policy.  One launch per level:
// the levels' sum.  One kernel: all work spread over the CUs, or the chain of
// the levels' longest tiles where that is longer. For a BF16 chain that holds
// most of the work, the mean of this and the levels' sum: little else fills a
// level's last round of tiles, but the next level's products whose producers are
// done do (spread alone, eight chained products of 768 beside thirty small
// problems were estimated at 95 us on 64x64 tiles, single BF16, and took 211; 87
// on 128x128; the sum alone slows chains with many rounds a level, split BF16,
// eight of 1616 beside twenty 376 -> 417). FP32 chains keep the spread: summed,
// some were chosen better (eight of 768 195 -> 122 us), others worse (sixteen of
// 400 101 -> 134, thirty-two of 768 367 -> 475), as launches per level are
// estimated low.
// BF16 tiles of 64x64 run two workgroups to a CU, which take turns: with more
// tiles than CUs a tile of the chain takes up to twice its time (split BF16, four
// chained products of 384 beside thirty small problems: estimated at 43 us
// without that, 77 measured; 52 on 128x128 tiles).
double policy_estimate(const GroupedPolicy& pol, ListSummary& list) {
  const mfx_precision prec = list.prec;
  const int big = grouped_config(prec, pol.big), small = grouped_config(prec, pol.small), cus = list.cus;
  const auto& sums = list.assigned(pol);
  if(pol.per_level == 1 && list.levels > 1) {
    double est = kLevelLaunchUs * (list.levels - 1);
    for(int l = 0; l < list.levels; ++l)
      est += std::min(level_estimate(prec, big, sums[l][0], small, sums[l][1], cus), list.best_us[l]);
    return est;
  }
  if(list.levels == 1) return level_estimate(prec, big, sums[0][0], small, sums[0][1], cus);
  const bool slow = pol.small == 2 || list.slow_wait;
  const double wait = !list.lone ? kLevelWaitUs : slow ? kSlowLevelWaitUs : kLoneLevelWaitUs;
  TileSums total[2];
  for(const auto& s : sums) {
    total[0].add(s[0]);
    total[1].add(s[1]);
  }
  const double busy = (double)(total[0].tiles + total[1].tiles) / cus;
  double last = 0.0, any = -1.0;
  const double work = sum_us(prec, big, total[0], busy, &last, &any) + sum_us(prec, small, total[1], busy, &last, &any);
  double path = wait * (list.levels - 1);
  // the first level's linked problems are as long as the longest tile at most
  path += last;
  const double share = prec != MFX_PREC_FP32 && pol.big == 2 && pol.small == 2 ? std::min(2.0, std::max(1.0, busy)) : 1.0;
  path += (share - 1.0) * (tile_cost(prec, 2).fixed + 1e-3 * ns_per_k(tile_cost(prec, 2), busy) * list.first_k);
  for(int l = 1; l < list.levels; ++l) {
    double longest = 0.0;
    sum_us(prec, big, sums[l][0], busy, &longest, &any);
    sum_us(prec, small, sums[l][1], busy, &longest, &any);
    path += share * longest;
  }
  const double spread = std::max(work / cus + 0.25 * last, path);
  if(!list.summed()) return spread;
  double summed = wait * (list.levels - 1);
  for(const auto& l : sums) summed += level_estimate(prec, big, l[0], small, l[1], cus);
  return 0.5 * (spread + summed);
}

// Policies that run the same launch for `prec`: FP32 has no direct form, and one
// tile for two configurations (grouped_config).
bool same_launch(mfx_precision prec, const GroupedPolicy& a, const GroupedPolicy& b) {
  return grouped_config(prec, a.big) == grouped_config(prec, b.big) && grouped_config(prec, a.small) == grouped_config(prec, b.small) &&
         a.bound == b.bound && a.per_level == b.per_level && (prec == MFX_PREC_FP32 || a.direct == b.direct);
}

}  // namespace

int grouped_policy_count() { return kPolicyCount; }

bool grouped_policy_direct(int id) { return id >= 0 && id < kPolicyCount && kPolicies[id].direct; }

bool grouped_policy_info(int id, int* big, int* small, double* bound, int* per_level) {
  if(id < 0 || id >= kPolicyCount) return false;
  *big = kPolicies[id].big;
  *small = kPolicies[id].small;
  *bound = kPolicies[id].bound;
  *per_level = kPolicies[id].per_level;
  return true;
}

// Tuning-table key of a grouped launch: precision, problem count, total
// contraction volume and dependency depth, each bucketed by powers of two.
std::string grouped_tune_key(mfx_precision p, const mfx_gemm_problem* problems, int count, const mfx_dep* deps,
    int ndeps) {
  double vol = 0.0;
  for(int i = 0; i < count; ++i) vol += (double)problems[i].m * problems[i].n * problems[i].k;
  const auto level = problem_levels(count, deps, ndeps);
  const int levels = count ? *std::max_element(level.begin(), level.end()) + 1 : 0;
  return "g" + tune_key(p, count, (int64_t)std::min(std::sqrt(vol), 1e18), levels);
}

// Policy of a grouped launch: the tuner's override, a forced configuration,
// a tuned entry, or the estimate.
// *us: the estimate, where the policy is not forced or tuned (-1).  *dense: the
// table says that dense launches were faster than any policy.
static int choose_grouped_policy(Handle* h, ListSummary& list, const mfx_dep* deps, int ndeps, double* us, bool* dense) {
  const mfx_precision prec = list.prec;
  *us = -1.0;
  *dense = false;
  if(h->grouped_policy >= 0) return h->grouped_policy;
  int forced = h->forced_config[prec];
  if(forced >= 0) {
    for(int i = 0; i < kPolicyCount; ++i)
      if(kPolicies[i].big == forced && kPolicies[i].small == forced && !kPolicies[i].per_level) return i;
  }
  const int tuned = tuned_any() ? tuned_lookup(grouped_tune_key(prec, list.problems, list.count, deps, ndeps)) : -1;
  if(tuned >= 0 && tuned < kPolicyCount) return tuned;
  *dense = tuned == kDenseListPolicy;
  // With dependency levels: one launch per level, or one kernel with in-kernel
  // waits, whose list-schedule order fills a chain's later levels' idle CUs
  // with other problems' tiles, by estimate.  Measured on MI355X: a lone 8-long
  // 2048^2 chain (split BF16) 0.45 ms per level against 0.66 ms in one kernel;
  // 30 problems of 128 to 1024 beside a chain of four 512^2 (single BF16) 46 us
  // in one kernel against 68 us per level.
  list.gather(deps, ndeps);
  int best = 0;
  for(int i = 0; i < kPolicyCount; ++i) {
    // without levels the two modes are the same launch
    if(kPolicies[i].per_level == 2 || (list.levels <= 1 && kPolicies[i].per_level == 1)) continue;
    // BF16: the direct tiles (no packing pass; measured 1.3x faster on the
    // batched workload); FP32 has nothing to pack
    if(prec != MFX_PREC_FP32 && !kPolicies[i].direct) continue;
    bool seen = false;
    for(int j = 0; j < i && !seen; ++j) seen = same_launch(prec, kPolicies[i], kPolicies[j]);
    if(seen) continue;
    const double e = policy_estimate(kPolicies[i], list);
    if(*us < 0 || e < *us) {
      *us = e;
      best = i;
    }
  }
  return best;
}

namespace {

// Clears the queue counters and the error flag before each launch (a kernel,
// so the reset can be part of a captured graph).
__global__ void zero_ints_kernel(int* p, int n, int* err) {
  for(int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0;
  if(blockIdx.x == 0 && threadIdx.x == 0) *err = 0;
}

// Bytes of the packed A and B copies of one problem (each rounded to 256).
std::pair<size_t, size_t> packed_sizes(const GProblem& P, int nhl) {
  const size_t ba = (size_t)round_up(P.M, 32) * P.kbs * 16 * nhl * 2;
  const size_t bb = (size_t)round_up(P.N, 32) * P.kbs * 16 * nhl * 2;
  return {(size_t)round_up(ba, 256), (size_t)round_up(bb, 256)};
}

}  // namespace

static mfx_status validate(mfx_precision prec, const mfx_gemm_problem* problems, int count, const mfx_dep* deps,
    int ndeps) {
  if(count < 0 || ndeps < 0) return invalid("negative problem or dependency count");
  if(count > 0 && !problems) return invalid("null problem list");
  if(ndeps > 0 && !deps) return invalid("null dependency list");
  for(int i = 0; i < count; ++i) {
    const auto& q = problems[i];
    if(q.m < 0 || q.n < 0 || q.k < 0 || q.m > (1 << 30) || q.n > (1 << 30) || q.k > (1 << 30))
      return invalid("problem " + std::to_string(i) + ": bad dimensions");
    if((q.transA != 0 && q.transA != 1) || (q.transB != 0 && q.transB != 1))
      return invalid("problem " + std::to_string(i) + ": transA / transB must be 0 or 1");
    const int64_t a_cols = q.transA ? q.m : q.k;
    const int64_t b_cols = q.transB ? q.k : q.n;
    if(q.m > 0 && q.n > 0) {
      if(prec != MFX_PREC_FP32 && !bf16_k_supported(q.k, prec == MFX_PREC_SPLIT_BF16 ? 2 : 1))
        return unsupported("problem " + std::to_string(i) + ": K is beyond the packed BF16 path's limit");
      if(!q.C || q.ldc < std::max<int64_t>(1, q.n)) return invalid("problem " + std::to_string(i) + ": bad C");
      if(q.k > 0 && (!q.A || !q.B)) return invalid("problem " + std::to_string(i) + ": null operand");
      if(q.lda < std::max<int64_t>(1, a_cols) || q.ldb < std::max<int64_t>(1, b_cols))
        return invalid("problem " + std::to_string(i) + ": leading dimension smaller than row length");
    }
  }
  for(int d = 0; d < ndeps; ++d) {
    if(deps[d].consumer < 0 || deps[d].consumer >= count || deps[d].producer < 0 || deps[d].producer >= count)
      return invalid("dependency " + std::to_string(d) + " names a problem out of range");
    if(deps[d].producer >= deps[d].consumer)
      return invalid("dependency " + std::to_string(d) + ": producers must come before their consumers");
  }
  return MFX_SUCCESS;
}

namespace {

// Cost model of the pipelined planner, in milliseconds, fitted to MI355X
// measurements of split-BF16 grouped launches: a tile of configuration c
// takes about kTileFixedMs + kTileMsPerUnit * bm * bn * K / kTileRate[c]
// (the 256x256 eight-wave tile at K = 2048: 0.2 ms under full load, with
// its panels streamed from HBM; the 512 uneven problems: 1.0 ms); the
// pre-pass packs kPrepassMsPerElem per operand element over the whole chip
// (0.53 ms for 361 M elements), and a pre-pack item costs one CU about
// kPrepackCuMsPerElem per element (the CU reads 4 and writes 4 bytes); and
// a launch moves at most kHbmBytesPerMs.
constexpr double kTileFixedMs = 0.005, kTileMsPerUnit = 1.67e-9;
constexpr double kPrepassMsPerElem = 1.47e-9, kPrepackCuMsPerElem = 1.0e-7, kHbmBytesPerMs = 5.0e9;
constexpr int kMinPipelineSegments = 3;
constexpr int PREPACK_BLOCKS = 32;  // 256-chunk blocks per pre-pack item (256 KiB of FP32 source)

double tile_ms(int c, int64_t k) {
  return kTileFixedMs + kTileMsPerUnit * cfg_bm(c) * cfg_bn(c) * (double)round_up(std::max<int64_t>(k, 1), 32) /
                            kTileRate[c];
}

// Pipelined segments.  Problems with producers or consumers keep their
// dependency level; every other problem goes, largest first, to the segment
// where it adds least to the estimated total time.  A segment's launch takes
// the longest of: its tile work plus the pre-pack items it runs for the next
// segment, spread over the CUs; its longest tile; its HBM traffic (each
// problem's packed operands read once -- its tiles share one XCD's L2 -- and
// C written, plus 4 + 2 * planes bytes per pre-packed element).  Its
// pre-pass comes on top: segment 0's packs all of its problems, a later
// one only those with producers; the others were packed by the previous
// segment's launch.
std::vector<int> balance_segments(const std::vector<GProblem>& P, const std::vector<char>& has_prod,
    const std::vector<char>& linked, const std::vector<int>& level, int cus, int nhl, int* nseg_out) {
  const bool packed = nhl > 0;
  const int count = (int)P.size();
  int nseg = 1;
  for(int i = 0; i < count; ++i) nseg = std::max(nseg, level[i] + 1);
  bool any_free = false;
  for(int i = 0; i < count; ++i) any_free = any_free || (!linked[i] && P[i].tiles_m * P[i].tiles_n > 0);
  if(any_free) nseg = std::max(nseg, kMinPipelineSegments);
  std::vector<double> work(nseg, 0.0), tmax(nseg, 0.0), prepass(nseg, 0.0), prepack(nseg, 0.0), bytes(nseg, 0.0);
  std::vector<int> seg(count, 0);
  auto elems = [&](int i) { return packed ? (double)(round_up(P[i].M, 32) + round_up(P[i].N, 32)) * P[i].kbs * 16 : 0.0; };
  auto add = [&](int i, int s, double sign) {
    const int tiles = P[i].tiles_m * P[i].tiles_n;
    if(tiles == 0) return;
    const double t = tile_ms(P[i].config, P[i].K);
    work[s] += sign * t * tiles;
    if(sign > 0) tmax[s] = std::max(tmax[s], t);
    const double e = elems(i);
    bytes[s] += sign * (e * 2 * std::max(nhl, 2) + (P[i].beta != 0.0f ? 8.0 : 4.0) * P[i].M * P[i].N);
    if(s == 0 || has_prod[i]) {
      prepass[s] += sign * e * kPrepassMsPerElem;
    } else {
      prepack[s - 1] += sign * e * kPrepackCuMsPerElem;
      bytes[s - 1] += sign * e * (4 + 2 * nhl);
    }
  };
  auto total = [&]() {
    double t = 0.0;
    for(int s = 0; s < nseg; ++s)
      t += std::max(std::max((work[s] + prepack[s]) / cus, tmax[s]), bytes[s] / kHbmBytesPerMs) + prepass[s];
    return t;
  };
  std::vector<int> free_list;
  for(int i = 0; i < count; ++i) {
    if(linked[i]) {
      seg[i] = level[i];
      add(i, seg[i], 1.0);
    } else if(P[i].tiles_m * P[i].tiles_n > 0) {
      free_list.push_back(i);
    }
  }
  std::stable_sort(free_list.begin(), free_list.end(), [&](int a, int b) {
    return tile_ms(P[a].config, P[a].K) * P[a].tiles_m * P[a].tiles_n >
           tile_ms(P[b].config, P[b].K) * P[b].tiles_m * P[b].tiles_n;
  });
  for(int i : free_list) {
    int best = 0;
    double best_t = -1.0;
    for(int s = 0; s < nseg; ++s) {
      const std::vector<double> keep = tmax;
      add(i, s, 1.0);
      const double t = total();
      add(i, s, -1.0);
      tmax = keep;
      if(best_t < 0 || t < best_t - 1e-12) {
        best_t = t;
        best = s;
      }
    }
    seg[i] = best;
    add(i, best, 1.0);
  }
  *nseg_out = nseg;
  return seg;
}

// Queue order of the one-kernel (in-kernel waits) mode when no problem has
// pack items: a list schedule of every tile on `workers` workgroups.  The
// next free workgroup takes a tile of the ready problem with the longest
// remaining path to the end of the launch (its tile time plus its longest
// consumer's, tile_ms estimates), ties to the larger K; a problem is ready
// once its producers' tiles are scheduled to have ended.  So a chain's
// later levels are queued as soon as their inputs are due, and the
// independent problems fill the time around them, instead of every later
// level waiting behind all first-level tiles.  A consumer's tiles follow all
// of its producers' tiles in the list, so the order stays a topological
// one: a workgroup that waits in-kernel only waits for tiles that other
// workgroups have already taken.  Producers have lower indices than their
// consumers (checked by validate).
std::vector<GItem> critical_path_items(const std::vector<int>& at, const std::vector<GProblem>& P, int workers) {
  const int count = (int)P.size();
  std::vector<char> in(count, 0);
  for(int i : at) in[i] = 1;
  std::vector<std::vector<int>> cons(count);
  std::vector<int> wait_for(count, 0);
  for(int i : at)
    for(int e = 0; e < P[i].ndeps; ++e)
      if(in[P[i].deps[e]]) {
        cons[P[i].deps[e]].push_back(i);
        ++wait_for[i];
      }
  std::vector<double> dur(count, 0.0), path(count, 0.0);
  for(int i : at) dur[i] = tile_ms(P[i].config, P[i].K);
  for(int i = count - 1; i >= 0; --i) {
    if(!in[i]) continue;
    double longest = 0.0;
    for(int c : cons[i]) longest = std::max(longest, path[c]);
    path[i] = dur[i] + longest;
  }
  auto lower = [&](int a, int b) {  // a goes after b
    if(path[a] != path[b]) return path[a] < path[b];
    if(P[a].K != P[b].K) return P[a].K < P[b].K;
    return a > b;
  };
  std::priority_queue<int, std::vector<int>, decltype(lower)> ready(lower);
  using Due = std::pair<double, int>;  // (time its inputs are due, problem)
  std::priority_queue<Due, std::vector<Due>, std::greater<Due>> pending;
  std::vector<double> due(count, 0.0), finish(count, 0.0);
  std::vector<int> next(count, 0);
  for(int i : at)
    if(wait_for[i] == 0) pending.push({0.0, i});
  // workgroups that are free from the same time on, taken together: a problem's
  // tiles are all alike, so they hand it out as one by one
  using Free = std::pair<double, int>;  // (time, workgroups)
  std::priority_queue<Free, std::vector<Free>, std::greater<Free>> free_at;
  free_at.push({0.0, std::max(1, workers)});
  std::vector<GItem> out;
  size_t total = 0;
  for(int i : at) total += (size_t)P[i].tiles_m * P[i].tiles_n;
  out.reserve(total);
  auto take = [&](int p, int n) {  // the next n tiles of problem p
    for(int tm = next[p] / P[p].tiles_n, tn = next[p] % P[p].tiles_n, i = 0; i < n; ++i) {
      out.push_back({ITEM_TILE, p, tm, tn});
      if(++tn == P[p].tiles_n) {
        tn = 0;
        ++tm;
      }
    }
    next[p] += n;
  };
  size_t to_come = at.size();  // problems that have not become ready
  auto arrives = [&] {
    ready.push(pending.top().second);
    pending.pop();
    --to_come;
  };
  while(to_come > 0) {
    double t = free_at.top().first;
    int group = free_at.top().second;
    free_at.pop();
    while(!pending.empty() && pending.top().first <= t) arrives();
    if(ready.empty()) {  // nothing due yet: one workgroup waits for the earliest
      if(group > 1) free_at.push({t, group - 1});
      group = 1;
      t = pending.top().first;
      arrives();
    }
    const int p = ready.top(), tiles = P[p].tiles_m * P[p].tiles_n;
    const int taken = std::min(group, tiles - next[p]);
    if(taken < group) free_at.push({t, group - taken});
    take(p, taken);
    finish[p] = std::max(finish[p], t + dur[p]);
    free_at.push({t + dur[p], taken});
    if(next[p] == tiles) {
      ready.pop();
      for(int c : cons[p]) {
        due[c] = std::max(due[c], finish[p]);
        if(--wait_for[c] == 0) pending.push({due[c], c});
      }
    }
  }
  // no further arrival can change the order, whatever the times
  for(; !ready.empty(); ready.pop()) take(ready.top(), P[ready.top()].tiles_m * P[ready.top()].tiles_n - next[ready.top()]);
  return out;
}

// Tiles of one problem that go to one queue: at most one round of an XCD's
// CUs (kQueueGroupTiles), whole tile rows where possible, so the group's
// tiles share their A panels (and B panels) in that XCD's L2.
constexpr int kQueueGroupTiles = 32;
struct TileGroup {
  int problem, first, count;  // tiles [first, first + count) in row-major tile order
};

// Splits a problem list over the GROUPED_QUEUES queues: each problem's tiles
// in groups of at most kQueueGroupTiles, groups by decreasing work to the
// least-loaded queue; a queue lists its groups in the order of `order`
// (largest K first), so long tiles start first everywhere.
std::vector<std::vector<TileGroup>> queue_tiles(const std::vector<int>& order, const std::vector<GProblem>& P) {
  std::vector<TileGroup> groups;
  std::vector<int> rank(P.size(), 0);
  for(size_t r = 0; r < order.size(); ++r) rank[order[r]] = (int)r;
  for(int i : order) {
    const int tiles = P[i].tiles_m * P[i].tiles_n;
    const int per = std::min(tiles, kQueueGroupTiles);
    const int ng = (tiles + per - 1) / per;
    for(int g = 0; g < ng; ++g) {
      const int first = (int)((int64_t)tiles * g / ng), last = (int)((int64_t)tiles * (g + 1) / ng);
      groups.push_back({i, first, last - first});
    }
  }
  auto work = [&](const TileGroup& g) { return tile_ms(P[g.problem].config, P[g.problem].K) * g.count; };
  std::vector<int> by_work(groups.size());
  std::iota(by_work.begin(), by_work.end(), 0);
  std::stable_sort(by_work.begin(), by_work.end(), [&](int a, int b) { return work(groups[a]) > work(groups[b]); });
  std::vector<double> load(GROUPED_QUEUES, 0.0);
  std::vector<int> q_of(groups.size(), 0);
  for(int gi : by_work) {
    const int q = (int)(std::min_element(load.begin(), load.end()) - load.begin());
    q_of[gi] = q;
    load[q] += work(groups[gi]);
  }
  std::vector<std::vector<TileGroup>> qs(GROUPED_QUEUES);
  for(size_t gi = 0; gi < groups.size(); ++gi) qs[q_of[gi]].push_back(groups[gi]);  // groups are in `order`
  return qs;
}

PackJob make_job(const GProblem& P, bool is_a, int first_block) {
  PackJob j;
  j.src = make_pack_src(is_a ? P.A : P.B, is_a ? P.lda : P.ldb, is_a ? P.M : P.N, P.K, is_a ? P.a_kmajor : P.b_kmajor);
  j.dst = nullptr;  // bound to the workspace by bind_grouped
  j.kbs = P.kbs;
  j.chunks = ceil_div(is_a ? P.M : P.N, 32) * P.kbs * 64;
  j.blocks = (int)ceil_div(j.chunks, 256);
  j.first_block = first_block;
  return j;
}

}  // namespace

// The checks of a list, its dependencies and its policy: what is needed to tell
// whether it runs as dense launches, before any table is laid out.
static mfx_status choose_plan(Handle* h, mfx_precision prec, const mfx_gemm_problem* problems, int count,
    const mfx_dep* deps, int ndeps, GroupedPlan& pl, std::optional<ListSummary>& list) {
  if(prec != MFX_PREC_FP32 && prec != MFX_PREC_SPLIT_BF16 && prec != MFX_PREC_BF16)
    return unsupported("grouped launch supports FP32, SPLIT_BF16 and BF16");
  MFX_CHECK(validate(prec, problems, count, deps, ndeps));
  pl.prec = prec;
  pl.problems.resize(count);
  for(int i = 0; i < count; ++i) pl.problems[i].ndeps = pl.problems[i].consumed = 0;
  for(int d = 0; d < ndeps; ++d) {
    GProblem& c = pl.problems[deps[d].consumer];
    bool dup = false;
    for(int e = 0; e < c.ndeps; ++e) dup |= c.deps[e] == deps[d].producer;
    if(dup) continue;
    if(c.ndeps == GROUPED_MAX_DEPS) return unsupported("a problem may depend on at most 4 producers");
    c.deps[c.ndeps++] = deps[d].producer;
    pl.problems[deps[d].producer].consumed = 1;
  }
  list.emplace(prec, problems, count, deps, ndeps, cus_of(h));
  pl.policy = choose_grouped_policy(h, *list, deps, ndeps, &pl.estimate, &pl.tuned_dense);
  pl.summed = list->summed();
  return MFX_SUCCESS;
}

static void plan_tables(Handle* h, ListSummary& list, const mfx_dep* deps, int ndeps, GroupedPlan& pl) {
  const mfx_precision prec = pl.prec;
  const mfx_gemm_problem* problems = list.problems;
  const int count = list.count;
  const std::vector<int>& level = list.level;
  std::vector<char> has_prod(count), linked(count);
  for(int i = 0; i < count; ++i) {
    has_prod[i] = pl.problems[i].ndeps > 0;
    linked[i] = has_prod[i] || pl.problems[i].consumed;
  }
  const GroupedPolicy& pol = kPolicies[pl.policy];
  pl.big = grouped_config(prec, pol.big);
  pl.small = grouped_config(prec, pol.small);
  const int cus = cus_of(h);
  const bool packed = prec != MFX_PREC_FP32;
  const int nhl = prec == MFX_PREC_SPLIT_BF16 ? 2 : 1;
  const int max_level = count ? *std::max_element(level.begin(), level.end()) : 0;
  pl.pipelined = pol.per_level == 2;
  // One launch per segment: kernel boundaries order the segments, so no
  // problem waits or publishes in-kernel and every operand is packed by a
  // pre-pass or by the previous segment's pre-pack items.
  pl.per_level = (pol.per_level == 1 && max_level > 0) || pl.pipelined;
  std::vector<int> cfg(count);
  if(pl.pipelined) {
    // Problems with producers sit on the critical path of the segments (a
    // chain's later levels): they take the small tile, so each of their
    // segments is short and the independent problems fill it.
    for(int i = 0; i < count; ++i)
      cfg[i] = has_prod[i] ? pl.small : problem_config(pol, prec, problems[i].m, problems[i].n);
  } else {
    cfg = assign_configs(pol, prec, problems, count, level, cus);
  }
  // With a launch per level, a level may take one tile for all its problems,
  // in a kernel of its own tile pair, when that is estimated shorter than the
  // policy's pair: the later levels of a chain hold few problems, and all
  // levels of a chain of small matrices would leave CUs idle on large tiles.
  std::vector<int> level_cfg(max_level + 1, -1);
  if(pl.per_level && !pl.pipelined) {
    if(list.best.empty()) list.gather(deps, ndeps);  // a forced or tuned policy
    const auto& sums = list.assigned(pol);
    for(int lv = 0; lv <= max_level; ++lv) {
      const double as_is = level_estimate(prec, pl.big, sums[lv][0], pl.small, sums[lv][1], cus);
      if(list.best_us[lv] < 0.97 * as_is) level_cfg[lv] = list.best[lv];
    }
    for(int i = 0; i < count; ++i)
      if(level_cfg[level[i]] >= 0) cfg[i] = level_cfg[level[i]];
  }

  size_t packed_bytes = 0;
  int panels = 0;
  for(int i = 0; i < count; ++i) {
    const auto& q = problems[i];
    GProblem& P = pl.problems[i];
    P.M = (int)q.m;
    P.N = (int)q.n;
    P.K = (int)q.k;
    P.alpha = q.alpha;
    P.beta = q.beta;
    P.A = q.A;
    P.lda = q.lda;
    P.B = q.B;
    P.ldb = q.ldb;
    P.C = q.C;
    P.ldc = q.ldc;
    P.a_kmajor = q.transA == 0;
    P.b_kmajor = q.transB == 1;
    P.config = cfg[i];
    const int bm = cfg_bm(P.config), bn = cfg_bn(P.config);
    P.tiles_m = (int)ceil_div(q.m, bm);
    P.tiles_n = (int)ceil_div(q.n, bn);
    if(q.m == 0 || q.n == 0) P.tiles_m = P.tiles_n = 0;
    P.vec_a = f32_vec_ok(q.A, q.lda, P.a_kmajor, P.M, P.K);
    P.vec_b = f32_vec_ok(q.B, q.ldb, P.b_kmajor, P.N, P.K);
    if(P.tiles_m * P.tiles_n > 0) pl.all_vec = pl.all_vec && P.vec_a && P.vec_b;
    P.kbs = 0;
    P.pack_slices = 0;
    P.packed_a = P.packed_b = nullptr;
    P.pack_a_ctr = P.pack_b_ctr = 0;
    P.prepacked = 0;
    P.direct = packed && pol.direct && P.tiles_m * P.tiles_n > 0 && q.k % 16 == 0 &&
               direct_operand_ok(q.A, q.lda, P.M, P.a_kmajor) && direct_operand_ok(q.B, q.ldb, P.N, P.b_kmajor);
    if(P.direct) {
      P.prepacked = 1;  // nothing to pack: the tiles read A and B themselves
    } else if(packed && P.tiles_m * P.tiles_n > 0) {
      // load_chunk8 takes 128-bit loads along k only
      P.vec_a = P.a_kmajor && P.vec_a;
      P.vec_b = P.b_kmajor && P.vec_b;
      P.kbs = (int)(round_up(q.k, 16 * kb_per_stage_of(nhl)) / 16);
      P.pack_slices = (int)ceil_div(P.kbs, PACK_KBLOCKS);
      packed_bytes += packed_sizes(P, nhl).first + packed_sizes(P, nhl).second;
      if(P.ndeps == 0 || pl.per_level) {
        // packed by a pre-pass kernel or pre-pack items before the tiles start
        P.prepacked = 1;
      } else {
        P.pack_a_ctr = panels;
        panels += P.tiles_m;
        P.pack_b_ctr = panels;
        panels += P.tiles_n;
      }
    }
    pl.flops += 2.0 * q.m * q.n * q.k;
  }

  // Segment of every problem.
  int nseg = 1;
  std::vector<int> seg(count, 0);
  if(pl.pipelined) {
    seg = balance_segments(pl.problems, has_prod, linked, level, cus, packed ? nhl : 0, &nseg);
  } else if(pl.per_level) {
    seg = level;
    nseg = max_level + 1;
  }

  // Items segment by segment.  In-kernel mode (one segment): the level's
  // pack items (largest K first, so the first tiles' panels are ready first),
  // then its tiles, largest K first, a problem's tiles row by row, all in
  // queue 0.  Launch-per-segment modes: each problem's tiles in one XCD
  // queue, problems largest K first, with the segment's pre-pack items
  // spread evenly over the queues.
  std::vector<std::pair<int, int>> pre_ops, prepack_ops;  // (problem, is_a)
  std::vector<int> pre_seg_end, prepack_seg_end;
  pl.seg_items.assign(1, 0);
  for(int sg = 0; sg < nseg; ++sg) {
    std::vector<int> at;
    for(int i = 0; i < count; ++i)
      if(seg[i] == sg && pl.problems[i].tiles_m * pl.problems[i].tiles_n > 0) at.push_back(i);
    std::stable_sort(at.begin(), at.end(), [&](int a, int b) { return pl.problems[a].K > pl.problems[b].K; });
    // operands packed by this segment's pre-pass
    for(int i : at)
      if(pl.problems[i].prepacked && pl.problems[i].kbs > 0 && (!pl.pipelined || sg == 0 || has_prod[i])) {
        pre_ops.push_back({i, 1});
        pre_ops.push_back({i, 0});
      }
    pre_seg_end.push_back((int)pre_ops.size());
    // operands of the next segment packed by this segment's pre-pack items
    const int prepack_first = (int)prepack_ops.size();
    if(pl.pipelined && packed && sg + 1 < nseg)
      for(int i = 0; i < count; ++i)
        if(seg[i] == sg + 1 && !has_prod[i] && pl.problems[i].kbs > 0 && pl.problems[i].tiles_m * pl.problems[i].tiles_n > 0) {
          prepack_ops.push_back({i, 1});
          prepack_ops.push_back({i, 0});
        }
    prepack_seg_end.push_back((int)prepack_ops.size());
    const size_t first_item = pl.items.size();
    bool no_pack_items = true;
    for(int i : at) no_pack_items = no_pack_items && (!packed || pl.problems[i].prepacked);
    if(!pl.per_level && no_pack_items) {
      // one queue in list-schedule order
      const auto order = critical_path_items(at, pl.problems, cus);
      pl.items.insert(pl.items.end(), order.begin(), order.end());
      pl.qbeg.push_back(0);
      for(int q = 0; q < GROUPED_QUEUES; ++q) pl.qbeg.push_back((int)(pl.items.size() - first_item));
    } else if(!pl.per_level) {
      // one queue, dependency level by level (pack items before their level's tiles)
      for(int lv = 0; lv <= max_level; ++lv) {
        if(packed)
          for(int i : at) {
            const GProblem& P = pl.problems[i];
            if(level[i] != lv || P.prepacked) continue;
            for(int b = 0; b < (int)ceil_div(P.M, 32); ++b)
              for(int sl = 0; sl < P.pack_slices; ++sl) pl.items.push_back({ITEM_PACK_A, i, b, sl});
            for(int b = 0; b < (int)ceil_div(P.N, 32); ++b)
              for(int sl = 0; sl < P.pack_slices; ++sl) pl.items.push_back({ITEM_PACK_B, i, b, sl});
          }
        for(int i : at)
          if(level[i] == lv)
            for(int tm = 0; tm < pl.problems[i].tiles_m; ++tm)
              for(int tn = 0; tn < pl.problems[i].tiles_n; ++tn) pl.items.push_back({ITEM_TILE, i, tm, tn});
      }
      pl.qbeg.push_back(0);
      for(int q = 0; q < GROUPED_QUEUES; ++q) pl.qbeg.push_back((int)(pl.items.size() - first_item));
    } else {
      // pre-pack items: PREPACK_BLOCKS blocks of this segment's pre-pack job list each
      int blocks = 0;
      for(int j = prepack_first; j < (int)prepack_ops.size(); ++j) {
        const GProblem& P = pl.problems[prepack_ops[j].first];
        blocks += (int)ceil_div(ceil_div(prepack_ops[j].second ? P.M : P.N, 32) * P.kbs * 64, 256);
      }
      std::vector<GItem> pre_items;
      for(int b = 0; b < blocks; b += PREPACK_BLOCKS)
        pre_items.push_back({ITEM_PREPACK, 0, b, std::min(PREPACK_BLOCKS, blocks - b)});
      const auto qs = queue_tiles(at, pl.problems);
      pl.qbeg.push_back(0);
      size_t next_pre = 0;
      for(int q = 0; q < GROUPED_QUEUES; ++q) {
        std::vector<GItem> tiles;
        for(const TileGroup& tg : qs[q]) {
          const int tn_count = pl.problems[tg.problem].tiles_n;
          for(int t = tg.first; t < tg.first + tg.count; ++t)
            tiles.push_back({ITEM_TILE, tg.problem, t / tn_count, t % tn_count});
        }
        // this queue's share of the pre-pack items, spread evenly over its tiles
        const size_t share = (pre_items.size() * (q + 1)) / GROUPED_QUEUES - (pre_items.size() * q) / GROUPED_QUEUES;
        const size_t nt = tiles.size();
        size_t ti = 0;
        for(size_t k = 0; k < share; ++k) {
          const size_t upto = nt * (k + 1) / (share + 1);
          while(ti < upto) pl.items.push_back(tiles[ti++]);
          pl.items.push_back(pre_items[next_pre++]);
        }
        while(ti < nt) pl.items.push_back(tiles[ti++]);
        pl.qbeg.push_back((int)(pl.items.size() - first_item));
      }
    }
    pl.seg_items.push_back((int)pl.items.size());
    pl.seg_big.push_back(pl.per_level && !pl.pipelined && level_cfg[sg] >= 0 ? level_cfg[sg] : pl.big);
    pl.seg_small.push_back(pl.per_level && !pl.pipelined && level_cfg[sg] >= 0 ? level_cfg[sg] : pl.small);
  }
  if(pl.per_level)
    for(auto& P : pl.problems) P.ndeps = P.consumed = 0;  // ordered by the launches
  const int segments = nseg;

  // Job tables: pre-pass jobs (block numbers from 0 within each segment),
  // then pre-pack jobs (likewise).
  pl.jobs.clear();
  pl.job_op.clear();
  pl.seg_jobs.assign(1, 0);
  pl.seg_blocks.assign(segments, 0);
  for(int sg = 0, j = 0; sg < segments; ++sg) {
    int blocks = 0;
    for(; j < pre_seg_end[sg]; ++j) {
      const PackJob job = make_job(pl.problems[pre_ops[j].first], pre_ops[j].second == 1, blocks);
      blocks += job.blocks;
      pl.jobs.push_back(job);
      pl.job_op.push_back(pre_ops[j]);
    }
    pl.seg_blocks[sg] = blocks;
    pl.seg_jobs.push_back((int)pl.jobs.size());
  }
  pl.npre = (int)pl.jobs.size();
  pl.seg_prejobs.assign(1, pl.npre);
  for(int sg = 0, j = 0; sg < segments; ++sg) {
    int blocks = 0;
    for(; j < prepack_seg_end[sg]; ++j) {
      const PackJob job = make_job(pl.problems[prepack_ops[j].first], prepack_ops[j].second == 1, blocks);
      blocks += job.blocks;
      pl.jobs.push_back(job);
      pl.job_op.push_back(prepack_ops[j]);
    }
    pl.seg_prejobs.push_back((int)pl.jobs.size());
  }

  pl.off_problems = 0;
  pl.off_items = round_up(sizeof(GProblem) * std::max(1, count), 256);
  pl.off_qbeg = pl.off_items + round_up(sizeof(GItem) * std::max<size_t>(1, pl.items.size()), 256);
  pl.off_jobs = pl.off_qbeg + round_up(sizeof(int) * pl.qbeg.size(), 256);
  pl.off_counters = pl.off_jobs + round_up(sizeof(PackJob) * std::max<size_t>(1, pl.jobs.size()), 256);
  // counters: error flag, GROUPED_QUEUES queue heads per segment, per-problem done, per-panel pack counts
  pl.counter_ints = 1 + (size_t)segments * GROUPED_QUEUES + (size_t)count + (size_t)panels;
  pl.off_packed = pl.off_counters + round_up(pl.counter_ints * sizeof(int), 256);
  pl.total_bytes = pl.off_packed + packed_bytes;
}

mfx_status plan_grouped(Handle* h, mfx_precision prec, const mfx_gemm_problem* problems, int count,
    const mfx_dep* deps, int ndeps, GroupedPlan& pl) {
  std::optional<ListSummary> list;
  MFX_CHECK(choose_plan(h, prec, problems, count, deps, ndeps, pl, list));
  plan_tables(h, *list, deps, ndeps, pl);
  return MFX_SUCCESS;
}

// Places the packed operands in the device buffer `ws`, uploads the tables
// (stream-ordered, from pinned staging memory owned by the handle) and fills
// the kernel arguments.
static mfx_status bind_grouped(Handle* h, GroupedPlan& pl, void* ws, GroupedArgs& g, hipStream_t s) {
  char* base = static_cast<char*>(ws);
  if(pl.prec != MFX_PREC_FP32) {
    const int nhl = pl.prec == MFX_PREC_SPLIT_BF16 ? 2 : 1;
    size_t off = pl.off_packed;
    for(auto& P : pl.problems) {
      if(P.kbs == 0) continue;
      const auto sz = packed_sizes(P, nhl);
      P.packed_a = reinterpret_cast<u32x4*>(base + off);
      off += sz.first;
      P.packed_b = reinterpret_cast<u32x4*>(base + off);
      off += sz.second;
    }
    for(size_t j = 0; j < pl.jobs.size(); ++j) {
      const GProblem& P = pl.problems[pl.job_op[j].first];
      pl.jobs[j].dst = pl.job_op[j].second == 1 ? P.packed_a : P.packed_b;
    }
  }
  // The previous upload from the staging buffer must have completed.
  if(h->staging_ready) MFX_HIP(hipEventSynchronize(h->staging_ready));
  if(h->staging_bytes < pl.off_counters) {
    if(h->staging) MFX_HIP(hipHostFree(h->staging));
    h->staging = nullptr;
    h->staging_bytes = 0;
    MFX_HIP(hipHostMalloc(&h->staging, pl.off_counters, hipHostMallocDefault));
    h->staging_bytes = pl.off_counters;
  }
  if(!h->staging_ready) MFX_HIP(hipEventCreateWithFlags(&h->staging_ready, hipEventDisableTiming));
  char* st = static_cast<char*>(h->staging);
  memcpy(st + pl.off_problems, pl.problems.data(), sizeof(GProblem) * pl.problems.size());
  memcpy(st + pl.off_items, pl.items.data(), sizeof(GItem) * pl.items.size());
  memcpy(st + pl.off_qbeg, pl.qbeg.data(), sizeof(int) * pl.qbeg.size());
  if(!pl.jobs.empty()) memcpy(st + pl.off_jobs, pl.jobs.data(), sizeof(PackJob) * pl.jobs.size());
  MFX_HIP(hipMemcpyAsync(base, st, pl.off_counters, hipMemcpyHostToDevice, s));
  MFX_HIP(hipEventRecord(h->staging_ready, s));
  int* counters = reinterpret_cast<int*>(base + pl.off_counters);
  g.problems = reinterpret_cast<const GProblem*>(base + pl.off_problems);
  g.items = reinterpret_cast<const GItem*>(base + pl.off_items);
  g.qbeg = reinterpret_cast<const int*>(base + pl.off_qbeg);
  pl.dev_jobs = reinterpret_cast<const PackJob*>(base + pl.off_jobs);
  g.nitems = (int)pl.items.size();
  const int segments = (int)pl.seg_items.size() - 1;
  g.error = counters;
  g.head = counters + 1;  // segment 0; segment l uses head + l * GROUPED_QUEUES
  g.done = counters + 1 + (size_t)segments * GROUPED_QUEUES;
  g.pack_ctr = g.done + pl.problems.size();
  g.spin_limit = h->spin_limit;
  g.prejobs = nullptr;
  g.nprejobs = 0;
  return MFX_SUCCESS;
}

// Enqueues the counter reset, then per segment the pre-pass and the
// persistent kernel.
static mfx_status launch_grouped_kernels(Handle* h, const GroupedPlan& pl, const GroupedArgs& g, hipStream_t s) {
  const int n = (int)pl.counter_ints;
  MFX_CHECK(timed_launch(h, "grouped_reset", s, [&] {
    zero_ints_kernel<<<(int)std::min<int64_t>(ceil_div(n, 256), 1024), 256, 0, s>>>(g.head - 1, n, g.error);
  }));
  if(pl.items.empty()) return MFX_SUCCESS;
  const int nhl = pl.prec == MFX_PREC_SPLIT_BF16 ? 2 : 1;
  const int segments = (int)pl.seg_items.size() - 1;
  for(int l = 0; l < segments; ++l) {
    if(pl.prec != MFX_PREC_FP32)
      MFX_CHECK(launch_pack_jobs(h, nhl, pl.dev_jobs + pl.seg_jobs[l], pl.seg_jobs[l + 1] - pl.seg_jobs[l],
          pl.seg_blocks[l], s));
    GroupedArgs gl = g;
    gl.items = g.items + pl.seg_items[l];
    gl.nitems = pl.seg_items[l + 1] - pl.seg_items[l];
    gl.head = g.head + (size_t)l * GROUPED_QUEUES;
    gl.qbeg = g.qbeg + (size_t)l * (GROUPED_QUEUES + 1);
    gl.prejobs = pl.dev_jobs + pl.seg_prejobs[l];
    gl.nprejobs = pl.seg_prejobs[l + 1] - pl.seg_prejobs[l];
    if(gl.nitems == 0) continue;
    const int big = pl.seg_big[l], small = pl.seg_small[l];
    // two persistent workgroups of the 64x64 tile (64 KiB of LDS) per CU, one
    // of the others
    const int grid = cus_of(h) * (big == 2 && small == 2 && gl.nitems > cus_of(h) ? 2 : 1);
    if(pl.prec == MFX_PREC_FP32) MFX_CHECK(launch_grouped_f32(h, big, small, pl.all_vec, gl, grid, s));
    else MFX_CHECK(launch_grouped_bf16(h, nhl, big, small, pl.all_vec, gl, grid, s));
  }
  return MFX_SUCCESS;
}

// A short list whose problems each fill the GPU runs as one dense launch per
// problem instead (same stream, in list order, which is a topological one):
// those kernels split k where tiles are few and reach a tile without queues
// and problem tables.  By estimate for untuned lists, by measurement for tuned
// ones (kDenseListPolicy); a forced or tuned policy is kept.
struct DenseList {
  std::vector<DenseOp> ops;  // empty: the grouped launch is estimated shorter
  std::vector<int> config;
  size_t packed = 0, partial = 0;  // bytes of packed operands and partial tiles, shared by the problems in turn
};
constexpr int kDenseListMax = 16;
// Uploading the tables, clearing the counters and the first item of a grouped
// launch; a dense FP32 / packed BF16 product's floor (its launches on the
// host); packing a BF16 problem's operands.
constexpr double kGroupedFixedUs = 20.0, kDenseFloorUs = 11.0, kSplitFloorUs = 14.0, kBf16FloorUs = 12.0;
constexpr double kPackFixedUs = 4.0, kPackBytesPerUs = 4.5e6;

// The dense launches of a list (none if it has no such form) and their estimate.
DenseList dense_form(Handle* h, mfx_precision prec, const mfx_gemm_problem* problems, int count, double* estimate) {
  DenseList d;
  if(count == 0 || count > kDenseListMax || h->forced_config[prec] >= 0) return d;
  const int cus = cus_of(h);
  const bool packed = prec != MFX_PREC_FP32, split = prec == MFX_PREC_SPLIT_BF16;
  double dense = 0.0;
  for(int i = 0; i < count; ++i) {
    const auto& q = problems[i];
    if(q.m == 0 || q.n == 0) continue;
    const int c = choose_config(h, prec, q.m, q.n, q.k);
    int bm, bn, bk, w;
    if(!config_info(prec, c, &bm, &bn, &bk, &w)) return DenseList{};  // an id of a loaded table that this library lacks
    double us = plan_splits(prec, c, ceil_div(q.m, bm) * ceil_div(q.n, bn), q.k, cus, kMaxPartialBytes, nullptr);
    if(packed) us += kPackFixedUs + 8.0 * (double)(q.m + q.n) * (double)q.k / kPackBytesPerUs;
    dense += std::max(split ? kSplitFloorUs : packed ? kBf16FloorUs : kDenseFloorUs, us);
    DenseOp op{};
    op.M = (int)q.m;
    op.N = (int)q.n;
    op.K = (int)q.k;
    op.A = q.A;
    op.lda = q.lda;
    op.a_kmajor = q.transA == 0;
    op.B = q.B;
    op.ldb = q.ldb;
    op.b_kmajor = q.transB == 1;
    op.nprod = 1;
    op.tiles = TILES_FULL;
    op.ep = Epilogue{q.C, q.ldc, q.alpha, q.beta, (int)q.m, (int)q.n, TILES_FULL, 0};
    d.ops.push_back(op);
    d.config.push_back(c);
    size_t partial = 0;
    if(packed) d.packed = std::max(d.packed, dense_bf16x_workspace(op, split, c, cus, h->forced_splits, &partial) - partial);
    else partial = dense_f32_workspace(op, c, cus, h->forced_splits);
    d.partial = std::max(d.partial, partial);
  }
  *estimate = dense;
  return d;
}

DenseList dense_list(Handle* h, mfx_precision prec, const mfx_gemm_problem* problems, int count, const GroupedPlan& pl) {
  DenseList d;
  if(pl.estimate < 0.0) return d;
  double dense = 0.0;
  d = dense_form(h, prec, problems, count, &dense);
  const double grouped = kGroupedFixedUs + pl.estimate;
  // Clearly ahead only: the estimates differ from the times by 10 to 20 %. FP32:
  // estimated at 0.91 of the grouped time, eight chained products of 300 take
  // 1.27 of it. A packed list pays two or three launches a problem, which the
  // model knows less well: at 0.82, six independent ones took 75 us dense and 55
  // grouped (single BF16), though most lists up to 0.9 are faster dense. Lone
  // chains have no such outliers below 0.9 (split BF16, eight of 640: 91 and 105
  // us, of 900: 132 and 175), but above (single BF16, sixteen of 1200: 286 and 219).
  if(!pl.tuned_dense && dense >= (prec == MFX_PREC_FP32 || pl.summed ? 0.9 : 0.8) * grouped) d.ops.clear();
  return d;
}

mfx_status launch_dense_list(Handle* h, mfx_precision prec, const DenseList& d, void* ws, void* partials, hipStream_t s) {
  for(size_t i = 0; i < d.ops.size(); ++i) {
    if(prec == MFX_PREC_FP32) MFX_CHECK(launch_dense_f32_ws(h, d.ops[i], d.config[i], partials, d.partial, s));
    else MFX_CHECK(launch_dense_bf16x_ws(h, d.ops[i], prec == MFX_PREC_SPLIT_BF16, d.config[i], ws, s, partials));
  }
  return MFX_SUCCESS;
}

// Memory of an eager dense list; false where it is not to be had.
bool dense_memory(Handle* h, const DenseList& d, hipStream_t s, void** ws, void** partials) {
  *ws = nullptr;
  *partials = d.partial > 0 ? stream_partials(h, s) : nullptr;
  if((*partials || d.partial == 0) && (d.packed == 0 || list_workspace(h, d.packed, ws) == MFX_SUCCESS)) return true;
  (void)hipGetLastError();
  return false;
}

mfx_status run_grouped(Handle* h, mfx_precision prec, const mfx_gemm_problem* problems, int count,
    const mfx_dep* deps, int ndeps, hipStream_t s) {
  GroupedPlan pl;
  std::optional<ListSummary> list;
  MFX_CHECK(choose_plan(h, prec, problems, count, deps, ndeps, pl, list));
  void* ws = nullptr;
  const DenseList dense = dense_list(h, prec, problems, count, pl);
  h->grouped_waits = true;
  void* partials = nullptr;
  // without the memory: the grouped kernels need less
  if(!dense.ops.empty() && !is_capturing(h, s) && dense_memory(h, dense, s, &ws, &partials)) {
    h->grouped_waits = false;
    return launch_dense_list(h, prec, dense, ws, partials, s);
  }
  plan_tables(h, *list, deps, ndeps, pl);
  MFX_CHECK(workspace(h, pl.total_bytes, &ws));
  GroupedArgs g;
  MFX_CHECK(bind_grouped(h, pl, ws, g, s));
  // The flag outlives the workspace (which later calls may regrow).
  if(!h->error_flag) MFX_HIP(hipMalloc(&h->error_flag, 256));
  g.error = h->error_flag;
  return launch_grouped_kernels(h, pl, g, s);
}

// Average milliseconds of `reps` back-to-back calls of `launch` after an untimed one.
template <class F>
static mfx_status time_launches(F&& launch, int reps, hipStream_t s, double* ms) {
  MFX_CHECK(launch());
  hipEvent_t a = nullptr, b = nullptr;
  MFX_HIP(hipEventCreate(&a));
  hipError_t e = hipEventCreate(&b);
  mfx_status st = e == hipSuccess ? MFX_SUCCESS : hip_fail(e, "hipEventCreate");
  if(st == MFX_SUCCESS && (e = hipEventRecord(a, s)) != hipSuccess) st = hip_fail(e, "hipEventRecord");
  for(int r = 0; r < reps && st == MFX_SUCCESS; ++r) st = launch();
  float t = 0.0f;
  if(st == MFX_SUCCESS) {
    e = hipEventRecord(b, s);
    if(e == hipSuccess) e = hipEventSynchronize(b);
    if(e == hipSuccess) e = hipEventElapsedTime(&t, a, b);
    if(e != hipSuccess) st = hip_fail(e, "grouped timing");
  }
  (void)hipEventDestroy(a);
  if(b) (void)hipEventDestroy(b);
  *ms = t / std::max(reps, 1);
  return st;
}

mfx_status time_grouped(Handle* h, mfx_precision prec, const mfx_gemm_problem* problems, int count,
    const mfx_dep* deps, int ndeps, int reps, hipStream_t s, double* ms) {
  GroupedPlan pl;
  MFX_CHECK(plan_grouped(h, prec, problems, count, deps, ndeps, pl));
  void* ws = nullptr;
  MFX_CHECK(workspace(h, pl.total_bytes, &ws));
  GroupedArgs g;
  MFX_CHECK(bind_grouped(h, pl, ws, g, s));
  if(!h->error_flag) MFX_HIP(hipMalloc(&h->error_flag, 256));
  g.error = h->error_flag;
  h->grouped_waits = true;
  return time_launches([&] { return launch_grouped_kernels(h, pl, g, s); }, reps, s, ms);
}

mfx_status time_dense_list(Handle* h, mfx_precision prec, const mfx_gemm_problem* problems, int count, int reps,
    hipStream_t s, double* ms) {
  *ms = -1.0;
  double estimate = 0.0;
  void *ws = nullptr, *partials = nullptr;
  const DenseList d = dense_form(h, prec, problems, count, &estimate);
  if(d.ops.empty() || is_capturing(h, s) || !dense_memory(h, d, s, &ws, &partials)) return MFX_SUCCESS;
  return time_launches([&] { return launch_dense_list(h, prec, d, ws, partials, s); }, reps, s, ms);
}

// Balanced-tree product of `count` n x n matrices as grouped problems.
mfx_status chain_problems(int count, const float* const* mats, int64_t n, float* const* scratch, float* out,
    std::vector<mfx_gemm_problem>& probs, std::vector<mfx_dep>& deps) {
  if(count < 2) return invalid("a chain needs at least two matrices");
  if(!mats || !out || (count > 2 && !scratch)) return invalid("null matrix list");
  struct Node {
    const float* p;
    int producer;  // problem index, -1 for an input
  };
  std::vector<Node> level;
  for(int i = 0; i < count; ++i) {
    if(!mats[i]) return invalid("null matrix in chain");
    level.push_back({mats[i], -1});
  }
  int next_scratch = 0;
  while(level.size() > 1) {
    std::vector<Node> up;
    for(size_t i = 0; i + 1 < level.size(); i += 2) {
      const bool last = level.size() == 2;
      float* dst = last ? out : scratch[next_scratch++];
      if(!dst) return invalid("null scratch buffer");
      const int idx = (int)probs.size();
      probs.push_back({n, n, n, 1.0f, 0.0f, level[i].p, n, 0, level[i + 1].p, n, 0, dst, n});
      if(level[i].producer >= 0) deps.push_back({idx, level[i].producer});
      if(level[i + 1].producer >= 0) deps.push_back({idx, level[i + 1].producer});
      up.push_back({dst, idx});
    }
    if(level.size() % 2) up.push_back(level.back());
    level.swap(up);
  }
  return MFX_SUCCESS;
}

}  // namespace mfx

using namespace mfx;

struct mfx_graph_s {
  int device = 0;
  void* mem = nullptr;  // tables, counters and packed operands of this graph
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  int* error = nullptr;
};

extern "C" {

mfx_status mfx_gemm_grouped(mfx_handle handle, mfx_precision prec, const mfx_gemm_problem* problems, int32_t count,
    const mfx_dep* deps, int32_t ndeps, mfx_stream stream) {
  if(!handle) return invalid("null handle");
  Handle* h = &handle->h;
  MFX_HIP(hipSetDevice(h->device));
  return run_grouped(h, prec, problems, count, deps, ndeps, static_cast<hipStream_t>(stream));
}

mfx_status mfx_chain(mfx_handle handle, mfx_precision prec, int32_t count, const float* const* mats, int64_t n,
    float* const* scratch, float* out, mfx_stream stream) {
  if(!handle) return invalid("null handle");
  Handle* h = &handle->h;
  MFX_HIP(hipSetDevice(h->device));
  if(n < 0) return invalid("negative dimension");
  std::vector<mfx_gemm_problem> probs;
  std::vector<mfx_dep> deps;
  MFX_CHECK(chain_problems(count, mats, n, scratch, out, probs, deps));
  return run_grouped(h, prec, probs.data(), (int)probs.size(), deps.data(), (int)deps.size(),
      static_cast<hipStream_t>(stream));
}

mfx_status mfx_grouped_status(mfx_handle handle, mfx_stream stream) {
  if(!handle) return invalid("null handle");
  Handle* h = &handle->h;
  MFX_HIP(hipSetDevice(h->device));
  MFX_HIP(hipStreamSynchronize(static_cast<hipStream_t>(stream)));
  if(!h->error_flag || !h->grouped_waits) return MFX_SUCCESS;
  int err = 0;
  MFX_HIP(hipMemcpy(&err, h->error_flag, sizeof(int), hipMemcpyDeviceToHost));
  if(err) {
    set_last_error("an in-kernel dependency wait of the last grouped launch exceeded its spin limit");
    return MFX_ERROR_TIMEOUT;
  }
  return MFX_SUCCESS;
}

mfx_status mfx_grouped_graph_create(mfx_handle handle, mfx_precision prec, const mfx_gemm_problem* problems,
    int32_t count, const mfx_dep* deps, int32_t ndeps, mfx_stream stream, mfx_graph* graph) {
  if(!handle || !graph) return invalid("null handle or graph pointer");
  *graph = nullptr;
  Handle* h = &handle->h;
  MFX_HIP(hipSetDevice(h->device));
  hipStream_t s = static_cast<hipStream_t>(stream);
  GroupedPlan pl;
  MFX_CHECK(plan_grouped(h, prec, problems, count, deps, ndeps, pl));
  auto* gr = new(std::nothrow) mfx_graph_s;
  if(!gr) return MFX_ERROR_ALLOC;
  gr->device = h->device;
  // The graph owns its tables, counters and packed operands, so later calls on
  // the handle (which may regrow the handle's workspace) cannot move them.
  DenseList dense = dense_list(h, prec, problems, count, pl);
  hipError_t ae = hipMalloc(&gr->mem, std::max<size_t>(dense.ops.empty() ? pl.total_bytes : dense.packed + dense.partial, 256));
  if(ae != hipSuccess && !dense.ops.empty()) {
    (void)hipGetLastError();
    dense.ops.clear();
    ae = hipMalloc(&gr->mem, std::max<size_t>(pl.total_bytes, 256));
  }
  if(ae != hipSuccess) {
    delete gr;
    return hip_fail(ae, "hipMalloc(grouped graph)");
  }
  GroupedArgs g{};
  mfx_status bs = dense.ops.empty() ? bind_grouped(h, pl, gr->mem, g, s) : MFX_SUCCESS;
  hipError_t se = hipStreamSynchronize(s);  // tables resident before capture
  if(bs != MFX_SUCCESS || se != hipSuccess) {
    (void)hipFree(gr->mem);
    delete gr;
    return bs != MFX_SUCCESS ? bs : hip_fail(se, "hipStreamSynchronize");
  }
  gr->error = g.error;  // null for dense launches, which wait for nothing
  // Capture on a private stream: the graph holds the counter reset (a
  // kernel, not a memset node) and the persistent kernel.
  hipStream_t cs = nullptr;
  hipError_t ce = hipStreamCreateWithFlags(&cs, hipStreamNonBlocking);
  if(ce != hipSuccess) {
    (void)hipFree(gr->mem);
    delete gr;
    return hip_fail(ce, "hipStreamCreateWithFlags");
  }
  const bool timing = h->timing;
  h->timing = false;
  h->capturing = true;
  mfx_status st = MFX_SUCCESS;
  hipError_t e = hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal);
  if(e == hipSuccess) {
    st = dense.ops.empty() ? launch_grouped_kernels(h, pl, g, cs) : launch_dense_list(h, prec, dense, gr->mem,
                                                                          static_cast<char*>(gr->mem) + dense.packed, cs);
    hipError_t e2 = hipStreamEndCapture(cs, &gr->graph);
    if(st == MFX_SUCCESS && e2 != hipSuccess) st = hip_fail(e2, "hipStreamEndCapture");
  } else {
    st = hip_fail(e, "hipStreamBeginCapture");
  }
  h->capturing = false;
  h->timing = timing;
  if(st == MFX_SUCCESS) {
    e = hipGraphInstantiate(&gr->exec, gr->graph, nullptr, nullptr, 0);
    if(e != hipSuccess) st = hip_fail(e, "hipGraphInstantiate");
  }
  (void)hipStreamDestroy(cs);
  if(st != MFX_SUCCESS) {
    if(gr->exec) (void)hipGraphExecDestroy(gr->exec);
    if(gr->graph) (void)hipGraphDestroy(gr->graph);
    (void)hipFree(gr->mem);
    delete gr;
    return st;
  }
  *graph = gr;
  return MFX_SUCCESS;
}

mfx_status mfx_graph_launch(mfx_graph graph, mfx_stream stream) {
  if(!graph) return invalid("null graph");
  MFX_HIP(hipSetDevice(graph->device));
  MFX_HIP(hipGraphLaunch(graph->exec, static_cast<hipStream_t>(stream)));
  return MFX_SUCCESS;
}

mfx_status mfx_graph_status(mfx_graph graph, mfx_stream stream) {
  if(!graph) return invalid("null graph");
  MFX_HIP(hipSetDevice(graph->device));
  MFX_HIP(hipStreamSynchronize(static_cast<hipStream_t>(stream)));
  if(!graph->error) return MFX_SUCCESS;
  int err = 0;
  MFX_HIP(hipMemcpy(&err, graph->error, sizeof(int), hipMemcpyDeviceToHost));
  if(err) {
    set_last_error("an in-kernel dependency wait of the last graph replay exceeded its spin limit");
    return MFX_ERROR_TIMEOUT;
  }
  return MFX_SUCCESS;
}

mfx_status mfx_graph_destroy(mfx_graph graph) {
  if(!graph) return MFX_SUCCESS;
  hipError_t e = hipSetDevice(graph->device);
  if(e == hipSuccess) e = hipDeviceSynchronize();  // no replay may still use the memory
  if(graph->exec && e == hipSuccess) e = hipGraphExecDestroy(graph->exec);
  if(graph->graph && e == hipSuccess) e = hipGraphDestroy(graph->graph);
  if(graph->mem && e == hipSuccess) e = hipFree(graph->mem);
  delete graph;
  return e == hipSuccess ? MFX_SUCCESS : hip_fail(e, "mfx_graph_destroy");
}

}  // extern "C"
