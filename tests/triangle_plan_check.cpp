// Host-only check of the FP32 triangle plans: whichever of whole tiles, k slices
// and a re-tiled last round is estimated shortest runs, and the memory a call asks
// for is that plan's. Prints "OK <plans>", or the first plan that differs.
#include <algorithm>
#include <cstdio>

#include "mfx_internal.h"

using namespace mfx;

int main() {
  int plans = 0, retiled = 0, sliced = 0;
  for(int cus : {256, 80})
    for(int64_t n : {100, 700, 1024, 2048, 2900, 3000, 4096, 5000, 5793, 6000, 8192, 9000, 12288})
      for(int64_t k : {1, 79, 512, 1024, 2500, 8192})
        for(int c = 0; c < config_count(MFX_PREC_FP32); ++c) {
          int bm, bn, bk, w;
          if(!config_info(MFX_PREC_FP32, c, &bm, &bn, &bk, &w) || bm != bn) continue;
          const int64_t T = ceil_div(n, bm), tiles = T * (T + 1) / 2;
          SplitPlan plan, slices;
          TriTail tail;
          const double us = plan_f32_triangle(c, T, k, cus, kMaxPartialBytes, &plan, &tail);
          const double whole = tile_span(MFX_PREC_FP32, c, tiles, (double)k, cus);
          const double split = plan_splits(MFX_PREC_FP32, c, tiles, k, cus, c == 2 ? 0 : kMaxPartialBytes, &slices);
          bool ok = us <= std::min(whole, split) && (int64_t)plan.head <= tiles;
          if(tail.small >= 0) {
            int sm;
            ok = ok && config_info(MFX_PREC_FP32, tail.small, &sm, &bn, &bk, &w) && sm * tail.ratio == bm && plan.splits == 1 &&
                 plan.head == tail.head &&
                 us == tile_span(MFX_PREC_FP32, c, tail.head, (double)k, cus) +
                           tile_span(MFX_PREC_FP32, tail.small, (tiles - tail.head) * tail.ratio * tail.ratio, (double)k, cus);
            ++retiled;
          } else {
            ok = ok && us == split && plan.head == slices.head && plan.splits == slices.splits;
            sliced += plan.splits > 1;
          }
          DenseOp op{};
          op.M = op.N = (int)n;
          op.K = (int)k;
          op.nprod = 1;
          op.tiles = TILES_LOWER;
          const size_t bytes = plan.splits > 1 ? (size_t)(tiles - plan.head) * plan.splits * bm * bm * 4 : 0;
          ok = ok && dense_f32_workspace(op, c, cus, -1) == bytes;
          if(!ok) {
            std::printf("FAILED n %lld k %lld configuration %d, %d CUs\n", (long long)n, (long long)k, c, cus);
            return 1;
          }
          ++plans;
        }
  if(retiled < 10 || sliced < 10) {
    std::printf("FAILED: %d re-tiled, %d sliced\n", retiled, sliced);
    return 1;
  }
  std::printf("OK %d\n", plans);
  return 0;
}
