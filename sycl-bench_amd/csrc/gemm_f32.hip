// FP32 dense contractions on v_mfma_f32_32x32x2_f32: one tile per workgroup
// (the tile body is in tile_f32.h).
//
// Replaces the naive one-work-item-per-element kernels of
// polybench/gemm.cpp:77-92, polybench/2mm.cpp:94-123, polybench/3mm.cpp:115-158,
// polybench/syrk.cpp:70-84, polybench/syr2k.cpp:73-88 and
// runtime/matmulchain.cpp:15-29.
#include "tile_f32.h"

namespace mfx {
namespace {

struct F32Params {
  DenseOp op;
  int tiles_m, tiles_n, group;
  SplitPlan plan;  // workgroups [0, head) take whole tiles, the rest slices
  int tiles;       // tiles of the schedule
  float* partial;
  int tail_first = -1, tail_ratio = 1, big_tiles = 0;  // triangle_tile's re-tiled last round
};

template <int BM, int BN, int WM, int WN, bool AK, bool BKM, bool VEC, int NB, int KG>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * KG * 64) void gemm_f32_kernel(const F32Params p) {
  __shared__ __align__(16) float smem[F32Cfg<BM, BN, WM, WN, VEC, NB, KG>::SMEM_FLOATS];
  constexpr int BK = F32_BK * KG;
  const int steps = (p.op.K + BK - 1) / BK * p.op.nprod;
  int tm, tn, s0 = 0, s1 = steps;
  Epilogue ep = p.op.ep;
  int er, ec;
  if((int)blockIdx.x < p.plan.head) {
    const int id = xcd_remap(blockIdx.x, p.plan.head);
    if(p.tail_first >= 0) {
      int ti, tj;
      if(!triangle_tile(id, p.tiles_m, p.group, p.tail_first, p.tail_ratio, p.big_tiles, ti, tj)) return;
      tm = p.op.tiles == TILES_LOWER ? ti : tj;
      tn = p.op.tiles == TILES_LOWER ? tj : ti;
    } else {
      tile_of(p.op.tiles, id, p.tiles_m, p.tiles_n, p.group, tm, tn);
    }
    er = tm * BM;
    ec = tn * BN;
  } else {
    // slice-major, as in gemm_bf16x_kernel
    const int rest = p.tiles - p.plan.head, splits = p.plan.splits;
    const int id = xcd_remap(blockIdx.x - p.plan.head, rest * splits);
    const int slice = id / rest, tile = id - slice * rest;
    tile_of(p.op.tiles, p.plan.head + tile, p.tiles_m, p.tiles_n, p.group, tm, tn);
    s0 = (int)((int64_t)steps * slice / splits);
    s1 = (int)((int64_t)steps * (slice + 1) / splits);
    ep = Epilogue{p.partial + ((int64_t)tile * splits + slice) * (BM * BN), BN, 1.0f, 0.0f, BM, BN, TILES_FULL, 0};
    er = ec = 0;
  }
  f32_tile<BM, BN, WM, WN, AK, BKM, VEC, NB, KG>(p.op, tm, tn, s0, s1, ep, er, ec, smem);
}

struct F32Config {
  int bm, bn, waves, bk;
};
// Compiled tile configurations; index = config id.
constexpr F32Config kF32Configs[] = {
    {256, 256, 4, 16}, // 0: 128x128 per wave
    {128, 128, 4, 16}, // 1: 64x64 per wave
    {64, 64, 4, 16},   // 2: 32x32 per wave, four stages buffered (four workgroups per CU)
    {256, 128, 4, 16}, // 3: 128x64 per wave
    {256, 256, 8, 16}, // 4: 128x64 per wave, two waves per SIMD
    {256, 128, 8, 16}, // 5: 64x64 per wave, two waves per SIMD
    {128, 128, 8, 16}, // 6: 64x32 per wave, two waves per SIMD
    {64, 64, 8, 32},   // 7: 32x32 per wave, two k-groups
};
// Configuration 2 covers load latency with workgroups instead of buffers.
constexpr int kF32Crowded = 2;
constexpr int kF32ConfigCount = sizeof(kF32Configs) / sizeof(kF32Configs[0]);

template <int BM, int BN, int WM, int WN, bool VEC, int NB, int KG>
void launch_layout(const F32Params& p, int grid, hipStream_t s) {
  constexpr int NT = F32Cfg<BM, BN, WM, WN, VEC, NB, KG>::NT;
  const bool ak = p.op.a_kmajor, bk = p.op.b_kmajor;
  if(ak && !bk) gemm_f32_kernel<BM, BN, WM, WN, true, false, VEC, NB, KG><<<grid, NT, 0, s>>>(p);
  else if(ak && bk) gemm_f32_kernel<BM, BN, WM, WN, true, true, VEC, NB, KG><<<grid, NT, 0, s>>>(p);
  else if(!ak && !bk) gemm_f32_kernel<BM, BN, WM, WN, false, false, VEC, NB, KG><<<grid, NT, 0, s>>>(p);
  else gemm_f32_kernel<BM, BN, WM, WN, false, true, VEC, NB, KG><<<grid, NT, 0, s>>>(p);
}

// 16-byte copies only when both operands allow them.
template <int BM, int BN, int WM, int WN, int NB = f32_stages<BM, BN>(), int KG = 1>
void launch_cfg(const F32Params& p, bool vec, int grid, hipStream_t s) {
  if(vec) launch_layout<BM, BN, WM, WN, true, NB, KG>(p, grid, s);
  else launch_layout<BM, BN, WM, WN, false, NB, KG>(p, grid, s);
}

mfx_status launch_f32_config(Handle* h, const F32Params& p, bool vec, int config, int grid, hipStream_t s) {
  return timed_launch(h, p.plan.splits > 1 ? "gemm_f32_splitk" : "gemm_f32_mfma", s, [&] {
    switch(config) {
      case 0: launch_cfg<256, 256, 128, 128>(p, vec, grid, s); break;
      case 1: launch_cfg<128, 128, 64, 64>(p, vec, grid, s); break;
      case 2: launch_cfg<64, 64, 32, 32, 4>(p, vec, grid, s); break;
      case 3: launch_cfg<256, 128, 128, 64>(p, vec, grid, s); break;
      case 4: launch_cfg<256, 256, 128, 64>(p, vec, grid, s); break;
      case 5: launch_cfg<256, 128, 64, 64>(p, vec, grid, s); break;
      case 6: launch_cfg<128, 128, 64, 32>(p, vec, grid, s); break;
      case 7: launch_cfg<64, 64, 32, 32, 4, 2>(p, vec, grid, s); break;
    }
  });
}

int64_t f32_tiles(const DenseOp& op, int config) {
  const int64_t tm = ceil_div(op.M, kF32Configs[config].bm), tn = ceil_div(op.N, kF32Configs[config].bn);
  return op.tiles == TILES_FULL ? tm * tn : tm * (tm + 1) / 2;
}

SplitPlan f32_split_plan(const DenseOp& op, int config, int cus, int forced_splits) {
  const F32Config& c = kF32Configs[config];
  const int64_t tiles = f32_tiles(op, config), steps = ceil_div(op.K, c.bk) * op.nprod;
  SplitPlan plan{(int)tiles, 1};
  if(forced_splits >= 2) {
    int64_t s = std::min<int64_t>(forced_splits, steps);
    while(s > 1 && tiles * s * c.bm * c.bn * 4 > kMaxPartialBytes) --s;
    if(s > 1) plan = SplitPlan{0, (int)s};
  } else if(forced_splits < 0 && config == kF32Crowded) {
    // many short slices: four workgroups per CU, each at least 128 k, at most
    // eight slices
    int64_t s = std::min<int64_t>(std::min<int64_t>(8, 4 * cus / std::max<int64_t>(tiles, 1)), op.K / 128);
    while(s > 1 && tiles * s * c.bm * c.bn * 4 > kMaxPartialBytes) --s;
    if(s > 1 && op.nprod == 1) plan = SplitPlan{0, (int)s};
  } else if(forced_splits < 0) {
    plan_splits(MFX_PREC_FP32, config, tiles, steps * c.bk, cus, kMaxPartialBytes, &plan);
  }
  return plan;
}

size_t partial_bytes(const SplitPlan& plan, int64_t tiles, const F32Config& c) {
  return plan.splits > 1 ? (size_t)(tiles - plan.head) * plan.splits * c.bm * c.bn * sizeof(float) : 0;
}

// How a call runs on one configuration: k slices, or a triangle's re-tiled last
// round (tail.small >= 0, the plan then whole), or neither.
struct F32Call {
  SplitPlan plan;
  TriTail tail;
  size_t partial = 0;  // bytes of partial tiles
};

F32Call f32_call(const DenseOp& op, int config, int cus, int forced_splits) {
  F32Call c;
  const int64_t tiles = f32_tiles(op, config);
  if(op.tiles != TILES_FULL && forced_splits < 2)
    plan_f32_triangle(config, ceil_div(op.M, kF32Configs[config].bm), (int64_t)op.K * op.nprod, cus,
        forced_splits == 1 ? 0 : kMaxPartialBytes, &c.plan, &c.tail);
  else
    c.plan = f32_split_plan(op, config, cus, forced_splits);
  c.partial = partial_bytes(c.plan, tiles, kF32Configs[config]);
  return c;
}

mfx_status run_f32(Handle* h, const DenseOp& op, int config, const F32Call& call, void* partial, hipStream_t s) {
  const F32Config& c = kF32Configs[config];
  F32Params p;
  p.op = op;
  p.tiles_m = (int)ceil_div(op.M, c.bm);
  p.tiles_n = (int)ceil_div(op.N, c.bn);
  p.group = 8;
  // a second product swaps the operands: one load width for both
  const bool vec = f32_vec_ok(op.A, op.lda, op.a_kmajor, op.M, op.K) && f32_vec_ok(op.B, op.ldb, op.b_kmajor, op.N, op.K);
  if(op.tiles != TILES_FULL && (op.M != op.N || c.bm != c.bn)) return invalid("triangular schedule needs square tiles");
  p.tiles = (int)f32_tiles(op, config);
  if(p.tiles == 0) return MFX_SUCCESS;
  p.plan = call.plan;
  p.partial = static_cast<float*>(partial);
  if(call.tail.small >= 0) {
    // the full rounds on this tile, the last round's big tiles re-tiled
    const TriTail& tail = call.tail;
    MFX_CHECK(launch_f32_config(h, p, vec, config, tail.head, s));
    F32Params q = p;
    q.tiles_m = q.tiles_n = (int)ceil_div(op.M, kF32Configs[tail.small].bm);
    q.tail_first = tail.head;
    q.tail_ratio = tail.ratio;
    q.big_tiles = p.tiles_m;
    q.plan.head = (p.tiles - tail.head) * tail.ratio * tail.ratio;
    return launch_f32_config(h, q, vec, tail.small, q.plan.head, s);
  }
  const int grid = p.plan.head + (p.tiles - p.plan.head) * p.plan.splits;
  MFX_CHECK(launch_f32_config(h, p, vec, config, grid, s));
  if(p.plan.splits == 1) return MFX_SUCCESS;
  const SplitReduceArgs r{p.partial, c.bm, c.bn, p.plan.splits, p.plan.head, p.tiles, op.tiles, p.tiles_m, p.tiles_n,
      p.group, op.ep};
  return launch_splitk_reduce(h, r, s);
}

// Full single products on at most one tile for every two CUs, which lose most
// unsplit: the ones that may keep their partial tiles in the handle's workspace
// where the stream has no buffer of its own.
bool few_tiles(const DenseOp& op, int config, int cus) {
  return op.tiles == TILES_FULL && op.nprod == 1 && kF32Configs[config].bm <= 128 && 2 * f32_tiles(op, config) <= cus;
}

}  // namespace

double plan_f32_triangle(int config, int64_t T, int64_t k, int cus, int64_t max_partial, SplitPlan* plan, TriTail* tail) {
  SplitPlan slices;
  const int64_t tiles = T * (T + 1) / 2;
  const double us = plan_splits(MFX_PREC_FP32, config, tiles, k, cus, config == kF32Crowded ? 0 : max_partial, &slices);
  TriTail t = tri_tail(MFX_PREC_FP32, config, T, cus, k);
  const bool retile = t.small >= 0 && t.us < us;
  if(!retile) t.small = -1;
  if(plan) *plan = retile ? SplitPlan{t.head, 1} : slices;
  if(tail) *tail = t;
  return retile ? t.us : us;
}

size_t dense_f32_workspace(const DenseOp& op, int config, int cus, int forced_splits) {
  if(config < 0 || config >= kF32ConfigCount) return 0;
  return f32_call(op, config, cus, forced_splits).partial;
}

int f32_config_count() { return kF32ConfigCount; }
bool f32_config_info(int c, int* bm, int* bn, int* bk, int* waves) {
  if(c < 0 || c >= kF32ConfigCount) return false;
  *bm = kF32Configs[c].bm;
  *bn = kF32Configs[c].bn;
  *bk = kF32Configs[c].bk;
  *waves = kF32Configs[c].waves;
  return true;
}

mfx_status launch_dense_f32(Handle* h, const DenseOp& op, int config, hipStream_t s) {
  if(config < 0 || config >= kF32ConfigCount) return invalid("FP32 tile configuration out of range");
  F32Call call = f32_call(op, config, cus_of(h), h->forced_splits);
  void* partial = nullptr;
  if(call.partial > 0) {
    partial = stream_partials(h, s);
    if(!partial && few_tiles(op, config, cus_of(h)) && (!is_capturing(h, s) || call.partial <= h->workspace_bytes))
      MFX_CHECK(workspace(h, call.partial, &partial));
    if(!partial) {
      config = whole_config(h, MFX_PREC_FP32, op, config);
      call = f32_call(op, config, cus_of(h), 1);
    }
  }
  return run_f32(h, op, config, call, partial, s);
}

mfx_status launch_dense_f32_ws(Handle* h, const DenseOp& op, int config, void* ws, size_t ws_bytes, hipStream_t s) {
  if(config < 0 || config >= kF32ConfigCount) return invalid("FP32 tile configuration out of range");
  const F32Call call = f32_call(op, config, cus_of(h), h->forced_splits);
  if(call.partial > ws_bytes) return unsupported("split-K partial tiles exceed the given buffer");
  return run_f32(h, op, config, call, ws, s);
}

}  // namespace mfx
