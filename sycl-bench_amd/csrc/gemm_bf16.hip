// Split-BF16 and single-BF16 dense contractions on v_mfma_f32_32x32x16_bf16
// (building blocks in tile_bf16.h).
//
// Two or three kernels per call:
//  1. pack: converts each operand once into fragment order (hi and lo), with
//     zero padding, so the contraction loop has no bounds checks and every
//     load is a contiguous 16-byte chunk; both operands in one launch;
//  2. contract: BM x BN tiles, LDS stages in the same fragment order
//     (ds_read_b128 of consecutive 16-byte chunks: conflict-free), fused
//     alpha/beta epilogue; tiles that do not fill a round of the CUs in k
//     slices (SplitPlan), summed by a third kernel.
// The same packed layout serves an operand in either role (A rows, or B
// columns), which is what lets syrk use one packed copy of A for both.
#include "tile_bf16.h"

namespace mfx {
namespace {

struct PackOperand {
  PackSrc s;
  int blocks;  // padded rows / 32
  int kbs;     // padded K / 16
  u32x4* dst;
};
struct PackParams {
  PackOperand a, b;
  int grid_a;  // workgroups of a; the rest are b's
};

// One lane-chunk per thread; a non-k-major source goes through the wave's
// LDS tile (load_chunk8_staged) so its reads are 128-byte row segments, with
// the (blk, kb) pairs walked kb-major so that neighbouring waves read
// neighbouring segments of the same source rows.
template <int NHL>
__global__ __launch_bounds__(256) void pack_bf16x_kernel(const PackParams pp) {
  __shared__ float tiles[4][STAGED_TILE_FLOATS];
  const bool first = (int)blockIdx.x < pp.grid_a;
  const PackOperand& p = first ? pp.a : pp.b;
  const int64_t gid = (int64_t)(first ? blockIdx.x : blockIdx.x - pp.grid_a) * 256 + threadIdx.x;
  const int64_t total = (int64_t)p.blocks * p.kbs * 64;
  const bool active = gid < total;
  const int lane = (int)(gid & 63);
  const int64_t t = gid >> 6;
  if(p.s.kmajor) {
    if(active) pack_chunk<NHL>(p.s, (int)(t / p.kbs), (int)(t % p.kbs), lane, p.kbs, p.dst);
    return;
  }
  const int blk = (int)(t % p.blocks), kb = (int)(t / p.blocks);
  float v[8];
  load_chunk8_staged(p.s, blk, kb, lane, active, v, tiles[threadIdx.x >> 6]);
  if(active) store_chunk<NHL>(p.dst, blk, kb, lane, p.kbs, v);
}

struct BfParams {
  BfTileArgs t;
  int tiles_m, tiles_n, group;
  int mode;        // TILES_FULL / LOWER / UPPER
  SplitPlan plan;  // workgroups [0, head) take whole tiles, the rest slices
  int tiles;       // tiles of the schedule
  float* partial;
};

template <int BM, int BN, int WM, int WN, int NHL, int MOST = 4>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64) void gemm_bf16x_kernel(const BfParams p) {
  using Cfg = BfCfg<BM, BN, WM, WN, NHL, MOST>;
  __shared__ u32x4 lds[Cfg::SMEM_CHUNKS];
  int tm, tn;
  const int steps = p.t.kbs / Cfg::KB * p.t.nprod;
  if((int)blockIdx.x < p.plan.head) {
    tile_of(p.mode, xcd_remap(blockIdx.x, p.plan.head), p.tiles_m, p.tiles_n, p.group, tm, tn);
    bf16_tile<BM, BN, WM, WN, NHL, MOST>(p.t, tm, tn, 0, steps, p.t.ep, tm * BM, tn * BN, lds);
    return;
  }
  // slice-major: an XCD's consecutive workgroups read the same k range of
  // neighbouring tiles, which share operand panels in its L2
  const int rest = p.tiles - p.plan.head, splits = p.plan.splits;
  const int id = xcd_remap(blockIdx.x - p.plan.head, rest * splits);
  const int slice = id / rest, tile = id - slice * rest;
  tile_of(p.mode, p.plan.head + tile, p.tiles_m, p.tiles_n, p.group, tm, tn);
  const int s0 = (int)((int64_t)steps * slice / splits), s1 = (int)((int64_t)steps * (slice + 1) / splits);
  float* slot = p.partial + ((int64_t)tile * splits + slice) * (BM * BN);
  const Epilogue ep{slot, BN, 1.0f, 0.0f, BM, BN, TILES_FULL, 0};
  bf16_tile<BM, BN, WM, WN, NHL, MOST>(p.t, tm, tn, s0, s1, ep, 0, 0, lds);
}

struct BfConfig {
  int bm, bn, waves;
};
constexpr BfConfig kBfConfigs[] = {
    {256, 256, 4},  // 0: 128x128 per wave
    {128, 128, 4},  // 1: 64x64 per wave
    {64, 64, 4},    // 2: 32x32 per wave
    {256, 128, 4},  // 3: 128x64 per wave
    {256, 256, 8},  // 4: 128x64 per wave, two waves per SIMD
    {256, 128, 8},  // 5: 64x64 per wave, two waves per SIMD
    {128, 128, 8},  // 6: 64x32 per wave, two waves per SIMD
};
constexpr int kBfConfigCount = sizeof(kBfConfigs) / sizeof(kBfConfigs[0]);

template <int BM, int BN, int WM, int WN, int MOST = 4>
mfx_status launch_bf_cfg(Handle* h, const BfParams& p, bool split, int grid, hipStream_t s) {
  if(split)
    return timed_launch(h, MOST == 2 ? "gemm_split_bf16_short_k" : "gemm_split_bf16_mfma", s, [&] {
      gemm_bf16x_kernel<BM, BN, WM, WN, 2, MOST><<<grid, BfCfg<BM, BN, WM, WN, 2>::NT, 0, s>>>(p);
    });
  return timed_launch(h, MOST == 2 ? "gemm_bf16_short_k" : "gemm_bf16_mfma", s, [&] {
    gemm_bf16x_kernel<BM, BN, WM, WN, 1, MOST><<<grid, BfCfg<BM, BN, WM, WN, 1>::NT, 0, s>>>(p);
  });
}

mfx_status launch_bf_config(Handle* h, const BfParams& p, bool split, int config, int grid, hipStream_t s) {
  switch(config) {
    case 0: return launch_bf_cfg<256, 256, 128, 128>(h, p, split, grid, s);
    case 1: return launch_bf_cfg<128, 128, 64, 64>(h, p, split, grid, s);
    case 2: return launch_bf_cfg<64, 64, 32, 32>(h, p, split, grid, s);
    case 3: return launch_bf_cfg<256, 128, 128, 64>(h, p, split, grid, s);
    case 4: return launch_bf_cfg<256, 256, 128, 64>(h, p, split, grid, s);
    case 5: return launch_bf_cfg<256, 128, 64, 64>(h, p, split, grid, s);
    case 6:
      if(p.plan.splits == 1 &&
         bf16_two_per_cu(split ? MFX_PREC_SPLIT_BF16 : MFX_PREC_BF16, config, p.tiles, p.t.kbs * 16 * p.t.nprod, cus_of(h)))
        return launch_bf_cfg<128, 128, 64, 32, 2>(h, p, split, grid, s);
      return launch_bf_cfg<128, 128, 64, 32>(h, p, split, grid, s);
  }
  return invalid("unknown BF16 configuration");
}

struct PackPlan {
  int64_t rows_pad_a, rows_pad_b, kbs;
  size_t bytes_a, bytes_b;  // rounded to 256
  int64_t tiles;
  SplitPlan split;
  size_t bytes_partial;
};

PackPlan plan(const DenseOp& op, bool split, int config, int cus, int forced_splits) {
  const BfConfig& c = kBfConfigs[config];
  PackPlan pl;
  const int nhl = split ? 2 : 1;
  // rows padded to 32 only (bf16_tile reads the last block again past them)
  pl.rows_pad_a = round_up(op.M, 32);
  pl.rows_pad_b = round_up(op.N, 32);
  const int stage = kb_per_stage_of(nhl);
  pl.kbs = round_up(op.K, 16 * stage) / 16;
  pl.bytes_a = (size_t)round_up(pl.rows_pad_a * pl.kbs * 16 * nhl * 2, 256);
  pl.bytes_b = (size_t)round_up(pl.rows_pad_b * pl.kbs * 16 * nhl * 2, 256);
  const int64_t tm = ceil_div(op.M, c.bm), tn = ceil_div(op.N, c.bn);
  pl.tiles = op.tiles == TILES_FULL ? tm * tn : tm * (tm + 1) / 2;
  pl.split = SplitPlan{(int)pl.tiles, 1};
  pl.bytes_partial = 0;
  const int64_t steps = pl.kbs / stage * op.nprod;
  if(forced_splits >= 2) {
    int64_t s = std::min<int64_t>(forced_splits, steps);
    while(s > 1 && pl.tiles * s * c.bm * c.bn * 4 > kMaxPartialBytes) --s;
    if(s > 1) pl.split = SplitPlan{0, (int)s};
  } else if(forced_splits < 0) {
    plan_splits(split ? MFX_PREC_SPLIT_BF16 : MFX_PREC_BF16, config, pl.tiles, steps * stage * 16, cus,
        kMaxPartialBytes, &pl.split);
  }
  if(pl.split.splits > 1)
    pl.bytes_partial = (size_t)(pl.tiles - pl.split.head) * pl.split.splits * c.bm * c.bn * sizeof(float);
  return pl;
}

PackOperand pack_operand(const float* src, int64_t ld, int rows, int K, bool kmajor, int64_t rows_pad, int64_t kbs,
    u32x4* dst) {
  PackOperand o;
  o.s = make_pack_src(src, ld, rows, K, kmajor);
  o.blocks = (int)(rows_pad / 32);
  o.kbs = (int)kbs;
  o.dst = dst;
  return o;
}

// Packs one operand, or both in one launch (b == nullptr: a alone).
mfx_status pack(Handle* h, const PackOperand& a, const PackOperand* b, int nhl, hipStream_t s) {
  PackParams pp;
  pp.a = a;
  pp.b = b ? *b : a;
  const int64_t grid_a = ceil_div((int64_t)a.blocks * a.kbs * 64, 256);
  const int64_t grid_b = b ? ceil_div((int64_t)b->blocks * b->kbs * 64, 256) : 0;
  if(grid_a + grid_b == 0) return MFX_SUCCESS;
  pp.grid_a = (int)grid_a;
  const unsigned grid = (unsigned)(grid_a + grid_b);
  if(nhl == 2)
    return timed_launch(h, "pack_split_bf16", s, [&] { pack_bf16x_kernel<2><<<grid, 256, 0, s>>>(pp); });
  return timed_launch(h, "pack_bf16", s, [&] { pack_bf16x_kernel<1><<<grid, 256, 0, s>>>(pp); });
}

}  // namespace

PackSrc make_pack_src(const float* src, int64_t ld, int rows, int K, bool kmajor) {
  PackSrc s;
  s.src = src;
  s.ld = ld;
  s.rows = rows;
  s.K = K;
  s.kmajor = kmajor;
  // 128-bit loads along the contiguous dimension (k if kmajor, rows if not)
  s.vec = (reinterpret_cast<uintptr_t>(src) & 15u) == 0 && ld % 4 == 0;
  return s;
}

int bf_config_count() { return kBfConfigCount; }
bool bf_config_info(int c, bool split, int* bm, int* bn, int* bk, int* waves) {
  if(c < 0 || c >= kBfConfigCount) return false;
  *bm = kBfConfigs[c].bm;
  *bn = kBfConfigs[c].bn;
  *bk = 16 * kb_per_stage_of(split ? 2 : 1);
  *waves = kBfConfigs[c].waves;
  return true;
}

size_t dense_bf16x_workspace(const DenseOp& op, bool split, int config, int cus, int forced_splits, size_t* partial) {
  if(partial) *partial = 0;
  if(config < 0 || config >= kBfConfigCount) return 0;
  const PackPlan pl = plan(op, split, config, cus, forced_splits);
  if(partial) *partial = pl.bytes_partial;
  // syrk (single operand used in both roles) still reserves two slots; the
  // second is simply unused.
  return pl.bytes_a + pl.bytes_b + pl.bytes_partial;
}

namespace {

// The pack kernels write every chunk of both padded panels (zeros past the
// matrix) and the slices every partial tile, so `ws` needs no clearing and
// may hold anything on entry.
mfx_status run_bf16x(Handle* h, const DenseOp& op, bool split, int config, const PackPlan& pl, void* ws, void* partials,
    hipStream_t s) {
  const BfConfig& c = kBfConfigs[config];
  const int nhl = split ? 2 : 1;
  const bool same = op.A == op.B && op.lda == op.ldb && op.a_kmajor == op.b_kmajor && op.M == op.N &&
                    pl.rows_pad_a == pl.rows_pad_b;
  if(op.nprod == 2 && pl.rows_pad_a != pl.rows_pad_b) return invalid("two-product form needs equal operand shapes");
  if(op.tiles != TILES_FULL && (op.M != op.N || c.bm != c.bn)) return invalid("triangular schedule needs square tiles");
  char* w = static_cast<char*>(ws);
  u32x4* pa = reinterpret_cast<u32x4*>(w);
  u32x4* pb = same ? pa : reinterpret_cast<u32x4*>(w + pl.bytes_a);
  // The B-role operand is indexed (n, k): B[n*ldb + k] if b_kmajor else B[k*ldb + n].
  const PackOperand oa = pack_operand(op.A, op.lda, op.M, op.K, op.a_kmajor, pl.rows_pad_a, pl.kbs, pa);
  const PackOperand ob = pack_operand(op.B, op.ldb, op.N, op.K, op.b_kmajor, pl.rows_pad_b, pl.kbs, pb);
  MFX_CHECK(pack(h, oa, same ? nullptr : &ob, nhl, s));
  BfParams p;
  p.t.PA = pa;
  p.t.PB = pb;
  p.t.kbs = (int)pl.kbs;
  p.t.nprod = op.nprod;
  p.t.ep = op.ep;
  p.t.nblk_a = (int)(pl.rows_pad_a / 32);
  p.t.nblk_b = (int)(pl.rows_pad_b / 32);
  p.tiles_m = (int)ceil_div(op.M, c.bm);
  p.tiles_n = (int)ceil_div(op.N, c.bn);
  p.group = 8;
  p.mode = op.tiles;
  p.plan = pl.split;
  p.tiles = (int)pl.tiles;
  p.partial = static_cast<float*>(partials);
  const int grid = p.plan.head + (p.tiles - p.plan.head) * p.plan.splits;
  MFX_CHECK(launch_bf_config(h, p, split, config, grid, s));
  if(p.plan.splits == 1) return MFX_SUCCESS;
  const SplitReduceArgs r{p.partial, c.bm, c.bn, p.plan.splits, p.plan.head, p.tiles, p.mode, p.tiles_m, p.tiles_n,
      p.group, op.ep};
  return launch_splitk_reduce(h, r, s);
}

}  // namespace

mfx_status launch_dense_bf16x(Handle* h, const DenseOp& op, bool split, int config, hipStream_t s) {
  if(config < 0 || config >= kBfConfigCount) return invalid("BF16 tile configuration out of range");
  if(op.M == 0 || op.N == 0) return MFX_SUCCESS;
  PackPlan pl = plan(op, split, config, cus_of(h), h->forced_splits);
  void *ws = nullptr, *partials = nullptr;
  MFX_CHECK(packed_workspace(h, pl.bytes_a + pl.bytes_b, pl.bytes_partial, s, &ws, &partials));
  if(pl.bytes_partial > 0 && !partials) {
    config = whole_config(h, split ? MFX_PREC_SPLIT_BF16 : MFX_PREC_BF16, op, config);
    pl = plan(op, split, config, cus_of(h), 1);
  }
  return run_bf16x(h, op, split, config, pl, ws, partials, s);
}

mfx_status launch_dense_bf16x_ws(Handle* h, const DenseOp& op, bool split, int config, void* ws, hipStream_t s,
    void* partials) {
  if(config < 0 || config >= kBfConfigCount) return invalid("BF16 tile configuration out of range");
  if(op.M == 0 || op.N == 0) return MFX_SUCCESS;
  const PackPlan pl = plan(op, split, config, cus_of(h), h->forced_splits);
  if(!partials) partials = static_cast<char*>(ws) + pl.bytes_a + pl.bytes_b;
  return run_bf16x(h, op, split, config, pl, ws, partials, s);
}

// Element-wise split used by mfx_split_bf16 (a test and tooling utility).
namespace {
__global__ void split_elementwise_kernel(int64_t n, const float* x, uint16_t* hi, uint16_t* lo) {
  for(int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    // the conversion the contraction kernels use (split_chunk)
    const uint32_t h = cvt_pk_bf16(x[i], 0.0f) & 0xffffu;
    hi[i] = (uint16_t)h;
    lo[i] = (uint16_t)(cvt_pk_bf16(x[i] - bf16_to_f32((uint16_t)h), 0.0f) & 0xffffu);
  }
}
}  // namespace

mfx_status launch_split_elementwise(Handle* h, int64_t n, const float* x, uint16_t* hi, uint16_t* lo, hipStream_t s) {
  if(n == 0) return MFX_SUCCESS;
  const int grid = (int)std::min<int64_t>(ceil_div(n, 256), 65536);
  return timed_launch(h, "split_bf16_elementwise", s, [&] { split_elementwise_kernel<<<grid, 256, 0, s>>>(n, x, hi, lo); });
}

}  // namespace mfx
