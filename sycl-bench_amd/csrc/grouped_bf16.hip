// Grouped kernels for split / single BF16.  A pre-pass kernel packs the
// operands of every problem without producers (the kernel boundary orders it
// before the tiles, with no in-kernel synchronisation).  In the persistent
// kernel, pack items split one 32-row block x PACK_KBLOCKS k blocks of an
// operand of a problem with producers once those are done; tile items run
// bf16_tile (LDS stages filled by global-to-LDS DMA) on the packed operands,
// for consumer problems once every pack item of their panels is published.
#include "grouped.h"

namespace mfx {
namespace {

// One pack item: all loads of a thread are issued before any of its stores
// (the stores could alias the loads as far as the compiler knows, so it
// would not reorder them itself).
template <int NHL, int NT>
__device__ void pack_item(const GProblem& P, bool is_a, int blk, int slice) {
  PackSrc s;
  s.src = is_a ? P.A : P.B;
  s.ld = is_a ? P.lda : P.ldb;
  s.rows = is_a ? P.M : P.N;
  s.K = P.K;
  s.kmajor = is_a ? P.a_kmajor : P.b_kmajor;
  s.vec = is_a ? P.vec_a : P.vec_b;
  u32x4* dst = is_a ? P.packed_a : P.packed_b;
  const int kb0 = slice * PACK_KBLOCKS;
  const int nkb = min(PACK_KBLOCKS, P.kbs - kb0);
  constexpr int PER = PACK_KBLOCKS * 64 / NT;
  float v[PER][8];
#pragma unroll
  for(int i = 0; i < PER; ++i) {
    const int c = threadIdx.x + i * NT;
    if((c >> 6) < nkb) load_chunk8(s, blk, kb0 + (c >> 6), c & 63, v[i]);
  }
#pragma unroll
  for(int i = 0; i < PER; ++i) {
    const int c = threadIdx.x + i * NT;
    if((c >> 6) < nkb) store_chunk<NHL>(dst, blk, kb0 + (c >> 6), c & 63, P.kbs, v[i]);
  }
}

// Pre-pass: block b packs chunks of the job whose block range holds b (jobs
// start on 256-chunk blocks, so each wave's 64 chunks are one (blk, kb)
// pair, as load_chunk8_staged needs; a non-k-major source walks the pairs
// kb-major, neighbouring waves on neighbouring row segments).
template <int NHL>
__global__ __launch_bounds__(256) void pack_jobs_kernel(const PackJob* jobs, int njobs) {
  __shared__ float tiles[4][STAGED_TILE_FLOATS];
  int lo = 0, hi = njobs - 1;
  const int b = blockIdx.x;
  while(lo < hi) {
    const int mid = (lo + hi + 1) / 2;
    if(jobs[mid].first_block <= b) lo = mid;
    else hi = mid - 1;
  }
  const PackJob& j = jobs[lo];
  const int64_t c = (int64_t)(b - j.first_block) * 256 + threadIdx.x;
  const bool active = c < j.chunks;
  const int lane = (int)(c & 63);
  const int64_t t = c >> 6;
  if(j.src.kmajor) {
    if(active) pack_chunk<NHL>(j.src, (int)(t / j.kbs), (int)(t % j.kbs), lane, j.kbs, j.dst);
    return;
  }
  const int nblk = (int)(j.chunks / ((int64_t)j.kbs * 64));
  const int blk = (int)(t % nblk), kb = (int)(t / nblk);
  float v[8];
  load_chunk8_staged(j.src, blk, kb, lane, active, v, tiles[threadIdx.x >> 6]);
  if(active) store_chunk<NHL>(j.dst, blk, kb, lane, j.kbs, v);
}

// Pre-pack item: chunks [b0 * 256, (b0 + nb) * 256) of the segment's pre-pack
// job list (pack_jobs_kernel's numbering: jobs start on 256-chunk blocks, so
// the 64 chunks of one wave and one pass slot are one (blk, kb) pair of one
// job).  Each thread keeps U chunks' global loads in flight per pass; a
// non-k-major source goes through the wave's own LDS tiles (U per wave, in
// the tile's LDS, which no tile uses while the workgroup runs this item).
template <int NHL, int NT, int U>
__device__ __forceinline__ void prepack_item(const PackJob* jobs, int njobs, int b0, int nb, float* tiles) {
  const int tid = threadIdx.x, lane = tid & 63;
  float* wtile = tiles + (tid >> 6) * U * STAGED_TILE_FLOATS;
  const int64_t c_end = (int64_t)(b0 + nb) * 256;
  for(int64_t base = (int64_t)b0 * 256; base < c_end; base += (int64_t)NT * U) {
    int jix[U], blk[U], kb[U];
    bool act[U], kmaj[U];
    float v[U][8];
    float4 x[U][2];
#pragma unroll
    for(int i = 0; i < U; ++i) {
      const int64_t c = base + tid + i * NT;
      // one 256-chunk block per wave and slot: the search runs on scalars
      const int b = __builtin_amdgcn_readfirstlane((int)(c >> 8));
      int lo = 0, hi = njobs - 1;
      while(lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if(jobs[mid].first_block <= b) lo = mid;
        else hi = mid - 1;
      }
      const PackJob& J = jobs[lo];
      jix[i] = lo;
      const int64_t local = c - (int64_t)J.first_block * 256;
      act[i] = c < c_end && local < J.chunks;
      kmaj[i] = J.src.kmajor != 0;
      const int64_t t = local >> 6;
      if(kmaj[i]) {
        blk[i] = (int)(t / J.kbs);
        kb[i] = (int)(t % J.kbs);
        if(act[i]) load_chunk8(J.src, blk[i], kb[i], lane, v[i]);
      } else {
        const int nblk = (int)(J.chunks / ((int64_t)J.kbs * 64));
        blk[i] = (int)(t % nblk);
        kb[i] = (int)(t / nblk);
        staged_load(J.src, blk[i], kb[i], lane, act[i], x[i]);
      }
    }
#pragma unroll
    for(int i = 0; i < U; ++i)
      if(!kmaj[i]) staged_write(x[i], lane, wtile + i * STAGED_TILE_FLOATS);
    __syncthreads();
#pragma unroll
    for(int i = 0; i < U; ++i)
      if(!kmaj[i]) staged_read(lane, wtile + i * STAGED_TILE_FLOATS, v[i]);
#pragma unroll
    for(int i = 0; i < U; ++i)
      if(act[i]) store_chunk<NHL>(jobs[jix[i]].dst, blk[i], kb[i], lane, jobs[jix[i]].kbs, v[i]);
    __syncthreads();  // the next pass rewrites the tiles
  }
}

// Grouped tiles mostly stream panels that no other running tile shares, so
// they run the deeper pipeline: four buffers of half a stage, three in
// flight, in the LDS that bf16_tile uses for two.
// The 64x64 tile, whose direct stages hold 8 KiB, buffers eight.
constexpr int PIPE_NB = 4;
template <int C>
constexpr int direct_nb() {
  return C == 2 ? 8 : PIPE_NB;
}
template <int NHL>
constexpr int pipe_kb() {
  return kb_per_stage<NHL>() / 2;
}

template <int NHL, int C>
__device__ __forceinline__ void run_tile(const BfTileArgs& t, int tm, int tn, u32x4* lds) {
  bf16_tile_pipe<Geo<C>::BM, Geo<C>::BN, Geo<C>::WM, Geo<C>::WN, NHL, pipe_kb<NHL>(), PIPE_NB>(t, tm, tn, lds);
}

template <int NHL, int C>
__device__ __forceinline__ void run_direct(const DirectTileArgs& t, int tm, int tn, u32x4* lds) {
  bf16_tile_direct<Geo<C>::BM, Geo<C>::BN, Geo<C>::WM, Geo<C>::WN, NHL, direct_nb<C>()>(t, tm, tn, lds);
}

template <int NHL, int C>
constexpr int bf16_smem_chunks() {
  constexpr int p = BfPipeCfg<Geo<C>::BM, Geo<C>::BN, Geo<C>::WM, Geo<C>::WN, NHL, pipe_kb<NHL>(), PIPE_NB>::SMEM_CHUNKS;
  constexpr int d = BfDirectCfg<Geo<C>::BM, Geo<C>::BN, Geo<C>::WM, Geo<C>::WN, direct_nb<C>()>::SMEM_CHUNKS;
  return p > d ? p : d;
}

template <int NHL, int BIG, int SMALL>
__global__ __launch_bounds__(geo_threads<BIG>()) void grouped_bf16x_kernel(const GroupedArgs g) {
  constexpr int NT = geo_threads<BIG>();
  static_assert(geo_threads<SMALL>() == NT, "both tiles of a policy use the same workgroup");
  constexpr int S0 = bf16_smem_chunks<NHL, BIG>(), S1 = bf16_smem_chunks<NHL, SMALL>();
  __shared__ u32x4 lds[S0 > S1 ? S0 : S1];
  __shared__ int slot, ready, tried;
  // pre-pack chunks in flight per thread: as many per-wave LDS tiles as fit
  constexpr int LDS_FLOATS = (S0 > S1 ? S0 : S1) * 4;
  constexpr int U = LDS_FLOATS / (NT / 64 * STAGED_TILE_FLOATS) < 4 ? LDS_FLOATS / (NT / 64 * STAGED_TILE_FLOATS) : 4;
  static_assert(U >= 1, "the tile's LDS holds at least one staging tile per wave");
  if(threadIdx.x == 0) tried = 0;
  for(;;) {
    const int it = take_item(g, &slot, &tried);
    if(it < 0) break;
    const GItem item = g.items[it];
    if(item.type == ITEM_PREPACK) {
      prepack_item<NHL, NT, U>(g.prejobs, g.nprejobs, item.x, item.y, reinterpret_cast<float*>(lds));
      continue;
    }
    const GProblem& P = g.problems[item.problem];
    const int bm = cfg_bm(P.config), bn = cfg_bn(P.config);
    if(item.type != ITEM_TILE) {
      const bool is_a = item.type == ITEM_PACK_A;
      if(P.ndeps > 0 && !wg_wait(&ready, [&] { return poll_producers(P, g); })) continue;
      pack_item<NHL, NT>(P, is_a, item.x, item.y);
      const int panel = item.x * 32 / (is_a ? bm : bn);
      signal(&g.pack_ctr[(is_a ? P.pack_a_ctr : P.pack_b_ctr) + panel]);
      continue;
    }
    if(P.direct) {
      // in-kernel mode: the producers' results are read straight from C
      if(P.ndeps > 0 && !wg_wait(&ready, [&] { return poll_producers(P, g); })) continue;
      DirectTileArgs d;
      d.a = DirectOp{P.A, P.lda, P.M, P.a_kmajor};
      d.b = DirectOp{P.B, P.ldb, P.N, P.b_kmajor};
      d.K = P.K;
      d.ep = Epilogue{P.C, P.ldc, P.alpha, P.beta, P.M, P.N, TILES_FULL, 0};
      if constexpr(BIG == SMALL) {
        run_direct<NHL, BIG>(d, item.x, item.y, lds);
      } else {
        if(P.config == BIG) run_direct<NHL, BIG>(d, item.x, item.y, lds);
        else run_direct<NHL, SMALL>(d, item.x, item.y, lds);
      }
      if(P.consumed) signal(&g.done[item.problem]);
      continue;
    }
    const int nblk_a = (P.M + 31) / 32, nblk_b = (P.N + 31) / 32;
    if(!P.prepacked && P.pack_slices > 0) {
      // pack items of a panel: its 32-row blocks that meet the matrix, each in pack_slices k slices
      const int need_a = (min((item.x + 1) * (bm / 32), nblk_a) - item.x * (bm / 32)) * P.pack_slices;
      const int need_b = (min((item.y + 1) * (bn / 32), nblk_b) - item.y * (bn / 32)) * P.pack_slices;
      if(!wg_wait(&ready, [&] {
           return poll_at_least(&g.pack_ctr[P.pack_a_ctr + item.x], need_a, g) &&
                  poll_at_least(&g.pack_ctr[P.pack_b_ctr + item.y], need_b, g);
         }))
        continue;
    } else if(!P.prepacked && P.ndeps > 0) {
      // K == 0: no pack items, but the tile still rewrites C (beta * C), so
      // it waits for the producers like any other consumer
      if(!wg_wait(&ready, [&] { return poll_producers(P, g); })) continue;
    }
    BfTileArgs t;
    t.PA = P.packed_a;
    t.PB = P.packed_b;
    t.kbs = P.kbs;
    t.nblk_a = nblk_a;
    t.nblk_b = nblk_b;
    t.nprod = 1;
    t.ep = Epilogue{P.C, P.ldc, P.alpha, P.beta, P.M, P.N, TILES_FULL, 0};
    if constexpr(BIG == SMALL) {
      run_tile<NHL, BIG>(t, item.x, item.y, lds);
    } else {
      if(P.config == BIG) run_tile<NHL, BIG>(t, item.x, item.y, lds);
      else run_tile<NHL, SMALL>(t, item.x, item.y, lds);
    }
    if(P.consumed) signal(&g.done[item.problem]);
  }
}

template <int NHL, int BIG, int SMALL>
void launch_one(const GroupedArgs& g, int grid, hipStream_t s) {
  grouped_bf16x_kernel<NHL, BIG, SMALL><<<grid, geo_threads<BIG>(), 0, s>>>(g);
}

template <int NHL>
bool launch_pair(int big, int small, const GroupedArgs& g, int grid, hipStream_t s) {
  switch(big * 8 + small) {
    case 0 * 8 + 0: launch_one<NHL, 0, 0>(g, grid, s); return true;
    case 0 * 8 + 1: launch_one<NHL, 0, 1>(g, grid, s); return true;
    case 0 * 8 + 2: launch_one<NHL, 0, 2>(g, grid, s); return true;
    case 3 * 8 + 3: launch_one<NHL, 3, 3>(g, grid, s); return true;
    case 3 * 8 + 1: launch_one<NHL, 3, 1>(g, grid, s); return true;
    case 3 * 8 + 2: launch_one<NHL, 3, 2>(g, grid, s); return true;
    case 1 * 8 + 1: launch_one<NHL, 1, 1>(g, grid, s); return true;
    case 1 * 8 + 2: launch_one<NHL, 1, 2>(g, grid, s); return true;
    case 2 * 8 + 2: launch_one<NHL, 2, 2>(g, grid, s); return true;
    case 4 * 8 + 4: launch_one<NHL, 4, 4>(g, grid, s); return true;
    case 4 * 8 + 5: launch_one<NHL, 4, 5>(g, grid, s); return true;
    case 4 * 8 + 6: launch_one<NHL, 4, 6>(g, grid, s); return true;
    case 5 * 8 + 5: launch_one<NHL, 5, 5>(g, grid, s); return true;
    case 5 * 8 + 6: launch_one<NHL, 5, 6>(g, grid, s); return true;
    case 6 * 8 + 6: launch_one<NHL, 6, 6>(g, grid, s); return true;
  }
  return false;
}

}  // namespace

mfx_status launch_pack_jobs(Handle* h, int nhl, const PackJob* jobs, int njobs, int blocks, hipStream_t s) {
  if(njobs == 0 || blocks == 0) return MFX_SUCCESS;
  return timed_launch(h, nhl == 2 ? "grouped_pack_split_bf16" : "grouped_pack_bf16", s, [&] {
    if(nhl == 2) pack_jobs_kernel<2><<<blocks, 256, 0, s>>>(jobs, njobs);
    else pack_jobs_kernel<1><<<blocks, 256, 0, s>>>(jobs, njobs);
  });
}

mfx_status launch_grouped_bf16(Handle* h, int nhl, int big, int small, bool vec, const GroupedArgs& g, int grid,
    hipStream_t s) {
  (void)vec;  // pack items choose their load width per operand
  bool known = false;
  const mfx_status st = timed_launch(h, nhl == 2 ? "grouped_split_bf16_mfma" : "grouped_bf16_mfma", s, [&] {
    known = nhl == 2 ? launch_pair<2>(big, small, g, grid, s) : launch_pair<1>(big, small, g, grid, s);
  });
  if(st == MFX_SUCCESS && !known) return invalid("no grouped BF16 kernel for this tile pair");
  return st;
}

}  // namespace mfx
