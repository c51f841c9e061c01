// Block-scaled FP8 (OCP e4m3) contractions on v_mfma_scale_f32_32x32x64_f8f6f4.
//
// Quantisation (one workgroup per 128 x 128 block; both operands in one
// launch): the block's
// largest magnitude fixes a power-of-two scale 2^e (the smallest e with
// amax <= 448 * 2^e), every element becomes q = e4m3_rne(x * 2^-e).  Powers of
// two make the scale an E8M0 byte that the MFMA applies itself, per operand,
// so products need no rescaling pass.  Two-term mode quantises the residual
// x - q1 * 2^e1 the same way (q2, e2) and contracts q1*q1 + q1*q2 + q2*q1.
//
// Packed layout (A role: rows = M; B role: rows = N), fragment order of the
// 32x32x64 MFMA: P[blk32][kb64][half][lane][16 bytes], lane l holding row
// blk32*32 + l%32 and k = kb64*64 + 32*(l/32) + 16*half + 0..15.  Rows and k
// are zero-padded to the tile and to 128.  Exponents: E[row/128][k/128].
//
// Contraction tiles: 256x256 (four waves of 128x128, or eight of 128x64),
// 128x128 (four waves of 64x64) or 64x64 (waves of 32x32);
// each wave's rows and columns lie inside one 128-block, so its A and B
// scales are one byte each per stage.  Stage = 128 k (single) or 64 k
// (two-term), up to four of them in LDS, filled by direct global-to-LDS loads,
// 16-byte chunks read conflict-free.  Tiles that do not fill a round of the
// CUs run as k slices (SplitPlan).
#include "lds_pipe.h"

namespace mfx {

int fp8_config_count();
bool fp8_config_info(int c, int* bm, int* bn, int* bk, int* waves);

namespace {

typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// Quantisation
// ---------------------------------------------------------------------------
struct QuantOperand {
  const float* src;
  int64_t ld;
  int rows, K;
  int kmajor;       // element (r, k) at src[r*ld + k], else src[k*ld + r]
  int vec;          // 16-byte aligned rows: 128-bit loads along the contiguous dimension
  int row_blocks, k_blocks;  // blocks of the padded operand
  u32x4* q1;        // packed, fragment order
  u32x4* q2;
  int* e1;          // [row_blocks][k_blocks]
  int* e2;
  // plain row-major output (mfx_quantize_fp8_block)
  uint8_t* plain;
  int64_t plain_ld;
};
struct QuantParams {
  QuantOperand a, b;
  int grid_a;  // workgroups of a; the rest are b's
};

// Largest v of the workgroup's NT threads.
template <int NT>
__device__ __forceinline__ float block_max(float v, float* sh) {
  for(int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
  if constexpr(NT > 64) {
    __syncthreads();
    if((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    v = sh[0];
#pragma unroll
    for(int i = 1; i < NT / 64; ++i) v = fmaxf(v, sh[i]);
  }
  return v;
}

// e4m3 codes of four floats, packed little-endian into one word, by the
// hardware conversion (v_cvt_pk_fp8_f32: OCP E4M3FN, round to nearest even).
// Inputs are scaled so |x| <= 448 (the block scale guarantees it), so no
// saturation is needed.
__device__ __forceinline__ uint32_t e4m3_pack4(float a, float b, float c, float d) {
  int w = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
  w = __builtin_amdgcn_cvt_pk_fp8_f32(c, d, w, true);
  return (uint32_t)w;
}

// Value of byte `j` (0..3) of a word of e4m3 codes (v_cvt_f32_fp8).
template <int J>
__device__ __forceinline__ float e4m3_byte(uint32_t w) {
  return __builtin_amdgcn_cvt_f32_fp8((int)w, J);
}

// Row pitch (bytes) of the LDS code tile: 128 codes + 16, so 16-byte reads
// of one column by consecutive rows spread over the banks.
constexpr int QPITCH = 144;

// One workgroup per B x B block, sixteen elements per thread in four 16-byte
// loads: of four rows, 4 k each (k-contiguous source; half a wave covers a
// 512-byte row segment), or of 4 k, four rows each (row-contiguous source; 8
// threads cover 128 bytes of a row of the source), so a thread packs four
// code words either way.  Neighbouring workgroups take neighbouring blocks
// along the source's contiguous dimension.  HBM-bound; sixteen elements per
// thread instead of sixty-four keep the two passes over the block (largest
// magnitude, codes) short and the CU full: a 16384^2 operand 288 us (4.65
// TB/s) -> 262 us (5.1 TB/s); the operands of a 1500 x 1100 x 2000 call 14.4 + 13.1
// -> 13 us in one launch.
template <int B, int T, bool PLAIN>
__global__ __launch_bounds__(B * B / 16) void quantize_fp8_kernel(const QuantParams pp) {
  constexpr int NT = B * B / 16;
  __shared__ float sh[16];
  __shared__ __align__(16) unsigned char qtile[PLAIN ? 1 : T][PLAIN ? 16 : 128 * QPITCH];
  const bool first = (int)blockIdx.x < pp.grid_a;
  const QuantOperand& p = first ? pp.a : pp.b;
  const int id = first ? blockIdx.x : blockIdx.x - pp.grid_a;
  const int rb = p.kmajor ? id / p.k_blocks : id % p.row_blocks;
  const int kb = p.kmajor ? id % p.k_blocks : id / p.row_blocks;
  const int t = threadIdx.x;
  // word w of the thread: codes of row lr + w * row_step, k lk .. lk + 3
  int lr, lk, row_step;
  float v[4][4];  // [word][k]
  float amax = 0.0f;
  if(p.kmajor) {
    lr = t / (B / 4);
    lk = t % (B / 4) * 4;
    row_step = B / 4;
#pragma unroll
    for(int w = 0; w < 4; ++w) {
      const int r = rb * B + lr + w * row_step, k = kb * B + lk;
      const float* src = p.src + (int64_t)r * p.ld + k;
      if(r < p.rows && p.vec && k + 4 <= p.K) {
        const float4 x = *reinterpret_cast<const float4*>(src);
        v[w][0] = x.x;
        v[w][1] = x.y;
        v[w][2] = x.z;
        v[w][3] = x.w;
      } else {
#pragma unroll
        for(int e = 0; e < 4; ++e) v[w][e] = r < p.rows && k + e < p.K ? src[e] : 0.0f;
      }
    }
  } else {
    // a wave covers 32 rows x 32 k
    constexpr int RW = B / 32;  // waves along the rows
    const int wave = t >> 6, lane = t & 63;
    lr = wave % RW * 32 + (lane & 7) * 4;
    lk = wave / RW * 32 + (lane >> 3) * 4;
    row_step = 1;
#pragma unroll
    for(int e = 0; e < 4; ++e) {
      const int r = rb * B + lr, k = kb * B + lk + e;
      const float* src = p.src + (int64_t)k * p.ld + r;
      if(k < p.K && p.vec && r + 4 <= p.rows) {
        const float4 x = *reinterpret_cast<const float4*>(src);
        v[0][e] = x.x;
        v[1][e] = x.y;
        v[2][e] = x.z;
        v[3][e] = x.w;
      } else {
#pragma unroll
        for(int w = 0; w < 4; ++w) v[w][e] = k < p.K && r + w < p.rows ? src[w] : 0.0f;
      }
    }
  }
#pragma unroll
  for(int w = 0; w < 4; ++w)
#pragma unroll
    for(int e = 0; e < 4; ++e) amax = fmaxf(amax, fabsf(v[w][e]));
  const int ex1 = fp8_block_exponent(block_max<NT>(amax, sh));
  const float inv1 = ldexpf(1.0f, -ex1), s1 = ldexpf(1.0f, ex1);
  uint32_t w1[4], w2[4];
  float amax2 = 0.0f;
#pragma unroll
  for(int w = 0; w < 4; ++w) {
    float* x = v[w];
    w1[w] = e4m3_pack4(x[0] * inv1, x[1] * inv1, x[2] * inv1, x[3] * inv1);
    if constexpr(T == 2) {
      x[0] -= e4m3_byte<0>(w1[w]) * s1;
      x[1] -= e4m3_byte<1>(w1[w]) * s1;
      x[2] -= e4m3_byte<2>(w1[w]) * s1;
      x[3] -= e4m3_byte<3>(w1[w]) * s1;
      amax2 = fmaxf(amax2, fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3]))));
    }
  }
  if(t == 0) p.e1[(int64_t)rb * p.k_blocks + kb] = ex1;
  if constexpr(T == 2) {
    const int ex2 = fp8_block_exponent(block_max<NT>(amax2, sh));
    const float inv2 = ldexpf(1.0f, -ex2);
    if(t == 0) p.e2[(int64_t)rb * p.k_blocks + kb] = ex2;
#pragma unroll
    for(int w = 0; w < 4; ++w) w2[w] = e4m3_pack4(v[w][0] * inv2, v[w][1] * inv2, v[w][2] * inv2, v[w][3] * inv2);
  }
  if constexpr(PLAIN) {
#pragma unroll
    for(int w = 0; w < 4; ++w) {
      const int r = rb * B + lr + w * row_step, k = kb * B + lk;
      if(r < p.rows)
        for(int e = 0; e < 4 && k + e < p.K; ++e) p.plain[(int64_t)r * p.plain_ld + k + e] = (uint8_t)(w1[w] >> (8 * e));
    }
  } else {
    static_assert(B == 128, "fragment order holds 128 x 128 blocks");
#pragma unroll
    for(int w = 0; w < 4; ++w) {
      *reinterpret_cast<uint32_t*>(&qtile[0][(lr + w * row_step) * QPITCH + lk]) = w1[w];
      if constexpr(T == 2) *reinterpret_cast<uint32_t*>(&qtile[T - 1][(lr + w * row_step) * QPITCH + lk]) = w2[w];
    }
    // The block's 1024 fragment-order chunks, consecutive threads on
    // consecutive chunks: chunk (blk, kb64, half, lane) holds the codes of row
    // blk*32 + lane%32, k = kb64*64 + 32*(lane/32) + 16*half + 0..15.
    __syncthreads();
    const int kb64s = p.k_blocks * 2;
    const int lane = t & 63, half = (t >> 6) & 1, kb64l = (t >> 7) & 1, blkl = t >> 8;
    const int row = blkl * 32 + (lane & 31), col = kb64l * 64 + 32 * (lane >> 5) + 16 * half;
    const int64_t at = ((((int64_t)(rb * 4 + blkl)) * kb64s + kb * 2 + kb64l) * 2 + half) * 64 + lane;
    p.q1[at] = *reinterpret_cast<const u32x4*>(&qtile[0][row * QPITCH + col]);
    if constexpr(T == 2) p.q2[at] = *reinterpret_cast<const u32x4*>(&qtile[T - 1][row * QPITCH + col]);
  }
}

// ---------------------------------------------------------------------------
// Contraction
// ---------------------------------------------------------------------------
struct Fp8TileArgs {
  const u32x4* A1;
  const u32x4* A2;
  const u32x4* B1;
  const u32x4* B2;
  const int* eA1;
  const int* eA2;
  const int* eB1;
  const int* eB2;
  int kb128s;            // padded K / 128
  int nblk_a, nblk_b;    // 32-row blocks held by A / B (rows padded to 128)
};

struct Fp8Params {
  Fp8TileArgs t;
  int tiles_m, tiles_n, group;
  SplitPlan plan;  // workgroups [0, head) take whole tiles, the rest slices
  float* partial;
  Epilogue ep;
};

template <int BM, int BN, int WM, int WN, int T>
struct Fp8Cfg {
  static constexpr int NWN = BN / WN, NT = (BM / WM) * (BN / WN) * 64;
  static constexpr int FM = WM / 32, FN = WN / 32;
  static constexpr int KS = T == 1 ? 2 : 1;                   // 64-wide k steps per stage
  static constexpr int RUN = KS * 2 * 64;                     // chunks of one 32-row block per stage and term
  static constexpr int CH_A = BM / 32 * RUN * T, CH_B = BN / 32 * RUN * T;
  static constexpr int PER_A = CH_A / NT, PER_B = CH_B / NT;
  static constexpr int FIT = 160 * 1024 / (16 * (CH_A + CH_B + NT / 4));
  static constexpr int NB = FIT < 4 ? FIT : 4;                // stages buffered
  static_assert(CH_A % NT == 0 && CH_B % NT == 0, "stage must split evenly");
  static_assert(WM <= 128 && 128 % WM == 0 && WN <= 128 && 128 % WN == 0, "a wave must sit in one scale block");
  static_assert(NB >= 2 && (NB - 1) * (PER_A + PER_B + 1) < 64, "in-flight DMA count fits vmcnt");
  // stages, and a 64-int slot of scales per buffer and wave
  static constexpr int SMEM_CHUNKS = NB * (CH_A + CH_B + NT / 4);
};

// Contracts k blocks (128 k) [s0, s1) of tile (tm, tn) and writes alpha * sum +
// beta * C through `ep` at row er, column ec.
//
// The pipeline is bf16_tile's: LDS reads of the next fragments between the
// MFMAs of the current ones and across the stage boundary, DMA of the stage
// NB further on spread over the MFMAs behind the barrier.  Two whole fragment
// sets would not fit 256 registers beside the accumulators (96 registers a set
// with two terms), so a product walks its A fragments in turn and each is
// replaced by the one that follows it as soon as its MFMAs are issued; only
// the B fragments, which live through the product, are held twice.  With one
// term the follower is the next k step's; with two, the A fragments go q2,
// then q1 (read during q2*q1, kept through q1*q2 and q1*q1), then the next
// stage's q2 (read during q1*q1, behind the boundary).
//
// A wave's scales (one per operand, term and 128 k) travel with the stage: one
// more DMA instruction per wave copies its four exponents into a slot beside
// the stage.  (Scalar loads in the loop return out of order with the LDS
// reads, so that every wait for one is a wait for all.)
template <int BM, int BN, int WM, int WN, int T>
__device__ __forceinline__ void fp8_tile(const Fp8TileArgs& t, int tm, int tn, int s0, int s1, const Epilogue& ep,
    int er, int ec, u32x4* lds) {
  using Cfg = Fp8Cfg<BM, BN, WM, WN, T>;
  constexpr int NT = Cfg::NT, FM = Cfg::FM, FN = Cfg::FN, KS = Cfg::KS, RUN = Cfg::RUN, NB = Cfg::NB;
  constexpr int SA = Cfg::CH_A, SB = Cfg::CH_B, STAGE = SA + SB, PER = Cfg::PER_A + Cfg::PER_B;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wid / Cfg::NWN, wn = wid % Cfg::NWN;
  // blocks past the operand's last one read it (and its scale) again: they
  // only feed outputs the epilogue does not store
  const int arow128 = min((tm * BM + wm * WM) / 128, t.nblk_a / 4 - 1);
  const int bcol128 = min((tn * BN + wn * WN) / 128, t.nblk_b / 4 - 1);

  floatx16 acc[FM][FN];
#pragma unroll
  for(int i = 0; i < FM; ++i)
#pragma unroll
    for(int j = 0; j < FN; ++j)
#pragma unroll
      for(int q = 0; q < 16; ++q) acc[i][j][q] = 0.0f;

  // DMA instruction i of a wave moves 64 consecutive chunks, contiguous in
  // the packed operand and in the LDS stage (RUN and SA / T are multiples of
  // 64); its source is uniform but for the lane's 16 bytes.
  const int64_t blk_stride = (int64_t)t.kb128s * 4 * 64;
  const int wave_base = wid * 64;
  constexpr int PER128 = 2 / KS;  // stages per 128 k
  int next = s0 * PER128;
  const int last = s1 * PER128;
  int64_t koff = (int64_t)next * RUN;
  u32x4* dst = lds;
  const u32x4* base[PER];
#pragma unroll
  for(int i = 0; i < PER; ++i) {
    const bool is_a = i < Cfg::PER_A;
    const int c = wave_base + (is_a ? i : i - Cfg::PER_A) * NT;
    const int term = c / ((is_a ? SA : SB) / T), cc = c % ((is_a ? SA : SB) / T);
    const int blk = cc / RUN, run = cc - blk * RUN;
    const u32x4* src = is_a ? (term ? t.A2 : t.A1) : (term ? t.B2 : t.B1);
    base[i] = src + (int64_t)(is_a ? min(tm * (BM / 32) + blk, t.nblk_a - 1) : min(tn * (BN / 32) + blk, t.nblk_b - 1)) * blk_stride + run;
  }
  auto issue_one = [&](int i) __attribute__((always_inline)) {
    const bool is_a = i < Cfg::PER_A;
    const char* src = reinterpret_cast<const char*>(base[i] + koff);
    lds_dma16(reinterpret_cast<const u32x4*>(src + (uint32_t)lane * 16),
        dst + (is_a ? i * NT : SA + (i - Cfg::PER_A) * NT) + wave_base);
  };
  // lane l fetches exponent l % 4 of (q1 of A, q1 of B, q2 of A, q2 of B)
  const int which = lane & 3;
  const int* escale = which == 0 ? t.eA1 : which == 1 ? t.eB1 : which == 2 ? t.eA2 : t.eB2;
  escale += (int64_t)(which & 1 ? bcol128 : arow128) * t.kb128s;
  int* const slots = reinterpret_cast<int*>(lds + NB * STAGE) + wid * 64;  // [buffer][wave][64]
  constexpr int SLOT = NT;                                                // ints of one buffer
  int kb_next = s0, slot_next = 0;
  auto issue_scales = [&]() __attribute__((always_inline)) {
    lds_dma4(escale + kb_next, slots + slot_next * SLOT);
  };
  struct Scales {
    int a1, b1, a2, b2;  // biased: E8M0 bytes
  };
  auto read_scales = [&](int slot) __attribute__((always_inline)) {
    const u32x4 e = *reinterpret_cast<const u32x4*>(slots + slot * SLOT);
    return Scales{(int)e.x + 127, (int)e.y + 127, (int)e.z + 127, (int)e.w + 127};
  };

  auto advance = [&]() __attribute__((always_inline)) {
    ++next;
    dst = dst + STAGE == lds + NB * STAGE ? lds : dst + STAGE;
    // past the end: the last stage again, into a buffer no one reads
    koff = next < last ? koff + RUN : koff;
    kb_next = min(next, last - 1) / PER128;
    slot_next = slot_next + 1 == NB ? 0 : slot_next + 1;
  };

  auto frag = [&](const u32x4* panel, int blk, int ks) __attribute__((always_inline)) {
    const u32x4* f = panel + blk * RUN + ks * 128 + lane;
    return __builtin_bit_cast(i32x8, __builtin_shufflevector(f[0], f[64], 0, 1, 2, 3, 4, 5, 6, 7));
  };
  // Calls b(j) and a(i) for the fragments to read before MFMA m of a product:
  // the B fragments first, A fragment i once the MFMAs of its predecessor in
  // place i are issued.
  auto reads_at = [&](auto mm, auto&& rb, auto&& ra) __attribute__((always_inline)) {
    constexpr int m = decltype(mm)::value, i = m / FN, j = m % FN;
    if constexpr(i == 0) rb(std::integral_constant<int, j>{});
    if constexpr(j == 0 && i > 0) ra(std::integral_constant<int, i - 1>{});
    if constexpr(m == FM * FN - 1) ra(std::integral_constant<int, FM - 1>{});
  };
  constexpr int NM = FM * FN;  // MFMAs of one product
  using Yes = std::true_type;
  using No = std::false_type;
  auto boundary = [&]() __attribute__((always_inline)) {
    // the next stage has landed (the NB - 2 issued after it may still be in
    // flight) and this wave has read all of the current one
    vm_wait<(NB - 2) * (PER + 1)>();
    lds_wait();
    bare_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  auto following = [&](const u32x4* st) __attribute__((always_inline)) {
    return st + STAGE == lds + NB * STAGE ? (const u32x4*)lds : st + STAGE;
  };

  if(last > next) {
#pragma unroll
    for(int p = 0; p < NB; ++p) {
#pragma unroll
      for(int i = 0; i < PER; ++i) issue_one(i);
      issue_scales();
      advance();
    }
    vm_wait<(NB - 1) * (PER + 1)>();  // the first stage
    bare_barrier();
    const u32x4* st = lds;
    int slot = 0;
    Scales sc = read_scales(0), sn = sc;
    if constexpr(T == 1) {
      i32x8 a[2][FM], b[2][FN];
      auto contract = [&](auto qq, const u32x4* p, int ks, auto reads, auto dma) __attribute__((always_inline)) {
        constexpr int q = decltype(qq)::value;
        static_for<NM>([&](auto mm) __attribute__((always_inline)) {
          constexpr int m = decltype(mm)::value, i = m / FN, j = m % FN;
          if constexpr(decltype(reads)::value)
            reads_at(mm, [&](auto x) __attribute__((always_inline)) { b[1 - q][x] = frag(p + SA, wn * FN + x, ks); },
                [&](auto x) __attribute__((always_inline)) { a[1 - q][x] = frag(p, wm * FM + x, ks); });
          constexpr int d0 = m * PER / NM, d1 = (m + 1) * PER / NM;
          if constexpr(decltype(dma)::value)
            static_for<d1 - d0>([&](auto x) __attribute__((always_inline)) { issue_one(d0 + decltype(x)::value); });
          acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a[q][i], b[q][j], acc[i][j], 0, 0, 0, sc.a1, 0, sc.b1);
          __builtin_amdgcn_sched_barrier(0);
        });
      };
      using Q0 = std::integral_constant<int, 0>;
      using Q1 = std::integral_constant<int, 1>;
      static_for<FN>([&](auto x) __attribute__((always_inline)) { b[0][x] = frag(st + SA, wn * FN + x, 0); });
      static_for<FM>([&](auto x) __attribute__((always_inline)) { a[0][x] = frag(st, wm * FM + x, 0); });
      for(int s = s0; s + 1 < s1; ++s) {
        contract(Q0{}, st, 1, Yes{}, No{});
        boundary();
        st = following(st);
        slot = slot + 1 == NB ? 0 : slot + 1;
        sn = read_scales(slot);
        issue_scales();
        contract(Q1{}, st, 0, Yes{}, Yes{});
        advance();
        sc = sn;
      }
      contract(Q0{}, st, 1, Yes{}, No{});
      contract(Q1{}, st, 0, No{}, No{});
    } else {
      i32x8 a1[FM], a2[FM], b1[FN], b2[FN], nb1[FN];
      auto q2q1 = [&](const u32x4* p) __attribute__((always_inline)) {
        static_for<NM>([&](auto mm) __attribute__((always_inline)) {
          constexpr int m = decltype(mm)::value, i = m / FN, j = m % FN;
          reads_at(mm, [&](auto x) __attribute__((always_inline)) { b2[x] = frag(p + SA + SB / 2, wn * FN + x, 0); },
              [&](auto x) __attribute__((always_inline)) { a1[x] = frag(p, wm * FM + x, 0); });
          acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a2[i], b1[j], acc[i][j], 0, 0, 0, sc.a2, 0, sc.b1);
          __builtin_amdgcn_sched_barrier(0);
        });
      };
      auto q1q2 = [&]() __attribute__((always_inline)) {
        static_for<NM>([&](auto mm) __attribute__((always_inline)) {
          constexpr int m = decltype(mm)::value, i = m / FN, j = m % FN;
          acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a1[i], b2[j], acc[i][j], 0, 0, 0, sc.a1, 0, sc.b2);
          __builtin_amdgcn_sched_barrier(0);
        });
      };
      auto q1q1 = [&](const u32x4* p, auto more) __attribute__((always_inline)) {
        static_for<NM>([&](auto mm) __attribute__((always_inline)) {
          constexpr int m = decltype(mm)::value, i = m / FN, j = m % FN;
          if constexpr(decltype(more)::value) {
            reads_at(mm, [&](auto x) __attribute__((always_inline)) { nb1[x] = frag(p + SA, wn * FN + x, 0); },
                [&](auto x) __attribute__((always_inline)) { a2[x] = frag(p + SA / 2, wm * FM + x, 0); });
            constexpr int d0 = m * PER / NM, d1 = (m + 1) * PER / NM;
            static_for<d1 - d0>([&](auto x) __attribute__((always_inline)) { issue_one(d0 + decltype(x)::value); });
          }
          acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a1[i], b1[j], acc[i][j], 0, 0, 0, sc.a1, 0, sc.b1);
          __builtin_amdgcn_sched_barrier(0);
        });
      };
      static_for<FN>([&](auto x) __attribute__((always_inline)) { b1[x] = frag(st + SA, wn * FN + x, 0); });
      static_for<FM>([&](auto x) __attribute__((always_inline)) { a2[x] = frag(st + SA / 2, wm * FM + x, 0); });
      for(int s = s0 * PER128; s + 1 < last; ++s) {
        q2q1(st);
        q1q2();
        boundary();
        st = following(st);
        slot = slot + 1 == NB ? 0 : slot + 1;
        sn = read_scales(slot);
        issue_scales();
        q1q1(st, Yes{});
#pragma unroll
        for(int j = 0; j < FN; ++j) b1[j] = nb1[j];
        advance();
        sc = sn;
      }
      q2q1(st);
      q1q2();
      q1q1(st, No{});
    }
  }
  lds_dma_wait();  // no copy into LDS is left behind

  static_for<FM * FN>([&](auto ij) __attribute__((always_inline)) {
    constexpr int i = decltype(ij)::value / FN, j = decltype(ij)::value % FN;
    store_block32(ep, acc[i][j], er + wm * WM + i * 32, ec + wn * WN + j * 32, lane);
  });
}

template <int BM, int BN, int WM, int WN, int T>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64) void gemm_fp8_kernel(const Fp8Params p) {
  using Cfg = Fp8Cfg<BM, BN, WM, WN, T>;
  __shared__ u32x4 lds[Cfg::SMEM_CHUNKS];
  int tm, tn;
  if((int)blockIdx.x < p.plan.head) {
    grouped_tile(xcd_remap(blockIdx.x, p.plan.head), p.tiles_m, p.tiles_n, p.group, tm, tn);
    fp8_tile<BM, BN, WM, WN, T>(p.t, tm, tn, 0, p.t.kb128s, p.ep, tm * BM, tn * BN, lds);
    return;
  }
  // slice-major, as in gemm_bf16x_kernel
  const int rest = p.tiles_m * p.tiles_n - p.plan.head, splits = p.plan.splits;
  const int id = xcd_remap(blockIdx.x - p.plan.head, rest * splits);
  const int slice = id / rest, tile = id - slice * rest;
  grouped_tile(p.plan.head + tile, p.tiles_m, p.tiles_n, p.group, tm, tn);
  const int s0 = (int)((int64_t)p.t.kb128s * slice / splits), s1 = (int)((int64_t)p.t.kb128s * (slice + 1) / splits);
  float* slot = p.partial + ((int64_t)tile * splits + slice) * (BM * BN);
  const Epilogue ep{slot, BN, 1.0f, 0.0f, BM, BN, TILES_FULL, 0};
  fp8_tile<BM, BN, WM, WN, T>(p.t, tm, tn, s0, s1, ep, 0, 0, lds);
}

struct Fp8Config {
  int bm, bn, waves;
};
constexpr Fp8Config kFp8Configs[] = {
    {256, 256, 4},  // 0: 128x128 per wave
    {128, 128, 4},  // 1: 64x64 per wave
    {256, 256, 8},  // 2: 128x64 per wave, two waves per SIMD
    {64, 64, 4},    // 3: 32x32 per wave
};
constexpr int kFp8ConfigCount = sizeof(kFp8Configs) / sizeof(kFp8Configs[0]);

struct Fp8Plan {
  int64_t rows_pad_a, rows_pad_b, kb128s;
  size_t q_a, q_b, e_a, e_b;  // bytes of one term
  int64_t tiles;
  SplitPlan split;
  size_t partial;
};

Fp8Plan fp8_plan(const DenseOp& op, bool two_term, int config, int cus, int forced_splits) {
  const Fp8Config& c = kFp8Configs[config];
  Fp8Plan pl;
  pl.rows_pad_a = round_up(op.M, 128);
  pl.rows_pad_b = round_up(op.N, 128);
  pl.kb128s = round_up(std::max(op.K, 1), 128) / 128;
  pl.q_a = (size_t)pl.rows_pad_a * pl.kb128s * 128;
  pl.q_b = (size_t)pl.rows_pad_b * pl.kb128s * 128;
  pl.e_a = (size_t)(pl.rows_pad_a / 128) * pl.kb128s * 4;
  pl.e_b = (size_t)(pl.rows_pad_b / 128) * pl.kb128s * 4;
  pl.tiles = ceil_div(op.M, c.bm) * ceil_div(op.N, c.bn);
  pl.split = SplitPlan{(int)pl.tiles, 1};
  if(forced_splits >= 2) {
    int64_t s = std::min<int64_t>(forced_splits, pl.kb128s);
    while(s > 1 && pl.tiles * s * c.bm * c.bn * 4 > kMaxPartialBytes) --s;
    if(s > 1) pl.split = SplitPlan{0, (int)s};
  } else if(forced_splits < 0) {
    plan_splits(two_term ? MFX_PREC_FP8_BLOCK2 : MFX_PREC_FP8_BLOCK, config, pl.tiles, pl.kb128s * 128, cus,
        kMaxPartialBytes, &pl.split);
  }
  pl.partial = pl.split.splits > 1 ? (size_t)(pl.tiles - pl.split.head) * pl.split.splits * c.bm * c.bn * 4 : 0;
  return pl;
}

template <int BM, int BN, int WM, int WN>
void launch_fp8_cfg(const Fp8Params& p, bool two_term, int grid, hipStream_t s) {
  if(two_term) gemm_fp8_kernel<BM, BN, WM, WN, 2><<<grid, Fp8Cfg<BM, BN, WM, WN, 2>::NT, 0, s>>>(p);
  else gemm_fp8_kernel<BM, BN, WM, WN, 1><<<grid, Fp8Cfg<BM, BN, WM, WN, 1>::NT, 0, s>>>(p);
}

QuantOperand quant_operand(const float* src, int64_t ld, int rows, int K, bool kmajor, int64_t rows_pad, int64_t kb128s,
    u32x4* q1, u32x4* q2, int* e1, int* e2) {
  QuantOperand o{};
  o.src = src;
  o.ld = ld;
  o.rows = rows;
  o.K = K;
  o.kmajor = kmajor;
  o.vec = (reinterpret_cast<uintptr_t>(src) & 15u) == 0 && ld % 4 == 0;
  o.row_blocks = (int)(rows_pad / 128);
  o.k_blocks = (int)kb128s;
  o.q1 = q1;
  o.q2 = q2;
  o.e1 = e1;
  o.e2 = e2;
  return o;
}

}  // namespace

int fp8_config_count() { return kFp8ConfigCount; }
bool fp8_config_info(int c, int* bm, int* bn, int* bk, int* waves) {
  if(c < 0 || c >= kFp8ConfigCount) return false;
  *bm = kFp8Configs[c].bm;
  *bn = kFp8Configs[c].bn;
  *bk = 128;
  *waves = kFp8Configs[c].waves;
  return true;
}

// Bytes of the packed operands and their exponents.
static size_t fp8_packed(const Fp8Plan& pl, bool two_term) {
  const int terms = two_term ? 2 : 1;
  return terms * (round_up(pl.q_a, 256) + round_up(pl.q_b, 256) + round_up(pl.e_a, 256) + round_up(pl.e_b, 256));
}

size_t dense_fp8_workspace(const DenseOp& op, bool two_term, int config, int cus) {
  if(config < 0 || config >= kFp8ConfigCount) return 0;
  const Fp8Plan pl = fp8_plan(op, two_term, config, cus, -1);
  return fp8_packed(pl, two_term) + pl.partial;
}

mfx_status launch_dense_fp8(Handle* h, const DenseOp& op, bool two_term, int config, hipStream_t s) {
  if(config < 0 || config >= kFp8ConfigCount) return invalid("FP8 tile configuration out of range");
  if(op.nprod != 1 || op.tiles != TILES_FULL) return unsupported("FP8 is built for plain gemm (not syrk / syr2k)");
  if(op.M == 0 || op.N == 0) return MFX_SUCCESS;
  Fp8Plan pl = fp8_plan(op, two_term, config, cus_of(h), h->forced_splits);
  void *ws = nullptr, *partials = nullptr;
  MFX_CHECK(packed_workspace(h, fp8_packed(pl, two_term), pl.partial, s, &ws, &partials));
  if(pl.partial > 0 && !partials) {
    config = whole_config(h, two_term ? MFX_PREC_FP8_BLOCK2 : MFX_PREC_FP8_BLOCK, op, config);
    pl = fp8_plan(op, two_term, config, cus_of(h), 1);
  }
  char* w = static_cast<char*>(ws);
  auto take = [&](size_t bytes) {
    char* p = w;
    w += round_up(bytes, 256);
    return p;
  };
  u32x4* qa1 = reinterpret_cast<u32x4*>(take(pl.q_a));
  u32x4* qb1 = reinterpret_cast<u32x4*>(take(pl.q_b));
  int* ea1 = reinterpret_cast<int*>(take(pl.e_a));
  int* eb1 = reinterpret_cast<int*>(take(pl.e_b));
  u32x4 *qa2 = nullptr, *qb2 = nullptr;
  int *ea2 = nullptr, *eb2 = nullptr;
  if(two_term) {
    qa2 = reinterpret_cast<u32x4*>(take(pl.q_a));
    qb2 = reinterpret_cast<u32x4*>(take(pl.q_b));
    ea2 = reinterpret_cast<int*>(take(pl.e_a));
    eb2 = reinterpret_cast<int*>(take(pl.e_b));
  }
  QuantParams q;
  q.a = quant_operand(op.A, op.lda, op.M, op.K, op.a_kmajor, pl.rows_pad_a, pl.kb128s, qa1, qa2, ea1, ea2);
  q.b = quant_operand(op.B, op.ldb, op.N, op.K, op.b_kmajor, pl.rows_pad_b, pl.kb128s, qb1, qb2, eb1, eb2);
  q.grid_a = q.a.row_blocks * q.a.k_blocks;
  const int qgrid = q.grid_a + q.b.row_blocks * q.b.k_blocks;
  MFX_CHECK(timed_launch(h, two_term ? "quantize_fp8_block2" : "quantize_fp8_block", s, [&] {
    if(two_term) quantize_fp8_kernel<128, 2, false><<<qgrid, 1024, 0, s>>>(q);
    else quantize_fp8_kernel<128, 1, false><<<qgrid, 1024, 0, s>>>(q);
  }));
  const Fp8Config& c = kFp8Configs[config];
  Fp8Params p;
  p.t = Fp8TileArgs{qa1, qa2 ? qa2 : qa1, qb1, qb2 ? qb2 : qb1, ea1, ea2 ? ea2 : ea1, eb1, eb2 ? eb2 : eb1,
      (int)pl.kb128s, (int)(pl.rows_pad_a / 32), (int)(pl.rows_pad_b / 32)};
  p.tiles_m = (int)ceil_div(op.M, c.bm);
  p.tiles_n = (int)ceil_div(op.N, c.bn);
  p.group = 8;
  p.plan = pl.split;
  p.partial = static_cast<float*>(partials);
  p.ep = op.ep;
  const int grid = p.plan.head + ((int)pl.tiles - p.plan.head) * p.plan.splits;
  MFX_CHECK(timed_launch(h, two_term ? "gemm_fp8_block2_mfma" : "gemm_fp8_block_mfma", s, [&] {
    switch(config) {
      case 0: launch_fp8_cfg<256, 256, 128, 128>(p, two_term, grid, s); break;
      case 1: launch_fp8_cfg<128, 128, 64, 64>(p, two_term, grid, s); break;
      case 2: launch_fp8_cfg<256, 256, 128, 64>(p, two_term, grid, s); break;
      case 3: launch_fp8_cfg<64, 64, 32, 32>(p, two_term, grid, s); break;
    }
  }));
  if(p.plan.splits == 1) return MFX_SUCCESS;
  const SplitReduceArgs r{p.partial, c.bm, c.bn, p.plan.splits, p.plan.head, (int)pl.tiles, TILES_FULL, p.tiles_m,
      p.tiles_n, p.group, op.ep};
  return launch_splitk_reduce(h, r, s);
}

mfx_status launch_quantize_fp8(Handle* h, int64_t rows, int64_t cols, const float* x, int64_t ldx, int block,
    uint8_t* q, int32_t* exps, hipStream_t s) {
  if(rows == 0 || cols == 0) return MFX_SUCCESS;
  QuantParams p{};
  QuantOperand& o = p.a;
  o.src = x;
  o.ld = ldx;
  o.rows = (int)rows;
  o.K = (int)cols;
  o.kmajor = 1;
  o.vec = (reinterpret_cast<uintptr_t>(x) & 15u) == 0 && ldx % 4 == 0;
  o.row_blocks = (int)ceil_div(rows, block);
  o.k_blocks = (int)ceil_div(cols, block);
  o.e1 = exps;
  o.plain = q;
  o.plain_ld = cols;
  const int64_t blocks = (int64_t)o.row_blocks * o.k_blocks;
  if(blocks > INT32_MAX) return unsupported("quantize: more than 2^31 blocks");
  p.grid_a = (int)blocks;
  const unsigned grid = (unsigned)blocks;
  return timed_launch(h, "quantize_fp8_block_plain", s, [&] {
    if(block == 128) quantize_fp8_kernel<128, 1, true><<<grid, 1024, 0, s>>>(p);
    else if(block == 64) quantize_fp8_kernel<64, 1, true><<<grid, 256, 0, s>>>(p);
    else quantize_fp8_kernel<32, 1, true><<<grid, 64, 0, s>>>(p);
  });
}

}  // namespace mfx
