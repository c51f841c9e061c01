// One BM x BN output tile of an FP32 contraction on v_mfma_f32_32x32x2_f32,
// shared by the single-problem kernels (gemm_f32.hip) and the persistent
// grouped kernel (grouped_f32.hip).
//
// A workgroup of (BM/WM) x (BN/WN) waves; each wave owns a WM x WN sub-tile
// held as (WM/32) x (WN/32) 32x32 accumulator blocks.  The operands go from
// global memory straight into LDS, 16 k of both panels per stage, several
// stages in flight, in a layout the DMA writes as it is and the MFMAs read as
// it is.  One 32-row block of an operand and stage is 512 floats:
//   k-contiguous operand (element (r, k) at p[r*ld + k]): 128 chunks of four
//     floats (kchunk_at);
//   row-contiguous operand (element (r, k) at p[k*ld + r]): a 16 x 32 (k x r)
//     array.
// Lane l feeds row l%32 to the MFMA and supplies k slot l/32 of its two, so
// half stage h, step e contracts k = 4h + e and 8 + 4h + e: any pairing of
// the k's is the same sum, and this one makes a lane's values of a half stage
// one 16-byte LDS read.
#pragma once

#include "lds_pipe.h"

namespace mfx {

constexpr int F32_BK = 16;  // k per stage and k-group

// Stages buffered: four, eight of the 64x64 tile (whose stage is 512 cycles of
// MFMA per wave).
template <int BM, int BN>
constexpr int f32_stages() {
  return BM * BN <= 64 * 64 ? 8 : 4;
}

// VEC: 16-byte copies into LDS, else 4-byte ones (four times as many).
// WANT: stages to buffer, as far as their copies fit vmcnt.
// KG: groups of waves that each contract the whole tile over their own 16 k of
// every KG * 16 deep stage (two waves per SIMD on a tile of four sub-tiles:
// one issues MFMAs while the other is at the barrier); their accumulators are
// summed through LDS at the end.
template <int BM, int BN, int WM, int WN, bool VEC, int WANT = f32_stages<BM, BN>(), int KG = 1>
struct F32Cfg {
  static constexpr int NWM = BM / WM, NWN = BN / WN, NWG = NWM * NWN, NW = NWG * KG, NT = NW * 64;
  static constexpr int FM = WM / 32, FN = WN / 32;
  static constexpr int BK = F32_BK * KG;
  static constexpr int FL_A = BM * BK, FL_B = BN * BK, STAGE = FL_A + FL_B;  // floats per stage
  static constexpr int W = VEC ? 4 : 1;                                              // floats per lane and copy
  static constexpr int PER_A = FL_A / (NT * W), PER_B = FL_B / (NT * W), PER = PER_A + PER_B;
  static constexpr int NB = WANT < 63 / PER + 1 ? WANT : 63 / PER + 1;
  static constexpr int SMEM_FLOATS = NB * STAGE;
  static_assert(FL_A % (NT * W) == 0 && FL_B % (NT * W) == 0, "stage must split evenly over threads");
  static_assert(NB >= 2 && (NB - 1) * PER < 64, "in-flight copies fit vmcnt");
  static_assert((KG - 1) * BM * BN <= NB * STAGE, "the other groups' accumulators fit the stages");
};

// 128-bit copies need 16-byte aligned rows and a contiguous extent that is a
// multiple of 4 (so a chunk is entirely inside or outside the matrix).
inline bool f32_vec_ok(const float* P, int64_t ld, bool kmajor, int rows, int K) {
  const int contig = kmajor ? K : rows;
  return (reinterpret_cast<uintptr_t>(P) & 15u) == 0 && ld % 4 == 0 && contig % 4 == 0;
}

// Float f of a stage's ROWS-row panel ([16 k][32-row block][512 floats]): its
// row within the panel and k within the stage.
template <int ROWS, bool KMAJOR, bool VEC>
__device__ __forceinline__ void f32_place(int f, int& r, int& k) {
  const int sub = f / (ROWS * F32_BK), blk = f % (ROWS * F32_BK) >> 9, g = f & 511;
  if(KMAJOR) {
    const int chunk = g >> 2;
    r = blk * 32 + kchunk_row(chunk);
    k = sub * F32_BK + 4 * kchunk_kq(chunk) + (VEC ? 0 : g & 3);
  } else {
    r = blk * 32 + (g & 31);
    k = sub * F32_BK + (g >> 5);
  }
}

// Contracts stages [s0, s1) of tile (tm, tn) of `op` (a product's stages are
// ceil(K / (16 KG)), the second product's follow the first's) and writes alpha *
// sum + beta * C through `ep` at row er, column ec.  `smem` holds
// F32Cfg::SMEM_FLOATS floats; the caller separates two calls that reuse it
// with a barrier.
//
// The pipeline is bf16_tile's (tile_bf16.h): the LDS reads of the next half
// stage between the MFMAs of the current one, across the stage boundary too,
// and the copies of the stage NB further on spread over the MFMAs behind the
// barrier.  The earlier form went through registers (global loads, then
// transposing LDS stores with both waves of a SIMD waiting at the barrier
// behind them) and lost 15 to 20 % of the MFMA time on big tiles, a third on
// small ones.  Measured on MI355X with a tile on every CU, ns per k before ->
// after: 256x256 250 -> 220 (130 -> 146 TFLOP/s), 128x128 80 -> 62, 64x64
// 20.8 -> 17.5.  With one wave per SIMD a stage costs about 300 cycles beyond
// its MFMAs (64x64: 21.0), with two the other wave's MFMAs fill them; four
// groups of the 64x64 tile are no better (19.6).
//
// Rows past the operand read its last row again and only feed outputs the
// epilogue does not store.  k past the end (K % 16) reads k inside it again
// and is zeroed in both operands' fragments in the last stage, so Inf and NaN
// stay where they belong.
template <int BM, int BN, int WM, int WN, bool AK, bool BKM, bool VEC, int WANT = f32_stages<BM, BN>(),
    int KG = 1>
__device__ __forceinline__ void f32_tile(const DenseOp& op, int tm, int tn, int s0, int s1, const Epilogue& ep, int er,
    int ec, float* smem) {
  using Cfg = F32Cfg<BM, BN, WM, WN, VEC, WANT, KG>;
  constexpr int NT = Cfg::NT, FM = Cfg::FM, FN = Cfg::FN, NB = Cfg::NB, W = Cfg::W;
  constexpr int STAGE = Cfg::STAGE, PER_A = Cfg::PER_A, PER = Cfg::PER, BK = Cfg::BK;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = KG > 1 ? wid / Cfg::NWG : 0, wave = wid - group * Cfg::NWG;
  const int wm = wave / Cfg::NWN, wn = wave % Cfg::NWN;
  const int m0 = tm * BM, n0 = tn * BN;

  // One 32x32 block per wave would make every MFMA wait for the one before:
  // two accumulators take turns then, added at the end.
  constexpr int NA = FM * FN == 1 ? 2 : 1;
  floatx16 acc[NA][FM][FN];
#pragma unroll
  for(int n = 0; n < NA; ++n)
#pragma unroll
    for(int i = 0; i < FM; ++i)
#pragma unroll
      for(int j = 0; j < FN; ++j)
#pragma unroll
        for(int q = 0; q < 16; ++q) acc[n][i][j][q] = 0.0f;

  const int KT = (op.K + BK - 1) / BK;
  const int tail = op.K % BK;  // k of a partial last stage
  const int hi = lane >> 5;
  const int chunk0 = kchunk_at(lane & 31, 2 * hi), chunk1 = kchunk_at(lane & 31, 2 * hi + 1);

  floatx4 a[2][FM], b[2][FN];
  constexpr int NR = FM + FN;         // fragments per half stage
  constexpr int NM = 4 * FM * FN;     // MFMAs per half stage
  using Yes = std::true_type;
  using No = std::false_type;
  using Q0 = std::integral_constant<int, 0>;
  using Q1 = std::integral_constant<int, 1>;

  // fragment r of half stage h of the stage at `st` into set q
  auto read_one = [&](const float* st, int h, auto qq, auto rr) __attribute__((always_inline)) {
    constexpr int q = decltype(qq)::value, r = decltype(rr)::value;
    constexpr bool is_b = r < FN, KM = is_b ? BKM : AK;
    const float* blk = is_b ? st + Cfg::FL_A + group * BN * F32_BK + (wn * FN + r) * 512
                            : st + group * BM * F32_BK + (wm * FM + r - FN) * 512;
    floatx4 v;
    if constexpr(KM) {
      v = *reinterpret_cast<const floatx4*>(blk + (h ? chunk1 : chunk0) * 4);
    } else {
#pragma unroll
      for(int e = 0; e < 4; ++e) v[e] = blk[(8 * hi + 4 * h + e) * 32 + (lane & 31)];
    }
    if constexpr(is_b) b[q][r] = v;
    else a[q][r - FN] = v;
  };

  // one product's stages [from, to), through the whole pipeline
  auto run = [&](const float* A, int64_t lda, const float* B, int64_t ldb, int from, int to) __attribute__((always_inline)) {
    const float* src[PER];
#pragma unroll
    for(int i = 0; i < PER; ++i) {
      int r, k;
      if(i < PER_A) {
        f32_place<BM, AK, VEC>((tid + i * NT) * W, r, k);
        src[i] = A + (AK ? (int64_t)min(m0 + r, op.M - 1) * lda + k : (int64_t)k * lda + min(m0 + r, op.M - W));
      } else {
        f32_place<BN, BKM, VEC>((tid + (i - PER_A) * NT) * W, r, k);
        src[i] = B + (BKM ? (int64_t)min(n0 + r, op.N - 1) * ldb + k : (int64_t)k * ldb + min(n0 + r, op.N - W));
      }
    }
    int next = from;
    float* dst = smem;
    // a copy's source moves on by one stage as soon as it is issued (one
    // addition of a uniform step); past the end it stays on the last stage,
    // which is then read again into a buffer no one reads
    const int64_t whole_a = AK ? BK : BK * lda, whole_b = BKM ? BK : BK * ldb;
    int64_t step_a, step_b;
    auto steps_for = [&]() __attribute__((always_inline)) {
      step_a = next + 1 < to ? whole_a : 0;
      step_b = next + 1 < to ? whole_b : 0;
    };
    auto issue_one = [&](int i) __attribute__((always_inline)) {
      float* d = dst + ((i < PER_A ? i * NT : Cfg::FL_A / W + (i - PER_A) * NT) + wid * 64) * W;
      if constexpr(VEC) lds_dma16(reinterpret_cast<const floatx4*>(src[i]), reinterpret_cast<floatx4*>(d));
      else lds_dma4(src[i], d);
      src[i] += i < PER_A ? step_a : step_b;
    };
    // the sources of a partial last stage go back inside K
    auto clamp_tail = [&]() __attribute__((always_inline)) {
      if(tail == 0 || next != KT - 1) return;
#pragma unroll
      for(int i = 0; i < PER; ++i) {
        const bool is_a = i < PER_A;
        const bool km = is_a ? AK : BKM;
        int r, k;
        if(is_a) f32_place<BM, AK, VEC>((tid + i * NT) * W, r, k);
        else f32_place<BN, BKM, VEC>((tid + (i - PER_A) * NT) * W, r, k);
        const int over = max(k - (tail - (km ? W : 1)), 0);
        src[i] -= km ? (int64_t)over : (int64_t)over * (is_a ? lda : ldb);
      }
    };
    auto advance = [&]() __attribute__((always_inline)) {
      if(next + 1 < to) {
        ++next;
        clamp_tail();
      } else {
        next = to;
      }
      dst = dst + STAGE == smem + NB * STAGE ? smem : dst + STAGE;
      steps_for();
    };
#pragma unroll
    for(int i = 0; i < PER; ++i) src[i] += (i < PER_A ? whole_a : whole_b) * from;
    clamp_tail();
    steps_for();
    // the MFMAs of fragment set q (half q of its stage); masked: k >= `keep` of
    // the stage zeroed
    auto contract = [&](auto qq, const float* st, int h, auto reads, auto dma, auto masked, int keep) __attribute__((always_inline)) {
      constexpr int q = decltype(qq)::value;
      if constexpr(decltype(masked)::value) {
#pragma unroll
        for(int e = 0; e < 4; ++e) {
          const bool in = group * F32_BK + 8 * hi + 4 * q + e < keep;
#pragma unroll
          for(int i = 0; i < FM; ++i) a[q][i][e] = in ? a[q][i][e] : 0.0f;
#pragma unroll
          for(int j = 0; j < FN; ++j) b[q][j][e] = in ? b[q][j][e] : 0.0f;
        }
      }
      static_for<NM>([&](auto mm) __attribute__((always_inline)) {
        constexpr int m = decltype(mm)::value;
        // the first at once, all of them three quarters through (64x64 tile:
        // before the first MFMA, the only ones that hide their latency)
        constexpr int MR = NM * 3 / 4 > 3 ? NM * 3 / 4 : 1;
        constexpr int r0 = m < MR ? (m * NR + MR - 1) / MR : NR, r1 = m < MR ? ((m + 1) * NR + MR - 1) / MR : NR;
        if constexpr(decltype(reads)::value)
          static_for<r1 - r0>([&](auto x) __attribute__((always_inline)) {
            read_one(st, h, std::integral_constant<int, 1 - q>{}, std::integral_constant<int, r0 + decltype(x)::value>{});
          });
        constexpr int d0 = m * PER / NM, d1 = (m + 1) * PER / NM;
        if constexpr(decltype(dma)::value)
          static_for<d1 - d0>([&](auto x) __attribute__((always_inline)) { issue_one(d0 + decltype(x)::value); });
        constexpr int e = m / (FM * FN), i = m % (FM * FN) / FN, j = m % FN;
        acc[e % NA][i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[q][i][e], b[q][j][e], acc[e % NA][i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      });
    };

#pragma unroll
    for(int p = 0; p < NB; ++p) {
#pragma unroll
      for(int i = 0; i < PER; ++i) issue_one(i);
      advance();
    }
    vm_wait<(NB - 1) * PER>();  // the first stage
    bare_barrier();
    const float* st = smem;
    static_for<NR>([&](auto rr) __attribute__((always_inline)) { read_one(st, 0, Q0{}, rr); });
    for(int s = from; s + 1 < to; ++s) {
      contract(Q0{}, st, 1, Yes{}, No{}, No{}, 0);
      // stage s + 1 has landed (the NB - 2 issued after it may still be in
      // flight) and this wave has read all of stage s
      vm_wait<(NB - 2) * PER>();
      lds_wait();
      bare_barrier();
      __builtin_amdgcn_sched_barrier(0);
      st = st + STAGE == smem + NB * STAGE ? (const float*)smem : st + STAGE;
      contract(Q1{}, st, 0, Yes{}, Yes{}, No{}, 0);
      advance();
    }
    const int keep = tail != 0 && to == KT ? tail : BK;
    contract(Q0{}, st, 1, Yes{}, No{}, Yes{}, keep);
    contract(Q1{}, st, 0, No{}, No{}, Yes{}, keep);
    lds_dma_wait();  // no copy into LDS is left behind
  };

  // the stages of each product that [s0, s1) covers
  if(s1 > s0) {
#pragma clang loop unroll(disable)
    for(int prod = s0 >= KT ? 1 : 0;; ++prod) {
      run(prod ? op.B : op.A, prod ? op.ldb : op.lda, prod ? op.A : op.B, prod ? op.lda : op.ldb,
          max(s0 - prod * KT, 0), min(s1 - prod * KT, KT));
      if(s1 <= (prod + 1) * KT) break;
      __syncthreads();  // the first product's last reads of smem
    }
  }

  if constexpr(NA == 2) acc[0][0][0] += acc[1][0][0];
  if constexpr(KG > 1) {
    __syncthreads();  // every wave is done with the stages
    float* mine = smem + (wave * FM * FN * 16) * 64 + lane;  // + (group - 1) * BM * BN, lane-contiguous
    if(group > 0)
      static_for<FM * FN>([&](auto ij) __attribute__((always_inline)) {
        constexpr int ij_ = decltype(ij)::value;
#pragma unroll
        for(int q = 0; q < 16; ++q) mine[(group - 1) * BM * BN + (ij_ * 16 + q) * 64] = acc[0][ij_ / FN][ij_ % FN][q];
      });
    __syncthreads();
    if(group > 0) return;
#pragma unroll
    for(int g = 0; g < KG - 1; ++g)
      static_for<FM * FN>([&](auto ij) __attribute__((always_inline)) {
        constexpr int ij_ = decltype(ij)::value;
#pragma unroll
        for(int q = 0; q < 16; ++q) acc[0][ij_ / FN][ij_ % FN][q] += mine[g * BM * BN + (ij_ * 16 + q) * 64];
      });
  }
  static_for<FM * FN>([&](auto ij) __attribute__((always_inline)) {
    constexpr int i = decltype(ij)::value / FN, j = decltype(ij)::value % FN;
    store_block32(ep, acc[0][i][j], er + wm * WM + i * 32, ec + wn * WN + j * 32, lane);
  });
}

}  // namespace mfx
