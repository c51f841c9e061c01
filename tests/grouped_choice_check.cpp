// Host-only check of the untuned choice of a grouped launch: small problems that
// are packed, beside a chain that is read directly and holds nearly all of the
// work, do not change the chain's policy; and a chain with several rounds of 64x64
// tiles a level does not take them in one kernel, where nothing fills the last
// round; but FP32 chains are not priced so, as launches per level are estimated
// low there. Nor does a packed precision's chain take two 64x64 workgroups per CU
// in one kernel where the problems beside it keep both busy; and a chain with many
// rounds of tiles a level stays in one kernel. Prints "OK" or the list that differs.
#include <cstdio>
#include <vector>

#include "grouped.h"

using namespace mfx;

static mfx_gemm_problem prob(int64_t m, int64_t n, int64_t k) {
  float* p = reinterpret_cast<float*>(uintptr_t(0x100000));  // planning reads no operand
  return mfx_gemm_problem{m, n, k, 1.0f, 0.0f, p, (k + 3) / 4 * 4, 0, p, n, 0, p, n};
}

int main() {
  const std::vector<mfx_dep> deps = {{4, 0}, {4, 1}, {5, 2}, {5, 3}, {6, 4}, {6, 5}};
  for(mfx_precision prec : {MFX_PREC_SPLIT_BF16, MFX_PREC_BF16})
    for(int64_t n : {384, 448, 512}) {
      int policy[2];
      for(int extra : {0, 1}) {
        std::vector<mfx_gemm_problem> list(7, prob(n, n, n));
        if(extra) list.push_back(prob(100, 90, 77));
        Handle h;
        h.cu_count = 256;
        GroupedPlan pl;
        if(plan_grouped(&h, prec, list.data(), (int)list.size(), deps.data(), (int)deps.size(), pl) != MFX_SUCCESS) return 1;
        policy[extra] = pl.policy;
      }
      if(policy[0] != policy[1]) {
        std::printf("FAILED precision %d, chain of %d: policy %d, %d with a packed problem beside it\n", (int)prec, (int)n,
            policy[0], policy[1]);
        return 1;
      }
    }
  // fifteen products of 640 in four levels: 238 us on 64x64 tiles in one kernel,
  // 138 on 128x128 (split BF16; 217 and 100 single)
  for(mfx_precision prec : {MFX_PREC_SPLIT_BF16, MFX_PREC_BF16}) {
    std::vector<mfx_dep> chain;
    for(int i = 8; i < 15; ++i)
      for(int j : {2 * i - 16, 2 * i - 15}) chain.push_back({i, j});
    const std::vector<mfx_gemm_problem> list(15, prob(640, 640, 640));
    Handle h;
    h.cu_count = 256;
    GroupedPlan pl;
    if(plan_grouped(&h, prec, list.data(), 15, chain.data(), (int)chain.size(), pl) != MFX_SUCCESS) return 1;
    if(!pl.per_level && pl.small == 2) {
      std::printf("FAILED precision %d: policy %d for the chain of 640\n", (int)prec, pl.policy);
      return 1;
    }
  }
  // FP32, sixteen products of 400: 101 us in one kernel, 134 in a launch per level
  {
    std::vector<mfx_dep> chain;
    for(int i = 8; i < 15; ++i)
      for(int j : {2 * i - 16, 2 * i - 15}) chain.push_back({i, j});
    const std::vector<mfx_gemm_problem> list(15, prob(400, 400, 400));
    Handle h;
    h.cu_count = 256;
    GroupedPlan pl;
    if(plan_grouped(&h, MFX_PREC_FP32, list.data(), 15, chain.data(), (int)chain.size(), pl) != MFX_SUCCESS) return 1;
    if(pl.per_level) {
      std::printf("FAILED policy %d for sixteen FP32 products of 400\n", pl.policy);
      return 1;
    }
  }
  // thirty small problems beside eight chained products of 384: 113 us on two
  // 64x64 workgroups per CU, 73 on 128x128 tiles (split BF16; 100 and 55 single)
  for(mfx_precision prec : {MFX_PREC_SPLIT_BF16, MFX_PREC_BF16}) {
    std::vector<mfx_gemm_problem> list(7, prob(384, 384, 384));
    for(int i = 0; i < 30; ++i) list.push_back(prob(64 + 112 * i % 448, 64 + 176 * i % 448, 64 + 304 * i % 448));
    Handle h;
    h.cu_count = 256;
    GroupedPlan pl;
    if(plan_grouped(&h, prec, list.data(), 37, deps.data(), (int)deps.size(), pl) != MFX_SUCCESS) return 1;
    if(!pl.per_level && pl.small == 2) {
      std::printf("FAILED precision %d: policy %d for the chain of 384 beside thirty problems\n", (int)prec, pl.policy);
      return 1;
    }
  }
  // eight split-BF16 products of 1600 beside small problems: 350 us in one kernel,
  // 382 in a launch per level
  {
    std::vector<mfx_gemm_problem> list(7, prob(1600, 1600, 1600));
    for(int i = 0; i < 20; ++i) list.push_back(prob(64 + 112 * i % 448, 64 + 176 * i % 448, 64 + 304 * i % 448));
    Handle h;
    h.cu_count = 256;
    GroupedPlan pl;
    if(plan_grouped(&h, MFX_PREC_SPLIT_BF16, list.data(), 27, deps.data(), (int)deps.size(), pl) != MFX_SUCCESS) return 1;
    if(pl.per_level) {
      std::printf("FAILED policy %d for the chain of 1600 beside twenty problems\n", pl.policy);
      return 1;
    }
  }
  std::printf("OK\n");
  return 0;
}
