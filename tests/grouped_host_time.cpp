// Host time of planning a grouped launch: choosing the policy of an untuned
// list may cost a few times what planning a given policy costs, and grows with
// the problems, not with problems times dependency levels. Prints "OK", or the
// list that takes longer, and exits non-zero.
#include <algorithm>
#include <chrono>
#include <cstdio>
#include <random>
#include <string>
#include <vector>

#include "grouped.h"

using namespace mfx;

static mfx_gemm_problem prob(int64_t m, int64_t n, int64_t k) {
  float* p = reinterpret_cast<float*>(uintptr_t(0x100000));  // planning reads no operand
  return mfx_gemm_problem{m, n, k, 1.0f, 0.0f, p, k, 0, p, n, 0, p, n};
}

static double plan_us(mfx_precision prec, int policy, const std::vector<mfx_gemm_problem>& list, const std::vector<mfx_dep>& deps) {
  double best = 1e30;
  for(int rep = 0; rep < 30; ++rep) {
    Handle h;
    h.cu_count = 256;
    h.grouped_policy = policy;
    GroupedPlan pl;
    const auto a = std::chrono::steady_clock::now();
    if(plan_grouped(&h, prec, list.data(), (int)list.size(), deps.data(), (int)deps.size(), pl) != MFX_SUCCESS) return 1e30;
    best = std::min(best, std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - a).count());
  }
  return best;
}

int main() {
  struct List {
    const char* name;
    std::vector<mfx_gemm_problem> problems;
    std::vector<mfx_dep> deps;
    double most;  // times the given policy's plan
  };
  std::mt19937 rng(3);
  std::uniform_int_distribution<int> size(32, 512);
  List uneven{"256 uneven problems beside two levels", {}, {}, 4.0}, row{"500 products in a row", {}, {}, 20.0};
  for(int i = 0; i < 256; ++i) uneven.problems.push_back(prob(size(rng), size(rng), size(rng)));
  for(int i = 0; i < 3; ++i) uneven.problems.push_back(prob(512, 512, 512));
  uneven.deps = {{258, 256}, {258, 257}};
  for(int i = 0; i < 500; ++i) {
    row.problems.push_back(prob(128, 128, 128));
    if(i) row.deps.push_back({i, i - 1});
  }
  int bad = 0;
  for(const List& l : {uneven, row})
    for(mfx_precision prec : {MFX_PREC_FP32, MFX_PREC_SPLIT_BF16, MFX_PREC_BF16}) {
      const double given = plan_us(prec, prec == MFX_PREC_FP32 ? 13 : 29, l.problems, l.deps);
      const double chosen = plan_us(prec, -1, l.problems, l.deps);
      std::printf("%s, precision %d: %.1f us with a given policy, %.1f choosing it\n", l.name, (int)prec, given, chosen);
      bad += chosen > l.most * given;
    }
  std::printf(bad ? "FAILED %d\n" : "OK\n", bad);
  return bad ? 1 : 0;
}
