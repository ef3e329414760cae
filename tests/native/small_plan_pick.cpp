// Prints what the rules of tilebench_amd/csrc/small_plan.h pick, a line per group of four arguments:
//   dense M N 0          0: 256 x 256, 1: 64 x 64, 2: 64 x 128, 3: 64 x 256, 4: 128 x 256
//   expert rows E N      0: 256 rows, 1: 32 x 128, 2: 32 x 256, 3: 64 x 256
//   fp8 M N K, fp8b M N K (block scales)
//                        0: 256 x 256, 1: 32 x 32, 2: 64 x 64, 3: 64 x 128, 4: 128 x 128
//   nt M N Kb            0: 256 x 256, 1: 64 x 64, 2: 64 x 128, 3: 128 x 128
//   decode CUs N K       columns of a slab, K splits, blocks launched
// Build: g++ -O2 -std=c++17 -I tilebench_amd/csrc tests/native/small_plan_pick.cpp
#include <cstdio>
#include <cstdlib>
#include <string>

#include "small_plan.h"

int main(int argc, char** argv) {
  using namespace tb::plan;
  for (int i = 1; i + 3 < argc; i += 4) {
    const std::string rule = argv[i];
    const long long a = std::atoll(argv[i + 1]), b = std::atoll(argv[i + 2]), c = std::atoll(argv[i + 3]);
    if (rule == "dense")
      std::printf("%d\n", (int)pick_dense_tile(a, b));
    else if (rule == "expert")
      std::printf("%d\n", (int)pick_expert_tile(a, b, c));
    else if (rule == "fp8" || rule == "fp8b")
      std::printf("%d\n", (int)pick_fp8_tile(a, b, c, rule == "fp8b"));
    else if (rule == "nt")
      std::printf("%d\n", (int)pick_nt_tile(a, b, c));
    else if (rule == "decode") {
      const DecodePlan p = pick_decode(b, c, (int)a);
      std::printf("%d %d %lld\n", p.cols, p.splits, (long long)decode_grid(p.cols, p.slabs, p.splits));
    } else {
      std::fprintf(stderr, "unknown rule %s\n", rule.c_str());
      return 1;
    }
  }
  return 0;
}
