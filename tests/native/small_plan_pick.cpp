// Prints the tile that tilebench_amd/csrc/small_plan.h picks for each
// "rows experts N" triple on the command line (0: 256 rows, 1: 32 x 128,
// 2: 32 x 256, 3: 64 x 256).
// Build: g++ -O2 -std=c++17 -I tilebench_amd/csrc tests/native/small_plan_pick.cpp
#include <cstdio>
#include <cstdlib>

#include "small_plan.h"

int main(int argc, char** argv) {
  for (int i = 1; i + 2 < argc; i += 3)
    std::printf("%d\n", (int)tb::plan::pick_expert_tile(std::atoll(argv[i]), std::atoll(argv[i + 1]), std::atoll(argv[i + 2])));
  return 0;
}
