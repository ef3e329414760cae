// Prints the tile that tilebench_amd/csrc/small_plan.h picks for each
// "rows experts N" triple on the command line (0: 256 rows, 1: 32 x 128,
// 2: 32 x 256, 3: 64 x 256); experts = 0 asks for the dense product of rows x N
// (0: 256 x 256, 1: 64 x 64, 2: 64 x 128, 3: 64 x 256, 4: 128 x 256), experts =
// -K / -K - 1 for the row- / block-scaled fp8 product (0: 256 x 256, 1: 32 x 32, 2:
// 64 x 64, 3: 64 x 128, 4: 128 x 128), experts = -10^9 - bytes of K for the plain
// product (0: 256 x 256, 1: 64 x 64, 2: 64 x 128, 3: 128 x 128), experts = -2 *
// 10^9 - K for the W4A16 decode of K x N on a device of `rows` CUs (10^9 x blocks
// launched + 1000 x columns of a slab + K splits).
// Build: g++ -O2 -std=c++17 -I tilebench_amd/csrc tests/native/small_plan_pick.cpp
#include <cstdio>
#include <cstdlib>

#include "small_plan.h"

int main(int argc, char** argv) {
  for (int i = 1; i + 2 < argc; i += 3) {
    const long long rows = std::atoll(argv[i]), experts = std::atoll(argv[i + 1]), N = std::atoll(argv[i + 2]);
    long long pick;
    if (experts <= -2000000000) {
      const auto p = tb::plan::pick_decode(N, -experts - 2000000000, (int)rows);
      pick = 1000000000ll * tb::plan::decode_grid(p.cols, p.slabs, p.splits) + 1000 * p.cols + p.splits;
    } else if (experts <= -1000000000)
      pick = (int)tb::plan::pick_nt_tile(rows, N, -experts - 1000000000);
    else if (experts < 0)
      pick = (int)tb::plan::pick_fp8_tile(rows, N, -experts / 128 * 128, experts % 128 != 0);
    else
      pick = experts ? (int)tb::plan::pick_expert_tile(rows, experts, N) : (int)tb::plan::pick_dense_tile(rows, N);
    std::printf("%lld\n", pick);
  }
  return 0;
}
