// Launchers of the small W4A16 tiles (w4a16_small.hip).
#pragma once
#include "small_plan.h"
#include "w4a16_tile.h"

namespace tb {
namespace w4a16 {

// Y [M, N] = A [M, K] @ dequant(W [K, N]).
struct DenseArgs {
  const _Float16* A;
  const uint8_t* W;
  const _Float16* S;
  const uint8_t* Z;
  _Float16* Y;
  int M, N, K, group;
};

// One product per expert: rows of the row space (offsets[e] .. offsets[e + 1] is
// expert e's) times W [K, N].  T_PLAIN: rows are A's and Y's.  T_GATE_UP: A is
// X [tokens, K], row m reads token ids[m] / topk, W is W13 (N = 2 I) and Y
// [rows, I].  T_DOWN: row m is scaled by weights[ids[m]] and stored at row
// ids[m] of Y.
struct ExpertArgs {
  const _Float16* A;
  const int* ids;
  const int* offsets;
  const float* weights;
  const uint8_t* W;
  const _Float16* S;
  const uint8_t* Z;
  _Float16* Y;
  int tokens, topk;
  int64_t rows;
  int experts, N, K, group;
};

// `tile` for tb_gemm_tile.
void describe_dense_small(plan::DenseTile tile, int64_t M, tb_tile* out);
void describe_experts_small(plan::ExpertTile tile, tb_tile* out);

tb_status launch_dense_small(const char* fn, plan::DenseTile tile, const DenseArgs& a, hipStream_t stream);

// Arguments checked by the caller (the limits of the 256-row kernels).
tb_status launch_experts_small(const char* fn, TileMode mode, plan::ExpertTile tile, const ExpertArgs& a,
                               hipStream_t stream);

}  // namespace w4a16
}  // namespace tb
