// Launcher of the small-tile scaled fp8 GEMMs (fp8_small.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "small_plan.h"
#include "tbhip.h"

namespace tb {
namespace fp8s {

// Operands of tb_fp8_scaled_gemm (sa [M], sw [N]) or tb_fp8_block_gemm (sa
// [K / 128, M], sw [ceil(N / 128), K / 128]), checked by the caller.
struct Fp8Args {
  const uint8_t* Aq;
  const uint8_t* WqT;
  const float* sa;
  const float* sw;
  uint16_t* Y;
  int M, N, K;
};

// `tile` for tb_gemm_tile.
void describe_small(plan::Fp8Tile tile, bool block_scaled, int64_t M, int64_t N, tb_tile* out);

tb_status launch_small(const char* fn, plan::Fp8Tile tile, bool block_scaled, const Fp8Args& a, hipStream_t stream);

}  // namespace fp8s
}  // namespace tb
