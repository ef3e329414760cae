// What tb_gemm_tile reports (tb_runtime.hip), by the file that launches it.
// Sizes are positive; everything the launchers refuse is left to them.
#pragma once
#include <stdint.h>

#include "tbhip.h"

namespace tb {

void describe_w4a16(int64_t M, int64_t N, int64_t K, tb_tile* out);
void describe_experts(int op, int64_t rows, int64_t N, int64_t experts, tb_tile* out);
void describe_fp8_scaled(int64_t M, int64_t N, int64_t K, tb_tile* out);
void describe_fp8_block(int64_t M, int64_t N, int64_t K, tb_tile* out);
void describe_matmul(int op, int64_t M, int64_t N, int64_t K, tb_tile* out);

}  // namespace tb
