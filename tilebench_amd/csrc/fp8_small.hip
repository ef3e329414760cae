// Scaled fp8 GEMMs of few rows (row/column scales: tb_fp8_scaled_gemm; 128 x 128
// block scales: tb_fp8_block_gemm).
//
// Such a call is bound by reading the weights (and, per column tile, the rows of
// A) once; 256 x 256 tiles leave most CUs idle: 32 rows x 8192 columns are 32
// blocks, 65 us for 67 MB of weights.  Here a block owns 32 MB rows x 32 columns
// and its KS wavefronts split K, so N / 32 blocks of KS wavefronts stream the
// weights at once.  Each wavefront loads its MFMA fragments straight from
// global memory into registers, D steps of 128 bytes of K ahead, with no LDS and
// no barrier in the loop: a fragment byte is used by one wavefront only, so
// staging it would only add the trip through LDS.
//
//   lanes : lane (r = lane % 32, h = lane / 32) loads 16-byte chunks h, 2 + h, 4 +
//           h and 6 + h of row r's 128 bytes (A and W alike, so the products
//           pair up whatever order the MFMA takes the bytes in): an instruction
//           covers 32 consecutive bytes of 32 rows;
//   bounds: buffer loads with an out-of-range offset for rows past M or N and for
//           steps past the wavefront's range (zeros, no traffic), so no load
//           sits behind a branch;
//   sums  : the KS partial sums go through LDS and are added in wavefront order
//           in fp32 (results are reproducible bit for bit), then scaled and
//           rounded once to bf16.
// Block scales: P = the step's two MFMAs from zero, acc += (sa * sw) * P in fp32
// (one FMA per element), the order of blocks within a wavefront's range.
#include "fp8_small.h"

#include "tb_common.h"

namespace tb {
namespace fp8s {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));

constexpr int TN = 32, STEP = 128, ROW = TN + 4;  // fp32 per staged row (16-byte pad)

// Blocks go round-robin over the 8 XCDs: each takes a contiguous run of tiles
// (row tiles of one column together), so that its L2 holds each weight row once.
__device__ __forceinline__ int xcd_run(int bid, int nb) {
  const int x = bid & 7, q = nb >> 3, rem = nb & 7;
  return x * q + min(x, rem) + (bid >> 3);
}

template <int MB, int KS, int D, bool BLK>
__global__ void __launch_bounds__(64 * KS, KS / 4 > 0 ? KS / 4 : 1)
    fp8_skinny(const uint8_t* __restrict__ Aq, const uint8_t* __restrict__ WqT, const float* __restrict__ sa,
               const float* __restrict__ sw, uint16_t* __restrict__ Y, int M, int N, int K, int tiles_m) {
  __shared__ __attribute__((aligned(16))) float part[KS][32 * MB * ROW];
  const int idx = xcd_run(blockIdx.x, gridDim.x);
  const int n0 = idx / tiles_m * TN, m0 = idx % tiles_m * (32 * MB);
  const int t = threadIdx.x, lane = t & 63, r = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int nk = K / STEP;
  const int k0 = (int)((int64_t)nk * wave / KS), k1 = (int)((int64_t)nk * (wave + 1) / KS);

  const buf_rsrc_t ra = buf_rsrc(Aq, (uint32_t)M * (uint32_t)K), rw = buf_rsrc(WqT, (uint32_t)N * (uint32_t)K);
  const uint32_t w_off = n0 + r < N ? (uint32_t)(n0 + r) * (uint32_t)K + (uint32_t)h * 16u : BUF_OOB;
  uint32_t a_off[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
    a_off[mb] = m0 + 32 * mb + r < M ? (uint32_t)(m0 + 32 * mb + r) * (uint32_t)K + (uint32_t)h * 16u : BUF_OOB;
  const buf_rsrc_t rsa = buf_rsrc(sa, BLK ? (uint32_t)nk * (uint32_t)M * 4u : 0u);
  const buf_rsrc_t rsw = buf_rsrc(sw, BLK ? (uint32_t)((N + 127) / 128) * (uint32_t)nk * 4u : 0u);

  struct Frag {
    i32x4 w[4], a[MB][4];
    float s[MB], b;
  };
  // the loads of step k, out of range past the wavefront's last one
  auto load = [&](Frag& f, int k) __attribute__((always_inline)) {
    const bool live = k < k1;  // uniform
    const uint32_t soff = (uint32_t)(live ? k : 0) * STEP, wo = live ? w_off : BUF_OOB;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      f.w[i] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, wo + 32u * i, soff, 0));
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const uint32_t ao = live ? a_off[mb] : BUF_OOB;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        f.a[mb][i] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(ra, ao + 32u * i, soff, 0));
    }
    if constexpr (BLK) {
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        const int m = m0 + 32 * mb + r;
        const uint32_t so = m < M && live ? ((uint32_t)k * (uint32_t)M + (uint32_t)m) * 4u : BUF_OOB;
        f.s[mb] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsa, so, 0, 0));
      }
      const uint32_t bo = live ? ((uint32_t)(n0 / 128) * (uint32_t)nk + (uint32_t)k) * 4u : BUF_OOB;
      f.b = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsw, bo, 0, 0));
    }
  };
  f32x16 acc[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) acc[mb] = f32x16{};
  // transposed product (W first): a lane holds four consecutive columns of one row per group of four elements
  auto mma = [&](const Frag& f) __attribute__((always_inline)) {
    const i32x8 w0 = __builtin_shufflevector(f.w[0], f.w[1], 0, 1, 2, 3, 4, 5, 6, 7);
    const i32x8 w1 = __builtin_shufflevector(f.w[2], f.w[3], 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const i32x8 a0 = __builtin_shufflevector(f.a[mb][0], f.a[mb][1], 0, 1, 2, 3, 4, 5, 6, 7);
      const i32x8 a1 = __builtin_shufflevector(f.a[mb][2], f.a[mb][3], 0, 1, 2, 3, 4, 5, 6, 7);
      f32x16 p = BLK ? f32x16{} : acc[mb];
      p = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w0, a0, p, 0, 0, 0, 0, 0, 0);
      p = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w1, a1, p, 0, 0, 0, 0, 0, 0);
      if constexpr (BLK) {
        const float s = f.s[mb] * f.b;
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[mb][e] = __builtin_fmaf(p[e], s, acc[mb][e]);
      } else {
        acc[mb] = p;
      }
    }
  };

  Frag f[D];
#pragma unroll
  for (int d = 0; d < D; ++d) load(f[d], k0 + d);
  for (int k = k0; k < k1; k += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (d > 0 && k + d >= k1) break;  // uniform
      mma(f[d]);
      __builtin_amdgcn_sched_barrier(0);
      load(f[d], k + d + D);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // element 4g + e of acc[mb]: row 32 mb + r, column 8 g + 4 h + e of the tile
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<f32x4*>(&part[wave][(32 * mb + r) * ROW + 8 * g + 4 * h]) =
          f32x4{acc[mb][4 * g], acc[mb][4 * g + 1], acc[mb][4 * g + 2], acc[mb][4 * g + 3]};
  __syncthreads();
  for (int q = t; q < 32 * MB * (TN / 4); q += 64 * KS) {
    const int row = q / (TN / 4), c = q % (TN / 4) * 4;
    const int m = m0 + row, n = n0 + c;
    if (m >= M || n >= N) continue;  // N % 8 == 0: four columns are all in or all out
    f32x4 v = *reinterpret_cast<const f32x4*>(&part[0][row * ROW + c]);
#pragma unroll
    for (int w = 1; w < KS; ++w) {
      const f32x4 u = *reinterpret_cast<const f32x4*>(&part[w][row * ROW + c]);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += u[e];
    }
    if constexpr (!BLK) {
      const float s = sa[m];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = v[e] * s * sw[n + e];
    }
    u32x2 o;
    o[0] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2v{v[0], v[1]}), bf16x2v));
    o[1] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2v{v[2], v[3]}), bf16x2v));
    *reinterpret_cast<u32x2*>(Y + (int64_t)m * N + n) = o;
  }
}

template <int MB, bool BLK>
tb_status launch(const char* fn, const Fp8Args& a, hipStream_t stream) {
  constexpr int KS = 4, D = 2;  // 8 wavefronts or deeper prefetch measured 0 - 5 % slower
  const int64_t tiles_m = (a.M + 32 * MB - 1) / (32 * MB), tiles_n = (a.N + TN - 1) / TN;
  TB_CHECK_ARG(tiles_m * tiles_n < (1ll << 31), "%s: problem too large", fn);
  hipLaunchKernelGGL((fp8_skinny<MB, KS, D, BLK>), dim3((unsigned)(tiles_m * tiles_n)), dim3(64 * KS), 0, stream, a.Aq,
                     a.WqT, a.sa, a.sw, a.Y, a.M, a.N, a.K, (int)tiles_m);
  return tb::launch_status(fn);
}

template <bool BLK>
tb_status launch_rows(const char* fn, int rows, const Fp8Args& a, hipStream_t stream) {
  if (rows == 32) return launch<1, BLK>(fn, a, stream);
  if (rows == 64) return launch<2, BLK>(fn, a, stream);
  return launch<4, BLK>(fn, a, stream);
}

tb_status launch_skinny(const char* fn, int rows, bool block_scaled, const Fp8Args& a, hipStream_t stream) {
  return block_scaled ? launch_rows<true>(fn, rows, a, stream) : launch_rows<false>(fn, rows, a, stream);
}

}  // namespace fp8s
}  // namespace tb
