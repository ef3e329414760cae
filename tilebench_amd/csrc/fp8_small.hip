// Scaled fp8 GEMMs (row/column scales: tb_fp8_scaled_gemm; 128 x 128 block
// scales: tb_fp8_block_gemm) whose 256 x 256 tiles would leave most CUs idle: 32
// rows x 8192 columns are 32 such tiles, 65 us for 67 MB of weights.
//
// fp8_skinny, up to about 32 rows, is bound by reading the weights (and the rows
// of A) once.  A block owns 32 rows x 32 columns and its KS wavefronts split K,
// so N / 32 blocks stream the weights at once.  Each wavefront loads its MFMA
// fragments straight from global memory into registers, D steps of 128 bytes of
// K ahead, with no LDS and no barrier in the loop.
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
// fp8_tile, the rest, shares both operands through LDS (see there).
// Block scales: P = the step's MFMAs from zero, acc += (sa * sw) * P in fp32 (one
// FMA per element), in block order within a K group: a wavefront's contiguous range in
// fp8_skinny, the even or the odd steps in fp8_tile with two groups, all of K otherwise.
// fp8_tile without K groups gives the 256 x 256 kernels' bits.
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

template <int KS, int D, bool BLK>
__global__ void __launch_bounds__(64 * KS, KS / 4 > 0 ? KS / 4 : 1)
    fp8_skinny(const uint8_t* __restrict__ Aq, const uint8_t* __restrict__ WqT, const float* __restrict__ sa,
               const float* __restrict__ sw, uint16_t* __restrict__ Y, int M, int N, int K, int tiles_m) {
  __shared__ __attribute__((aligned(16))) float part[KS][32 * ROW];
  const int idx = xcd_run(blockIdx.x, gridDim.x);
  const int n0 = idx / tiles_m * TN, m0 = idx % tiles_m * 32;
  const int t = threadIdx.x, lane = t & 63, r = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int nk = K / STEP;
  const int k0 = (int)((int64_t)nk * wave / KS), k1 = (int)((int64_t)nk * (wave + 1) / KS);

  const buf_rsrc_t ra = buf_rsrc(Aq, (uint32_t)M * (uint32_t)K), rw = buf_rsrc(WqT, (uint32_t)N * (uint32_t)K);
  const uint32_t w_off = n0 + r < N ? (uint32_t)(n0 + r) * (uint32_t)K + (uint32_t)h * 16u : BUF_OOB;
  const uint32_t a_off = m0 + r < M ? (uint32_t)(m0 + r) * (uint32_t)K + (uint32_t)h * 16u : BUF_OOB;
  const buf_rsrc_t rsa = buf_rsrc(sa, BLK ? (uint32_t)nk * (uint32_t)M * 4u : 0u);
  const buf_rsrc_t rsw = buf_rsrc(sw, BLK ? (uint32_t)((N + 127) / 128) * (uint32_t)nk * 4u : 0u);

  struct Frag {
    i32x4 w[4], a[4];
    float s, b;
  };
  // the loads of step k, out of range past the wavefront's last one
  auto load = [&](Frag& f, int k) __attribute__((always_inline)) {
    const bool live = k < k1;  // uniform
    const uint32_t soff = (uint32_t)(live ? k : 0) * STEP, wo = live ? w_off : BUF_OOB, ao = live ? a_off : BUF_OOB;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      f.w[i] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, wo + 32u * i, soff, 0));
#pragma unroll
    for (int i = 0; i < 4; ++i)
      f.a[i] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(ra, ao + 32u * i, soff, 0));
    if constexpr (BLK) {
      const uint32_t so = m0 + r < M && live ? ((uint32_t)k * (uint32_t)M + (uint32_t)(m0 + r)) * 4u : BUF_OOB;
      f.s = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsa, so, 0, 0));
      const uint32_t bo = live ? ((uint32_t)(n0 / 128) * (uint32_t)nk + (uint32_t)k) * 4u : BUF_OOB;
      f.b = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsw, bo, 0, 0));
    }
  };
  f32x16 acc = f32x16{};
  // transposed product (W first): a lane holds four consecutive columns of one row per group of four elements
  auto mma = [&](const Frag& f) __attribute__((always_inline)) {
    const i32x8 w0 = __builtin_shufflevector(f.w[0], f.w[1], 0, 1, 2, 3, 4, 5, 6, 7);
    const i32x8 w1 = __builtin_shufflevector(f.w[2], f.w[3], 0, 1, 2, 3, 4, 5, 6, 7);
    const i32x8 a0 = __builtin_shufflevector(f.a[0], f.a[1], 0, 1, 2, 3, 4, 5, 6, 7);
    const i32x8 a1 = __builtin_shufflevector(f.a[2], f.a[3], 0, 1, 2, 3, 4, 5, 6, 7);
    f32x16 p = BLK ? f32x16{} : acc;
    p = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w0, a0, p, 0, 0, 0, 0, 0, 0);
    p = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w1, a1, p, 0, 0, 0, 0, 0, 0);
    if constexpr (BLK) {
      const float s = f.s * f.b;
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[e] = __builtin_fmaf(p[e], s, acc[e]);
    } else {
      acc = p;
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

  // element 4g + e: row r, column 8 g + 4 h + e of the tile
#pragma unroll
  for (int g = 0; g < 4; ++g)
    *reinterpret_cast<f32x4*>(&part[wave][r * ROW + 8 * g + 4 * h]) =
        f32x4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
  __syncthreads();
  for (int q = t; q < 32 * (TN / 4); q += 64 * KS) {
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

// ------------------------------------------------------------------ 64- and 128-row tiles
// Calls of some hundred rows: enough work that the loads of 32-column blocks
// (every A row once per 32 columns) bound them, too few 256 x 256 tiles to fill
// the device.  One 64 FI x 64 FJ tile per block (FI, FJ = 1 or 2), four
// wavefronts of FI x FJ fragments of 32 x 32; both operands stream HBM -> LDS by DMA, ST stages of 128 bytes of K
// with the row swizzle of the other fp8 kernels (chunk c of row r at slot
// c ^ ((r ^ (r >> 3)) & 7)).  While a 64-byte substep's MFMAs run, the next one's
// fragments are read; the barrier sits between the two substeps of a step, when
// the step's stage has been read by every wavefront and takes the DMAs of the
// step ST later.  KG = 2 runs a second such group of wavefronts, with a ring of its
// own, on every other step, and adds the two sums.  Bound by LDS: at 128 x 128, 64 KiB of fragment reads and 32 KiB
// of DMA writes per step against 512 cycles of MFMAs.
constexpr int MAXKB = 512;
constexpr uint32_t RSRC_DW3 = 0x00020000u;

template <int FI_, int FJ_, int ST_, bool BLK, int KG_ = 1>
struct Tile {
  static constexpr int FI = FI_, FJ = FJ_, ST = ST_, KG = KG_;
  static constexpr int TM = 64 * FI, TN = 64 * FJ;
  static constexpr int A_ST = TM * STEP, STAGE = A_ST + TN * STEP;  // A rows, then W rows
  static constexpr int SA_OFF = ST * STAGE;                         // BLK: the stages' activation scales
  static constexpr int PAD_OFF = SA_OFF + (BLK ? ST * TM * 4 : 0);  // the idle wavefronts' scale DMA lands here
  static constexpr int SW_OFF = PAD_OFF + (BLK ? 256 : 0);          // BLK, after the groups: weight scales, K / 128 floats
  static constexpr int GROUP = SW_OFF;                              // one K group's part
  static constexpr int LDS_BYTES = KG * GROUP + (BLK ? MAXKB * 4 : 0);
  static constexpr int C_STRIDE = TN + 8;  // bf16 per staged row (16-byte pad)
  static_assert(LDS_BYTES <= 160 * 1024 && TM * C_STRIDE * 2 <= ST * STAGE, "LDS budget");
  static_assert(KG == 1 || TM * TN * 4 <= GROUP, "room for the other group's sums");
};

__device__ __forceinline__ i32x4 rsrc4(const void* p, uint32_t bytes) {
  const uint64_t base = (uint64_t)(uintptr_t)p;
  i32x4 r;
  r[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)base);
  r[1] = __builtin_amdgcn_readfirstlane((int)(uint32_t)(base >> 32) & 0xFFFF);
  r[2] = __builtin_amdgcn_readfirstlane((int)bytes);
  r[3] = (int)RSRC_DW3;
  return r;
}
// DMAs into LDS at m0 (wave-uniform base; lane l lands at +16 l or +4 l), as
// inline asm so that the compiler does not tie barriers to their completion;
// the kernel waits for them (vmcnt) before the barrier that publishes them.
__device__ __forceinline__ void dma16(uint32_t lds_addr, uint32_t voff, const i32x4& rsrc, uint32_t soff) {
  asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :
               : "s"(__builtin_amdgcn_readfirstlane((int)lds_addr)), "v"(voff), "s"(rsrc),
                 "s"(__builtin_amdgcn_readfirstlane((int)soff))
               : "memory", "m0");
}
__device__ __forceinline__ void dma4(uint32_t lds_addr, uint32_t voff, const i32x4& rsrc, uint32_t soff) {
  asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dword %1, %2, %3 offen lds"
               :
               : "s"(__builtin_amdgcn_readfirstlane((int)lds_addr)), "v"(voff), "s"(rsrc),
                 "s"(__builtin_amdgcn_readfirstlane((int)soff))
               : "memory", "m0");
}

template <int FI, int FJ, int ST, bool BLK, int KG>
__global__ void __launch_bounds__(256 * KG, 1)
    fp8_tile(const uint8_t* __restrict__ Aq, const uint8_t* __restrict__ WqT, const float* __restrict__ sa,
                const float* __restrict__ sw, uint16_t* __restrict__ Y, int M, int N, int K, int tiles_m) {
  typedef Tile<FI, FJ, ST, BLK, KG> C;
  extern __shared__ __attribute__((aligned(128))) uint8_t lds[];
  const int idx = xcd_run(blockIdx.x, gridDim.x);
  const int n0 = idx / tiles_m * C::TN, m0 = idx % tiles_m * C::TM;
  const int t = threadIdx.x, lane = t & 63, r = lane & 31, h = lane >> 5;
  const int wave8 = __builtin_amdgcn_readfirstlane(t >> 6), wave = wave8 & 3, grp = wave8 >> 2;
  const int wm = wave >> 1, wn = wave & 1;
  const int nk = K / STEP, ni = (nk + KG - 1) / KG;  // steps in all, of a group (its step i is step KG i + grp)
  const i32x4 ra = rsrc4(Aq, (uint32_t)M * (uint32_t)K), rw = rsrc4(WqT, (uint32_t)N * (uint32_t)K);
  const i32x4 rsa = rsrc4(sa, BLK ? (uint32_t)nk * (uint32_t)M * 4u : 0u);
  const uint32_t lds_base = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(uintptr_t)(
      __attribute__((address_space(3))) void*)lds);
  const uint32_t lds0 = lds_base + (uint32_t)(grp * C::GROUP);  // the group's part
  const uint8_t* const part = lds + grp * C::GROUP;
  auto live_rsrc = [](bool live, i32x4 v) __attribute__((always_inline)) {
    v[2] = __builtin_amdgcn_readfirstlane(live ? v[2] : 0);
    return v;
  };

  // DMA d of a step: 8 A rows per instruction for d < DA, 8 W rows for d < DA + DW
  // (lane L: row + L / 8, slot L % 8), then BLK's activation scales (64 rows per
  // wavefront)
  constexpr int DA = 2 * FI, DW = 2 * FJ, PER = DA + DW + (BLK ? 1 : 0);
  uint32_t off[DA + DW], s_off = BUF_OOB;
#pragma unroll
  for (int d = 0; d < DA + DW; ++d) {
    const int row = 8 * (d < DA ? DA * wave + d : DW * wave + d - DA) + (lane >> 3);
    const int c = (lane & 7) ^ ((row ^ (row >> 3)) & 7), g = (d < DA ? m0 : n0) + row;
    off[d] = g < (d < DA ? M : N) ? (uint32_t)g * (uint32_t)K + (uint32_t)c * 16u : BUF_OOB;
  }
  if (BLK && wave < FI && m0 + 64 * wave + lane < M) s_off = (uint32_t)(m0 + 64 * wave + lane) * 4u;
  auto issue_one = [&](int i, int st, int d) __attribute__((always_inline)) {
    const int k = KG * i + grp;
    const bool live = k < nk;  // past the last step: empty resources (zeros, no traffic)
    const uint32_t dst = lds0 + (uint32_t)(st * C::STAGE);
    if (d < DA)
      dma16(dst + (uint32_t)(8 * (DA * wave + d) * STEP), off[d], live_rsrc(live, ra), (uint32_t)(live ? k : 0) * STEP);
    else if (d < DA + DW)
      dma16(dst + (uint32_t)(C::A_ST + 8 * (DW * wave + d - DA) * STEP), off[d], live_rsrc(live, rw),
            (uint32_t)(live ? k : 0) * STEP);
    else
      dma4(lds0 + (uint32_t)(wave < FI ? C::SA_OFF + st * C::TM * 4 + wave * 256 : C::PAD_OFF), s_off,
           live_rsrc(live, rsa), (uint32_t)(live ? k : 0) * (uint32_t)M * 4u);
  };
  if constexpr (BLK) {
    // the tile's weight scales sw[n0 / 128, 0 .. nk - 1], 64 per DMA (first in
    // the queue: landed before step 0's data)
    const i32x4 rsw = rsrc4(sw + (int64_t)(n0 / 128) * nk, (uint32_t)nk * 4u);
    for (int q = wave8; q < (nk + 63) / 64; q += 4 * KG)
      dma4(lds_base + (uint32_t)(KG * C::GROUP + q * 256), q * 64 + lane < nk ? (uint32_t)(q * 64 + lane) * 4u : BUF_OOB, rsw, 0u);
  }

  // fragment f (f < FI: A rows 32 (FI wm + f) .., then W rows 32 (FJ wn + f - FI) ..)
  // of substep s: chunks 4 s + 2 h and 4 s + 2 h + 1 of the lane's row
  typedef __attribute__((address_space(3))) uint8_t lds_u8;
  constexpr int NFR = FI + FJ;
  uint32_t base[NFR][2];  // LDS byte offsets of the two halves; substep 1 flips bit 6
#pragma unroll
  for (int f = 0; f < NFR; ++f)
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int row = 32 * (f < FI ? FI * wm + f : FJ * wn + f - FI) + r;
      base[f][q] = lds0 + (uint32_t)((f < FI ? 0 : C::A_ST) + row * STEP + (((2 * h + q) ^ ((row ^ (row >> 3)) & 7)) << 4));
    }
  struct Frag {
    i32x8 v[NFR];
  };
  auto read_one = [&](Frag& fr, int st, int s, int f) __attribute__((always_inline)) {
    typedef __attribute__((address_space(3))) const i32x4 lds_i4;
    const i32x4 lo = *(lds_i4*)((lds_u8*)(uintptr_t)(base[f][0] ^ (uint32_t)(s << 6)) + st * C::STAGE);
    const i32x4 hi = *(lds_i4*)((lds_u8*)(uintptr_t)(base[f][1] ^ (uint32_t)(s << 6)) + st * C::STAGE);
    fr.v[f] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };

  f32x16 acc[FI][FJ], p[FI][FJ];
#pragma unroll
  for (int i = 0; i < FI; ++i)
#pragma unroll
    for (int j = 0; j < FJ; ++j) acc[i][j] = p[i][j] = f32x16{};
  float s_cur[FI] = {};
  const float* const lsw = reinterpret_cast<const float*>(lds + KG * C::GROUP);
  auto fold = [&](int i, int j) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[i][j][e] = __builtin_fmaf(p[i][j][e], s_cur[i], acc[i][j][e]);
  };

  constexpr int VM0 = PER * (ST - 1), VM1 = PER * (ST - 2);
  static_assert(VM0 < 64, "vmcnt range");
  constexpr int WAIT_PRO = (VM0 & 15) | ((VM0 >> 4) << 14) | (7 << 4) | (15 << 8);
  constexpr int WAIT_STEP = (VM1 & 15) | ((VM1 >> 4) << 14) | (7 << 4) | (0 << 8);
  auto barrier = [&]() __attribute__((always_inline)) {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
#pragma unroll
  for (int st = 0; st < ST; ++st)
#pragma unroll
    for (int d = 0; d < PER; ++d) issue_one(st, st, d);
  __builtin_amdgcn_s_waitcnt(WAIT_PRO);
  barrier();
  Frag f0, f1;
#pragma unroll
  for (int f = 0; f < NFR; ++f) read_one(f0, 0, 0, f);

  constexpr int NQ = FI * FJ;  // MFMAs per substep
  auto step = [&](int i0, int st) __attribute__((always_inline)) {
    // substep 0; the stage's substep 1 read beside its MFMAs
    float s_new[FI] = {};
    if constexpr (BLK) {
      const int k = KG * i0 + grp;
      const float b = KG == 1 || k < nk ? lsw[k] : 0.f;
#pragma unroll
      for (int i = 0; i < FI; ++i)
        s_new[i] = *reinterpret_cast<const float*>(part + C::SA_OFF + st * C::TM * 4 + (32 * (FI * wm + i) + r) * 4) * b;
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int i = q / FJ, j = q % FJ;
      if constexpr (BLK) {
        fold(i, j);  // the previous step's block sum (zeros before the first step)
        p[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(f0.v[FI + j], f0.v[i], f32x16{}, 0, 0, 0, 0, 0, 0);
      } else {
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(f0.v[FI + j], f0.v[i], acc[i][j], 0, 0, 0, 0, 0, 0);
      }
#pragma unroll
      for (int f = 0; f < NFR; ++f)
        if (f * NQ / NFR == q) read_one(f1, st, 1, f);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (BLK) {
#pragma unroll
      for (int i = 0; i < FI; ++i) s_cur[i] = s_new[i];
    }
    // step k + 1 landed, and every wavefront has read this stage
    __builtin_amdgcn_s_waitcnt(WAIT_STEP);
    barrier();
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int i = q / FJ, j = q % FJ;
      f32x16& d = BLK ? p[i][j] : acc[i][j];
      d = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(f1.v[FI + j], f1.v[i], d, 0, 0, 0, 0, 0, 0);
#pragma unroll
      for (int f = 0; f < NFR; ++f)
        if (f * NQ / NFR == q) read_one(f0, (st + 1) % ST, 0, f);
#pragma unroll
      for (int e = 0; e < PER; ++e)
        if (e * NQ / PER == q) issue_one(i0 + ST, st, e);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  for (int i = 0; i < ni; i += ST) {
#pragma unroll
    for (int st = 0; st < ST; ++st)
      if (i + st < ni) step(i + st, st);
  }
  if constexpr (BLK) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) fold(q / FJ, q % FJ);
  }
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if constexpr (KG == 2) {  // group 0 adds group 1's sums, left in group 1's part
    f32x4* const sums = reinterpret_cast<f32x4*>(lds + C::GROUP) + wave * (NQ * 4 * 64) + lane;
#pragma unroll
    for (int q = 0; q < NQ * 4; ++q) {
      f32x16& a = acc[q / 4 / FJ][q / 4 % FJ];
      const int g = q % 4;
      if (grp == 1) sums[q * 64] = f32x4{a[4 * g], a[4 * g + 1], a[4 * g + 2], a[4 * g + 3]};
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NQ * 4; ++q) {
      f32x16& a = acc[q / 4 / FJ][q / 4 % FJ];
      const int g = q % 4;
      if (grp == 0) {
        const f32x4 v = sums[q * 64];
#pragma unroll
        for (int e = 0; e < 4; ++e) a[4 * g + e] += v[e];
      }
    }
  }

  // element 4g + e of fragment (i, j): row 32 (FI wm + i) + r, column 32 (FJ wn + j)
  // + 8 g + 4 h + e; staged in LDS so that the stores write whole row runs
  uint16_t* const ct = reinterpret_cast<uint16_t*>(lds);
#pragma unroll
  for (int i = 0; i < FI; ++i) {
    if (grp != 0) break;
    const int row = 32 * (FI * wm + i) + r;
    const float s = !BLK && m0 + row < M ? sa[m0 + row] : 1.f;
#pragma unroll
    for (int j = 0; j < FJ; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int col = 32 * (FJ * wn + j) + 8 * g + 4 * h;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] = acc[i][j][4 * g + e];
          if (!BLK) v[e] = v[e] * s * (n0 + col < N ? sw[n0 + col + e] : 1.f);
        }
        u32x2 o;
        o[0] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2v{v[0], v[1]}), bf16x2v));
        o[1] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2v{v[2], v[3]}), bf16x2v));
        *reinterpret_cast<u32x2*>(ct + row * C::C_STRIDE + col) = o;
      }
  }
  __syncthreads();
  for (int q = t; q < C::TM * (C::TN / 8); q += 256 * KG) {
    const int row = q / (C::TN / 8), ch = q % (C::TN / 8) * 8;
    if (m0 + row < M && n0 + ch < N)
      *reinterpret_cast<u32x4*>(Y + (int64_t)(m0 + row) * N + n0 + ch) =
          *reinterpret_cast<const u32x4*>(ct + row * C::C_STRIDE + ch);
  }
}

constexpr int SKINNY_KS = 4, SKINNY_D = 2;  // 8 wavefronts or deeper prefetch measured 0 - 5 % slower

template <bool BLK>
tb_status launch_skinny(const char* fn, const Fp8Args& a, hipStream_t stream) {
  const int64_t tiles_m = (a.M + 31) / 32, tiles_n = (a.N + TN - 1) / TN;
  TB_CHECK_ARG(tiles_m * tiles_n < (1ll << 31), "%s: problem too large", fn);
  hipLaunchKernelGGL((fp8_skinny<SKINNY_KS, SKINNY_D, BLK>), dim3((unsigned)(tiles_m * tiles_n)), dim3(64 * SKINNY_KS), 0,
                     stream, a.Aq, a.WqT, a.sa, a.sw, a.Y, a.M, a.N, a.K, (int)tiles_m);
  return tb::launch_status(fn);
}

template <class C, bool BLK>
tb_status launch_tile(const char* fn, const Fp8Args& a, hipStream_t stream) {
  auto kern = &fp8_tile<C::FI, C::FJ, C::ST, BLK, C::KG>;
  constexpr size_t lds = C::LDS_BYTES;
  if (tb_status st = tb::reserve_lds(reinterpret_cast<const void*>(kern), lds, fn)) return st;
  const int64_t tiles_m = (a.M + C::TM - 1) / C::TM, tiles_n = (a.N + C::TN - 1) / C::TN;
  TB_CHECK_ARG(tiles_m * tiles_n < (1ll << 31), "%s: problem too large", fn);
  hipLaunchKernelGGL(kern, dim3((unsigned)(tiles_m * tiles_n)), dim3(256 * C::KG), lds, stream, a.Aq, a.WqT, a.sa, a.sw,
                     a.Y, a.M, a.N, a.K, (int)tiles_m);
  return tb::launch_status(fn);
}

// f(shape) of an LDS tile: launch and describe take the same one.
// Ring stages: as deep as pays while one block runs per CU (64 x 64: four, 15.4
// against 18.9 us with three at 64 x 8192 x 8192; 64 x 128: four, 11.9 against 13.1
// at 300 x 5000 x 4096); two or three where several tiles share a CU, so that two
// blocks fit (128 x 128: 1024 x 8192 x 8192 60 us with two, 70 with three).  With
// block scales, one block per CU and one wavefront per SIMD, the scale FMAs wait for
// the MFMAs; two K groups fill each other's waits (weights from HBM, 200 x 2112 x 7168 17.0 ->
// 13.7 us, 128 x 8192 x 8192 27.3 -> 22.4, 300 x 5000 x 4096 13.4 -> 12.7, 256 x 4096 x 4096
// 10.9 -> 9.5; row scales: no gain).
template <bool BLK, class F>
tb_status with_tile(plan::Fp8Tile tile, int64_t M, int64_t N, const F& f) {
  auto tiles = [&](int64_t tm, int64_t tn) { return (M + tm - 1) / tm * ((N + tn - 1) / tn); };
  switch (tile) {
    case plan::FP8_64x64:
      if (BLK && tiles(64, 64) <= 256) return f(Tile<1, 1, 3, BLK, BLK ? 2 : 1>{});
      return f(Tile<1, 1, BLK ? 3 : 4, BLK>{});
    case plan::FP8_64x128:
      if (tiles(64, 128) <= 256) return f(Tile<1, 2, BLK ? 3 : 4, BLK, BLK ? 2 : 1>{});
      return f(Tile<1, 2, 3, BLK>{});
    default:
      if (tiles(128, 128) <= 256) return f(Tile<2, 2, 3, BLK>{});
      return f(Tile<2, 2, 2, BLK>{});
  }
}

template <bool BLK>
tb_status launch(const char* fn, plan::Fp8Tile tile, const Fp8Args& a, hipStream_t stream) {
  if (tile == plan::FP8_32x32) return launch_skinny<BLK>(fn, a, stream);
  return with_tile<BLK>(tile, a.M, a.N, [&](auto shape) { return launch_tile<decltype(shape), BLK>(fn, a, stream); });
}

tb_status launch_small(const char* fn, plan::Fp8Tile tile, bool block_scaled, const Fp8Args& a, hipStream_t stream) {
  return block_scaled ? launch<true>(fn, tile, a, stream) : launch<false>(fn, tile, a, stream);
}

void describe_small(plan::Fp8Tile tile, bool block_scaled, int64_t M, int64_t N, tb_tile* out) {
  auto f = [&](auto shape) {
    typedef decltype(shape) C;
    *out = tb_tile{"fp8_tile", C::TM, C::TN, 4 * C::KG, C::KG, 1};
    return TB_OK;
  };
  if (tile == plan::FP8_32x32)
    *out = tb_tile{"fp8_skinny", 32, TN, SKINNY_KS, SKINNY_KS, 1};
  else if (block_scaled)
    with_tile<true>(tile, M, N, f);
  else
    with_tile<false>(tile, M, N, f);
}

}  // namespace fp8s
}  // namespace tb
