// W4A16 GEMM on small tiles: the dense, grouped and MoE products of
// w4a16_gemm.hip for calls whose 256 x 256 tiles would leave most of the
// device idle (few rows, few columns) or multiply mostly padding (an expert's
// few rows).
//
// What bounds such a call is the stream of int4 weights from HBM and, where a
// block walks all of K alone, the latency of one K step; not the MFMAs.  So a
// block owns a tile of 32 RB rows x 64 CW columns over the whole of K, many
// blocks fill the device (several per CU), and its loads run ST K steps ahead
// through an LDS ring:
//
//   ring : per K step of 64 the A tile, the packed W tile and the step's scales
//          and zero-points stream HBM -> LDS by DMA (buffer_load ... lds), ST
//          stages, one barrier per step; 16-byte W DMAs where every row of W
//          and every tile column starts on 16 bytes (WIDE), 4-byte ones
//          otherwise;
//   regs : after the barrier a wavefront reads the whole next step's fragments
//          into registers (A by ds_read_b128, the W byte columns by the
//          transposing ds_read_b64_tr_b8), so a step's arithmetic never waits
//          on LDS and the stage is free again one barrier later;
//   waves: WM row groups x CW column groups of 64 columns; with PS the even and
//          the odd columns of a column group are two wavefronts (each lane
//          dequantises one nibble of its byte column), which keeps four
//          wavefronts busy on a tile of few rows.
//
// Arithmetic and order are those of the 256-column tiles: the same exact
// dequantisation to fp16, the same v_mfma_f32_32x32x16_f16 operands in the same
// K order per output element, the same epilogue roundings; results are
// bit-identical to them, so neither the choice of tile nor the call that uses
// it shows in an output.  Only the 64-column dense tiles (S32x64k4, S64x64k4), which take
// products of at most 64 rows unless N alone fills the device with wider ones,
// split K, over four groups of wavefronts of one block whose fp32 sums are added
// through LDS in group order: reproducible, but not the unsplit order.
// No workspace is needed.
#include "w4a16_small.h"

#include <type_traits>

#pragma clang fp contract(off)

namespace tb {
namespace w4a16 {
namespace sm {

// One tile shape.  RB: 32-row blocks per tile; CW: 64-column groups; PS: even
// and odd columns on two wavefronts; WM: row groups; ST: ring stages; KS: K
// groups.
template <int RB_, int CW_, bool PS_, int WM_, int ST_, int KS_ = 1>
struct Shape {
  static constexpr int RB = RB_, CW = CW_, WM = WM_, ST = ST_, KS = KS_;
  static constexpr bool PS = PS_;
  static constexpr int WAVES = WM * CW * (PS ? 2 : 1);  // per K group
  static constexpr int THREADS = 64 * WAVES * KS;
  static constexpr int MBW = RB / WM;    // 32-row blocks per wavefront
  static constexpr int NF = PS ? 1 : 2;  // column fragments per wavefront
  static constexpr int TM = 32 * RB, TN = 64 * CW;
  static constexpr int WROW = 32 * CW;  // packed bytes per K row of the tile
  static constexpr int A_ST = TM * BK * 2, W_ST = BK * WROW;
  // scales (256-byte DMAs), zero-points and the idle wavefronts' landing pad
  static constexpr int SW = CW > 2 ? CW / 2 : 1;  // wavefronts that fetch scales
  static constexpr int S_OFF = A_ST + W_ST, Z_OFF = S_OFF + 256 * SW, PAD_OFF = Z_OFF + 256;
  static constexpr int STAGE = PAD_OFF + 256;
  static constexpr int AI = TM / 8 / WAVES;  // A DMA instructions per wavefront and step
  static constexpr int C_BYTES = TM * (TN + 8) * 2;
  static constexpr int RED_BYTES = (KS - 1) * TM * TN * 4;  // the other K groups' fp32 sums
  static constexpr int RING = ST * STAGE;
  static constexpr int LDS_BYTES = KS * RING > C_BYTES + RED_BYTES ? KS * RING : C_BYTES + RED_BYTES;
  static constexpr int MIN_WAVES = THREADS / 256 > 2 ? THREADS / 256 : RB * NF / WM <= 4 ? 2 : 1;  // per SIMD
  static_assert(MBW * WM == RB && AI * 8 * WAVES == TM, "wave grid");
  static_assert(CW == 1 || CW == 2 || CW == 4, "column groups");
  static_assert(LDS_BYTES <= 160 * 1024, "LDS budget");
};

// The shapes in use.  Three stages (four measured the same, two 10 - 30 % slower); four
// at 64 x 128, where three blocks of 51 KiB still share a CU.
typedef Shape<1, 2, true, 1, 3> S32x128;
typedef Shape<1, 4, false, 1, 3> S32x256;
typedef Shape<2, 4, false, 1, 3> S64x256;
typedef Shape<1, 1, true, 1, 3, 4> S32x64k4;
typedef Shape<2, 1, true, 1, 3, 4> S64x64k4;
typedef Shape<2, 2, true, 1, 4> S64x128;
typedef Shape<4, 4, false, 1, 3> S128x256;

// 16-byte chunk c of packed row r sits at slot c ^ wswz(r): the eight rows of a
// transposing read (and its two chunks) then sit in different banks.
template <int CW>
__device__ __forceinline__ int wswz(int r) {
  return CW == 4 ? r & 7 : CW == 2 ? ((r >> 2) & 1) << 1 : 0;
}

template <class C, bool WIDE, int MODE>
__device__ __forceinline__ void tile(uint8_t* __restrict__ lds, const _Float16* __restrict__ A,
                                     const uint8_t* __restrict__ W, const _Float16* __restrict__ S,
                                     const uint8_t* __restrict__ Z, _Float16* __restrict__ Y, int M, int N, int K,
                                     int group, int m0, int n0, int a_rows, const RowMap rm) {
  constexpr int CW = C::CW, ST = C::ST, MBW = C::MBW, NF = C::NF, AI = C::AI, WAVES = C::WAVES;
  constexpr int TM = C::TM, TN = C::TN, WROW = C::WROW, STAGE = C::STAGE;
  // W DMA instructions per step: 1 KiB (WIDE) or 256 bytes each
  constexpr int WTOT = C::W_ST / (WIDE ? 1024 : 256);
  constexpr int WI = WTOT / WAVES > 0 ? WTOT / WAVES : 1;
  // with fewer W instructions than wavefronts the first ones issue them and the
  // next ones fetch the scales and zero-points; otherwise the first ones do both
  // (the rest's scale DMA lands in the pad, so that every wavefront counts the
  // same)
  constexpr bool SHARED = WTOT < WAVES;
  static_assert(SHARED || WTOT % WAVES == 0, "W DMA split");
  constexpr int PER = AI + WI + (SHARED ? 0 : 1);  // DMAs per wavefront and step
  static_assert(PER * (ST - 1) < 64, "vmcnt range");
  const int t = threadIdx.x, lane = t & 63, h = lane >> 5, j = lane & 31;
  const int w = __builtin_amdgcn_readfirstlane((t >> 6) % WAVES);
  const int kg = __builtin_amdgcn_readfirstlane((t >> 6) / WAVES);  // K group
  const int wn = w % CW, wq = w / CW;
  const int par = C::PS ? wq & 1 : 0;  // PS: this wavefront's column parity
  const int wm = C::PS ? wq >> 1 : wq;
  // K group kg takes steps k0 .. k0 + mine - 1; every group runs nk of them (the
  // barrier is the block's), the last ones of a shorter group on zeros
  const int nk_all = K / BK, nk = (nk_all + C::KS - 1) / C::KS;
  const int k0 = min(nk_all, kg * nk), mine = min(nk, nk_all - k0);
  const uint32_t half_n = (uint32_t)(N / 2);
  const int I = N / 2, a0 = n0 / 2;  // T_GATE_UP: activation columns
  if (MODE == T_PLAIN) a_rows = M;

  const i32x4 ra = rsrc4(A, (uint32_t)a_rows * (uint32_t)K * 2u);
  const i32x4 rw = rsrc4(W, (uint32_t)K * half_n);
  const i32x4 rs = rsrc4(S, (uint32_t)(K / group) * (uint32_t)N * 2u);
  const i32x4 rz = rsrc4(Z, (uint32_t)(K / group) * half_n);
  // past the last step the DMAs go through empty resources (zeros, no traffic)
  auto live_rsrc = [](bool live, i32x4 r) __attribute__((always_inline)) {
    r[2] = __builtin_amdgcn_readfirstlane(live ? r[2] : 0);
    return r;
  };

  // A DMA: instruction i of wavefront w fills rows 8 (AI w + i) .. +7 (lane L:
  // row + L / 8, 16-byte slot L % 8 holding chunk slot ^ swizzle)
  uint32_t a_off[AI];
#pragma unroll
  for (int i = 0; i < AI; ++i) {
    const int row = 8 * (AI * w + i) + (lane >> 3);
    const int c = (lane & 7) ^ ((row ^ (row >> 3)) & 7);
    const int m = m0 + row;
    int src = m;
    if (MODE == T_GATE_UP && m < M) {
      const int pid = rm.ids[m];
      src = (unsigned)pid < (unsigned)rm.pairs ? pid / rm.topk : a_rows;
    }
    a_off[i] = m < M && src < a_rows ? ((uint32_t)src * (uint32_t)K + (uint32_t)c * 8u) * 2u : OOB;
  }
  // W DMA: lane bytes of an instruction are consecutive in the stage's rows
  constexpr int LB = WIDE ? 16 : 4, ROWS_PER = 64 * LB / WROW, LPR = WROW / LB;  // lanes per row
  uint32_t w_off[WI];
#pragma unroll
  for (int i = 0; i < WI; ++i) {
    const int r = ROWS_PER * (WI * w + i) + lane / LPR;
    const int byte = (lane % LPR) * LB;  // in the stage row
    const int c = (byte >> 4) ^ wswz<CW>(r);
    uint32_t col;
    bool ok;
    if (MODE == T_GATE_UP) {
      // chunk c: gate (c even) or up (c odd) of activation columns a0 + 32 (c / 2) ..
      const int acol = a0 + 32 * (c >> 1) + 2 * (byte & 15);
      col = (uint32_t)((c & 1) * (I / 2) + acol / 2);
      ok = acol < I;
    } else {
      col = (uint32_t)(n0 / 2 + c * 16 + (byte & 15));
      ok = col < half_n;
    }
    w_off[i] = ok && (!SHARED || w < WTOT) ? (uint32_t)r * half_n + col : OOB;
  }
  // scales (4-byte DMAs of 128 columns, lane L columns 2L, 2L + 1) and
  // zero-points (lane L bytes 4L .. 4L + 3) of a step's group
  constexpr int S_WAVE = SHARED ? WTOT : 0, Z_WAVE = S_WAVE + C::SW;
  static_assert(Z_WAVE < WAVES, "a wavefront for the zero-points");
  const bool zw = w == Z_WAVE;
  uint32_t sz_off = OOB, sz_lds = C::PAD_OFF;
  if (w >= S_WAVE && w < Z_WAVE) {
    const int t2 = 128 * (w - S_WAVE) + 2 * lane;
    if (MODE == T_GATE_UP) {
      const int acol = a0 + 32 * (t2 >> 6) + (t2 & 31);
      sz_off = t2 < TN && acol < I ? (uint32_t)(((t2 & 32) ? I : 0) + acol) * 2u : OOB;
    } else {
      const uint32_t col = (uint32_t)(n0 + t2);
      sz_off = t2 < TN && col < (uint32_t)N ? col * 2u : OOB;
    }
    sz_lds = C::S_OFF + 256 * (w - S_WAVE);
  } else if (zw) {
    if (MODE == T_GATE_UP) {
      const int b = 4 * lane, acol = a0 + 32 * (b >> 5) + 2 * (b & 15);
      sz_off = b < WROW && acol < I ? (uint32_t)(((b & 16) ? I / 2 : 0) + acol / 2) : OOB;
    } else {
      const uint32_t col = (uint32_t)(n0 / 2 + 4 * lane);
      sz_off = 4 * lane < WROW && col < half_n ? col : OOB;
    }
    sz_lds = C::Z_OFF;
  }
  typedef __attribute__((address_space(3))) uint8_t lds_u8;
  lds_u8* const lring = (lds_u8*)(__attribute__((address_space(3))) void*)lds + kg * C::RING;
  const uint32_t lds0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(uintptr_t)lring);

  // The next step's DMAs into stage st; everything that advances per step is
  // scalar.
  int i_left = mine, i_rem = group / BK - k0 % (group / BK);
  uint32_t i_a = (uint32_t)(k0 * BK) * 2u, i_w = (uint32_t)(k0 * BK) * half_n;
  const uint32_t s_step = zw ? half_n : (uint32_t)N * 2u;
  uint32_t i_s = (uint32_t)(k0 * BK / group) * s_step;
  // DMA d (0 .. PER - 1) of the step the trackers stand at, into stage st
  auto issue_one = [&](int st, int d) __attribute__((always_inline)) {
    const bool live = i_left > 0;
    const uint32_t dst0 = lds0 + (uint32_t)(st * STAGE);
    if (d < AI) {
      dma16(dst0 + (uint32_t)(8 * (AI * w + d) * 128), a_off[d], live_rsrc(live, ra), i_a);
    } else if (d < AI + WI && (!SHARED || w < WTOT)) {
      const uint32_t dst = dst0 + (uint32_t)(C::A_ST + (WI * w + d - AI) * 64 * LB);
      if (WIDE)
        dma16(dst, w_off[d - AI], live_rsrc(live, rw), i_w);
      else
        dma4(dst, w_off[d - AI], live_rsrc(live, rw), i_w);
    } else {
      dma4(dst0 + sz_lds, sz_off, live_rsrc(live, zw ? rz : rs), i_s);
    }
  };
  auto issue_next = [&]() __attribute__((always_inline)) {
    --i_left;
    i_a += BK * 2;
    i_w += BK * half_n;
    if (--i_rem == 0) {
      i_rem = group / BK;
      i_s += s_step;
    }
  };

  // Fragment offsets in a stage.  A fragment mb of slice c: row 32 (MBW wm + mb)
  // + j, chunk 2c + h; the swizzle depends on the row's 32-row block through its
  // parity only.
  uint32_t fa_off[2];
#pragma unroll
  for (int pb = 0; pb < 2; ++pb) {
    const int sw = (j ^ (4 * pb + (j >> 3))) & 7;
    fa_off[pb] = (uint32_t)(wm * MBW * 4096 + j * 128 + ((h ^ sw) << 4));
  }
  // Transposing byte read of slice c: as in the 256-column tiles (byte r of the
  // result holds row pi(r), pi swapping 1 <-> 2 and 5 <-> 6, so a k-row pair
  // sits in bytes 0 and 2, or, shifted down by 8, in bytes 1 and 3).
  uint32_t wt_off;
  {
    const int p = lane & 15, r = p >> 1, b = p & 1, G = lane >> 4;
    const int pr = (r & 4) | ((r & 1) << 1) | ((r >> 1) & 1);
    const int cb = 2 * wn + (G & 1);
    wt_off = (uint32_t)(C::A_ST + (8 * (G >> 1) + pr) * WROW + ((cb ^ wswz<CW>(pr)) << 4) + 8 * b);
  }
  // bases of the fragment reads (the stage is an immediate offset)
  lds_u8* const p_s = lring + C::S_OFF + (wn * 64 + 2 * j) * 2;
  lds_u8* const p_z = lring + C::Z_OFF + wn * 32 + j;
  lds_u8* const p_w = lring + wt_off;
  lds_u8* p_a[4][MBW > 1 ? 2 : 1];
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int q = 0; q < (MBW > 1 ? 2 : 1); ++q) p_a[c][q] = lring + (fa_off[(MBW * wm + q) & 1] ^ (uint32_t)(c << 5));

  struct Frag {
    h8 a[4][MBW];
    v2i x[4];
    uint32_t s2, zb;
  };
  // LDS read r (0 .. NR - 1) of stage st: the byte columns, scales and
  // zero-points first, then the A fragments in slice order
  constexpr int NR = 6 + 4 * MBW;
  auto read_one = [&](Frag& f, int st, int r) __attribute__((always_inline)) {
    if (r < 4) {
      f.x[r] = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
          (__attribute__((address_space(3))) v2i*)(p_w + st * STAGE + r * 16 * WROW));
    } else if (r == 4) {
      f.s2 = *(__attribute__((address_space(3))) const uint32_t*)(p_s + st * STAGE);
    } else if (r == 5) {
      f.zb = *(p_z + st * STAGE);
    } else {
      const int c = (r - 6) / MBW, mb = (r - 6) % MBW;
      f.a[c][mb] = *(__attribute__((address_space(3))) const h8*)(p_a[c][mb & 1] + st * STAGE + mb * 4096);
    }
  };

  f32x16 acc[MBW][NF];
#pragma unroll
  for (int i = 0; i < MBW; ++i)
#pragma unroll
    for (int nb = 0; nb < NF; ++nb) acc[i][nb] = f32x16{};

  // Column fragment nb's nibble mask, fp16 magic and scale selector: even
  // columns (bits 3:0) under 0x64 read 1024 + q, odd ones (bits 7:4) under 0x54
  // read 64 + q.
  uint32_t mask[NF], magic[NF], ssel[NF];
#pragma unroll
  for (int nb = 0; nb < NF; ++nb) {
    const bool odd = C::PS ? par != 0 : nb != 0;
    mask[nb] = (uint32_t)__builtin_amdgcn_readfirstlane(odd ? 0x00F000F0 : 0x000F000F);
    magic[nb] = (uint32_t)__builtin_amdgcn_readfirstlane(odd ? 0x54005400 : 0x64006400) + (uint32_t)(lane >> 6);
    ssel[nb] = (uint32_t)__builtin_amdgcn_readfirstlane(odd ? 0x03020302 : 0x01000100);
  }
  uint32_t sc[NF], zp[NF];
  auto load_scales = [&](const Frag& f) __attribute__((always_inline)) {
#pragma unroll
    for (int nb = 0; nb < NF; ++nb) {
      sc[nb] = perm(f.s2, f.s2, ssel[nb]);
      zp[nb] = and_or(f.zb | (f.zb << 16), mask[nb], magic[nb]);
    }
  };
  // k-row pair q of a byte column, all of the wavefront's column fragments
  u32x4 wf[2][NF];
  auto dequant_pair = [&](const v2i x, int buf, int q) __attribute__((always_inline)) {
    const uint32_t src = (uint32_t)x[q >> 1];
    const uint32_t d = (q & 1) ? src >> 8 : src;  // k rows 2q, 2q + 1 in bytes 0 and 2
    uint32_t v[NF];
#pragma unroll
    for (int nb = 0; nb < NF; ++nb) v[nb] = and_or(d, mask[nb], magic[nb]);
#pragma unroll
    for (int nb = 0; nb < NF; ++nb) v[nb] = as_u32(as_h2(v[nb]) - as_h2(zp[nb]));
#pragma unroll
    for (int nb = 0; nb < NF; ++nb) wf[buf][nb][q] = as_u32(as_h2(v[nb]) * as_h2(sc[nb]));
  };

  // s_waitcnt immediates: vmcnt (bits 3:0 and 15:14), lgkmcnt(0), expcnt unused
  constexpr int VM0 = PER * (ST - 1), VM1 = PER * (ST - 2);
  constexpr int WAIT_PRO = (VM0 & 15) | ((VM0 >> 4) << 14) | (7 << 4) | (15 << 8);
  constexpr int WAIT_STEP = (VM1 & 15) | ((VM1 >> 4) << 14) | (7 << 4) | (0 << 8);
  auto barrier = [&]() __attribute__((always_inline)) {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

#pragma unroll
  for (int i = 0; i < ST; ++i) {
#pragma unroll
    for (int d = 0; d < PER; ++d) issue_one(i, d);
    issue_next();
  }
  __builtin_amdgcn_s_waitcnt(WAIT_PRO);  // step 0 landed (each wavefront waits for its own DMAs)
  barrier();
  Frag f0, f1;
#pragma unroll
  for (int r = 0; r < NR; ++r) read_one(f0, 0, r);
  load_scales(f0);
#pragma unroll
  for (int q = 0; q < 4; ++q) dequant_pair(f0.x[0], 0, q);
  // A step of stage st on `cur`: once the next step has landed and every
  // wavefront has this step's fragments in registers (the barrier), the stage
  // takes the DMAs of the step ST later (slices 1 .. 3) and the next step's
  // fragments are read (slices 0 .. 2); each slice dequantises the next one
  // (the last one the next step's first) between its MFMAs, so the matrix pipe
  // and the VALU work side by side in one wavefront.  Past the last step the
  // DMAs read nothing and the fragments are not used.
  constexpr int NQ = MBW * NF;  // MFMAs per slice
  auto step = [&](int st, const Frag& cur, Frag& nxt) __attribute__((always_inline)) {
    __builtin_amdgcn_s_waitcnt(WAIT_STEP);
    barrier();
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int b = c & 1;
      if (c == 3) load_scales(nxt);
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const int mb = q / NF, nb = q % NF, slot = c * NQ + q;
        acc[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8, wf[b][nb]), cur.a[c][mb],
                                                             acc[mb][nb], 0, 0, 0);
#pragma unroll
        for (int r = 0; r < NR; ++r)
          if (r * 3 * NQ / NR == slot) read_one(nxt, (st + 1) % ST, r);
#pragma unroll
        for (int d = 0; d < PER; ++d)
          if (NQ + d * 3 * NQ / PER == slot) issue_one(st, d);
#pragma unroll
        for (int p = 0; p < 4; ++p)
          if (p * NQ / 4 == q) dequant_pair(c < 3 ? cur.x[c + 1] : nxt.x[0], b ^ 1, p);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    issue_next();
  };
  constexpr int UN = ST % 2 ? 2 * ST : ST;  // steps per iteration: stages and fragment registers are constants
  for (int kt = 0; kt < nk; kt += UN) {
#pragma unroll
    for (int u = 0; u < UN; u += 2) {
      if (kt + u < nk) step(u % ST, f0, f1);
      if (kt + u + 1 < nk) step((u + 1) % ST, f1, f0);
    }
  }
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();  // the ring is free

  if constexpr (C::KS > 1) {
    // the K groups' sums, added in group order by group 0
    typedef __attribute__((address_space(3))) f32x4 lds_f4;
    lds_f4* const red = (lds_f4*)((__attribute__((address_space(3))) uint8_t*)(__attribute__((address_space(3))) void*)lds +
                                  C::C_BYTES);
    constexpr int PW = MBW * NF * 4 * 64;  // 16-byte words per wavefront
    if (kg > 0) {
#pragma unroll
      for (int mb = 0; mb < MBW; ++mb)
#pragma unroll
        for (int nb = 0; nb < NF; ++nb)
#pragma unroll
          for (int g = 0; g < 4; ++g)
            red[((kg - 1) * WAVES + w) * PW + ((mb * NF + nb) * 4 + g) * 64 + lane] =
                f32x4{acc[mb][nb][4 * g], acc[mb][nb][4 * g + 1], acc[mb][nb][4 * g + 2], acc[mb][nb][4 * g + 3]};
    }
    __syncthreads();
    if (kg == 0) {
#pragma unroll
      for (int q = 0; q < C::KS - 1; ++q)
#pragma unroll
        for (int mb = 0; mb < MBW; ++mb)
#pragma unroll
          for (int nb = 0; nb < NF; ++nb)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
              const f32x4 v = red[(q * WAVES + w) * PW + ((mb * NF + nb) * 4 + g) * 64 + lane];
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[mb][nb][4 * g + e] += v[e];
            }
    }
  }

  // Epilogue: element 4g + e of accumulator (mb, nb) is row 32 (MBW wm + mb) + j,
  // column 64 wn + 16 g + 8 h + 2 e + (nb or the wavefront's parity) of the
  // tile.  The fp16 tile is staged in LDS (the ring is free) so that the stores
  // write whole row runs.
  constexpr int TC = MODE == T_GATE_UP ? TN / 2 : TN;  // output columns of the tile
  constexpr int CS = TC + 8;                           // staged row stride (halves)
  typedef __attribute__((address_space(3))) _Float16 lds_h;
  lds_h* const cb = (lds_h*)(__attribute__((address_space(3))) void*)lds;
  if (kg == 0)
#pragma unroll
  for (int mb = 0; mb < MBW; ++mb) {
    const int r = 32 * (MBW * wm + mb) + j;
    float rwt = 1.f;
    if (MODE == T_DOWN) {
      const int pid = m0 + r < M ? rm.ids[m0 + r] : -1;
      rwt = (unsigned)pid < (unsigned)rm.pairs ? rm.w[pid] : 0.f;
    }
#pragma unroll
    for (int g = 0; g < (MODE == T_GATE_UP ? 2 : 4); ++g) {
      _Float16 v[NF][4];
#pragma unroll
      for (int nb = 0; nb < NF; ++nb)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (MODE == T_GATE_UP) {
            // g: gate, g + 2: up of activation column a0 + 32 wn + 16 g + 8 h + 2 e + ..
            const float gv = (float)(_Float16)acc[mb][nb][4 * g + e];
            const float uv = (float)(_Float16)acc[mb][nb][4 * (g + 2) + e];
            float sg = 1.0f + expf(-gv);
            asm volatile("" : "+v"(sg));
            v[nb][e] = h_of_rounded(gv / sg * uv);
          } else if (MODE == T_DOWN) {
            v[nb][e] = h_of_rounded(acc[mb][nb][4 * g + e] * rwt);
          } else {
            v[nb][e] = (_Float16)acc[mb][nb][4 * g + e];
          }
        }
      const int col = (MODE == T_GATE_UP ? 32 : 64) * wn + 16 * g + 8 * h;
      if constexpr (C::PS) {
#pragma unroll
        for (int e = 0; e < 4; ++e) cb[r * CS + col + 2 * e + par] = v[0][e];
      } else {
        u32x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = as_u32(f16x2{v[0][e], v[NF - 1][e]});
        *(__attribute__((address_space(3))) u32x4*)(cb + r * CS + col) = o;
      }
    }
  }
  __syncthreads();
  constexpr int CPR = TC / 8;  // 16-byte chunks per row
  const int ldy = MODE == T_GATE_UP ? I : N, c0 = MODE == T_GATE_UP ? a0 : n0;
#pragma unroll 2
  for (int idx = t; idx < TM * CPR; idx += C::THREADS) {
    const int r = idx / CPR, ch = idx % CPR;
    const int m = m0 + r;
    if (m >= M || c0 + ch * 8 >= ldy) continue;
    int64_t dst = m;
    if (MODE == T_DOWN) {
      dst = rm.ids[m];
      if ((unsigned)dst >= (unsigned)rm.pairs) continue;
    }
    *reinterpret_cast<u32x4*>(Y + dst * ldy + c0 + ch * 8) =
        *(__attribute__((address_space(3))) const u32x4*)(cb + r * CS + ch * 8);
  }
}

// Blocks go round-robin over the 8 XCDs: XCD x takes a contiguous run of tiles,
// so that the blocks of one L2 share W lines and A rows.
__device__ __forceinline__ int xcd_run(int bid, int nb) {
  const int x = bid & 7, q = nb >> 3, rem = nb & 7;
  return x * q + min(x, rem) + (bid >> 3);
}

// Dense: tiles in column order, all row tiles of a column together.
template <class C, bool WIDE>
__global__ void __launch_bounds__(C::THREADS, C::MIN_WAVES)
    w4a16_dense(const _Float16* __restrict__ A, const uint8_t* __restrict__ W, const _Float16* __restrict__ S,
                const uint8_t* __restrict__ Z, _Float16* __restrict__ Y, int M, int N, int K, int group, int tiles_m) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int idx = xcd_run(blockIdx.x, gridDim.x);
  const int nt = idx / tiles_m, mt = idx - nt * tiles_m;
  tile<C, WIDE, T_PLAIN>(lds, A, W, S, Z, Y, M, N, K, group, mt * C::TM, nt * C::TN, M, RowMap{});
}

// Grouped, gate/up and down products: the kernels of w4a16_gemm.hip on small
// tiles (rows: pairs; A is X for the gate/up projection).
template <class C, bool WIDE, int MODE>
__global__ void __launch_bounds__(C::THREADS, C::MIN_WAVES)
    w4a16_experts(const _Float16* __restrict__ A, const int* __restrict__ ids, const int* __restrict__ offsets,
                  const float* __restrict__ wts, const uint8_t* __restrict__ W, const _Float16* __restrict__ S,
                  const uint8_t* __restrict__ Z, _Float16* __restrict__ Y, int tokens, int topk, int rows, int experts,
                  int N, int K, int group, int tiles_n) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  int e = 0, m0 = 0, m_end = 0, nt = 0;
  if (!grouped_tile<C::TM>(offsets, experts, rows, tiles_n, e, m0, m_end, nt)) return;  // beyond the last tile: uniform
  const int64_t wstride = (int64_t)K * (N / 2), sstride = (int64_t)(K / group) * N,
                zstride = (int64_t)(K / group) * (N / 2);
  RowMap rm;
  if (MODE != T_PLAIN) rm.ids = ids + m0;
  rm.w = wts;
  rm.topk = topk;
  rm.pairs = rows;
  const int ldy = MODE == T_GATE_UP ? N / 2 : N;
  tile<C, WIDE, MODE>(lds, MODE == T_GATE_UP ? A : A + (int64_t)m0 * K, W + e * wstride, S + e * sstride,
                      Z + e * zstride, MODE == T_DOWN ? Y : Y + (int64_t)m0 * ldy, m_end - m0, N, K, group, 0,
                      nt * C::TN, MODE == T_GATE_UP ? tokens : m_end - m0, rm);
}
template <class C, bool WIDE>
tb_status launch_dense_shape(const char* fn, const DenseArgs& a, hipStream_t stream) {
  auto kern = &w4a16_dense<C, WIDE>;
  if (tb_status st = tb::reserve_lds(reinterpret_cast<const void*>(kern), C::LDS_BYTES, fn)) return st;
  const int64_t tiles_m = (a.M + C::TM - 1) / C::TM, tiles_n = (a.N + C::TN - 1) / C::TN;
  TB_CHECK_ARG(tiles_m * tiles_n < (1ll << 31), "%s: problem too large", fn);
  hipLaunchKernelGGL(kern, dim3((unsigned)(tiles_m * tiles_n)), dim3(C::THREADS), C::LDS_BYTES, stream, a.A, a.W, a.S,
                     a.Z, a.Y, a.M, a.N, a.K, a.group, (int)tiles_m);
  return tb::launch_status(fn);
}

template <class C, bool WIDE, int MODE>
tb_status launch_shape(const char* fn, const ExpertArgs& a, hipStream_t stream) {
  auto kern = &w4a16_experts<C, WIDE, MODE>;
  if (tb_status st = tb::reserve_lds(reinterpret_cast<const void*>(kern), C::LDS_BYTES, fn)) return st;
  const int64_t tiles_n = (a.N + C::TN - 1) / C::TN;
  const int64_t tile_rows = (a.rows + C::TM - 1) / C::TM + a.experts;  // upper bound on sum_e ceil(rows_e / TM)
  const int64_t blocks = tile_rows * tiles_n;
  TB_CHECK_ARG(blocks < (1ll << 31), "%s: problem too large", fn);
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(C::THREADS), C::LDS_BYTES, stream, a.A, a.ids, a.offsets,
                     a.weights, a.W, a.S, a.Z, a.Y, a.tokens, a.topk, (int)a.rows, a.experts, a.N, a.K, a.group,
                     (int)tiles_n);
  return tb::launch_status(fn);
}

// f(shape) of a pick: launch and describe take the same one.
template <class F>
tb_status with_expert_shape(plan::ExpertTile tile, const F& f) {
  switch (tile) {
    case plan::TILE_32x128:
      return f(S32x128{});
    case plan::TILE_32x256:
      return f(S32x256{});
    default:
      return f(S64x256{});
  }
}

template <class F>
tb_status with_dense_shape(plan::DenseTile tile, int64_t M, const F& f) {
  switch (tile) {
    case plan::DENSE_64x64_K4:
      // Up to 32 rows half of a 64-row tile's MFMAs, A DMAs and A reads are padding
      // that the CU's LDS and load paths carry (deeper rings or other K group
      // counts gained nothing).  The same K groups in the same order: the bits are those of
      // the 64-row tile.  Kernel, us, 64 -> 32 rows: 32 x 11008 (K 4096) 13.9 -> 12.5, 24 x
      // 4096 (K 11008) 33.2 -> 29.0, 20 x 12288 (K 1024) 7.3 -> 6.3.
      return M <= 32 ? f(S32x64k4{}) : f(S64x64k4{});
    case plan::DENSE_64x128:
      return f(S64x128{});
    case plan::DENSE_64x256:
      return f(S64x256{});
    default:
      return f(S128x256{});
  }
}

template <class C>
tb_status describe(const char* kernel, tb_tile* out) {
  *out = tb_tile{kernel, C::TM, C::TN, C::THREADS / 64, C::KS, 1};
  return TB_OK;
}

template <int MODE>
tb_status launch_mode(const char* fn, plan::ExpertTile tile, const ExpertArgs& a, hipStream_t stream) {
  // 16-byte W DMAs need every K row of every expert, and in gate/up the up half
  // of a row, to start on 16 bytes
  const bool wide = tb::aligned(a.W, 16) && a.N % (MODE == T_GATE_UP ? 64 : 32) == 0;
  return with_expert_shape(tile, [&](auto shape) {
    typedef decltype(shape) C;
    return wide ? launch_shape<C, true, MODE>(fn, a, stream) : launch_shape<C, false, MODE>(fn, a, stream);
  });
}
}  // namespace sm

void describe_dense_small(plan::DenseTile tile, int64_t M, tb_tile* out) {
  sm::with_dense_shape(tile, M, [&](auto shape) { return sm::describe<decltype(shape)>("w4a16_dense", out); });
}

void describe_experts_small(plan::ExpertTile tile, tb_tile* out) {
  sm::with_expert_shape(tile, [&](auto shape) { return sm::describe<decltype(shape)>("w4a16_experts", out); });
}

tb_status launch_dense_small(const char* fn, plan::DenseTile tile, const DenseArgs& a, hipStream_t stream) {
  const bool wide = tb::aligned(a.W, 16) && a.N % 32 == 0;
  return sm::with_dense_shape(tile, a.M, [&](auto shape) {
    typedef decltype(shape) C;
    return wide ? sm::launch_dense_shape<C, true>(fn, a, stream) : sm::launch_dense_shape<C, false>(fn, a, stream);
  });
}

tb_status launch_experts_small(const char* fn, TileMode mode, plan::ExpertTile tile, const ExpertArgs& a,
                               hipStream_t stream) {
  switch (mode) {
    case T_GATE_UP:
      return sm::launch_mode<T_GATE_UP>(fn, tile, a, stream);
    case T_DOWN:
      return sm::launch_mode<T_DOWN>(fn, tile, a, stream);
    default:
      return sm::launch_mode<T_PLAIN>(fn, tile, a, stream);
  }
}
}  // namespace w4a16
}  // namespace tb
