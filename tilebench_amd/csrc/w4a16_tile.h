// Device helpers shared by the W4A16 tile kernels (w4a16_gemm.hip: 256-column
// tiles of the dense, grouped and MoE kernels; w4a16_small.hip: the small tiles
// that serve calls with too few rows or columns to fill the device).
#pragma once
#include "tb_common.h"

namespace tb {
namespace w4a16 {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

typedef __amdgpu_buffer_rsrc_t rsrc_t;
typedef int i32x4 __attribute__((ext_vector_type(4)));
constexpr uint32_t RSRC_DW3 = 0x00020000u;
constexpr uint32_t OOB = 0x80000000u;
__device__ __forceinline__ rsrc_t make_rsrc(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, (int)RSRC_DW3);
}

// Row map of the MoE pipeline's tiles: tile row m is (token, slot) pair
// ids[m]; the pair's token is ids[m] / topk and its routing weight w[ids[m]].
struct RowMap {
  const int* ids = nullptr;
  const float* w = nullptr;
  int topk = 1;
  int pairs = 0;
};

// fp16 of an fp32 value that is already rounded: the empty asm keeps the
// conversion from being folded into the preceding multiply (a mixed-precision
// FMA would round the exact product once, not the fp32 product).
__device__ __forceinline__ _Float16 h_of_rounded(float f) {
  asm volatile("" : "+v"(f));
  return (_Float16)f;
}

// Tile of this block in a grouped launch: expert e, rows m0 .. m_end - 1 of the
// row space (R rows; expert e owns rows offsets[e] .. offsets[e+1], cut into
// TM-row tiles) and tile column nt of tiles_n.  Offsets are clamped to [0, R]
// so that malformed ones never address rows outside A / Y.  Returns false for
// the blocks past the last tile (the grid is the host's upper bound).
//
// Every wavefront takes 256 experts at a time, four per lane with all their
// loads in flight together (then prefix sums of tile counts and a ballot), so
// the search costs one load round trip per 256 experts.  The tiles that exist
// are counted first and shared out over the 8 XCDs as one contiguous run each
// (block ids go round-robin over them): splitting the upper bound instead put
// every tile of a small call on the first XCDs (one token, 8 of 64 experts:
// gate/up 84 us with all 88 tiles on one XCD) and left the last ones part-idle
// on large calls (64 experts, 4096 tokens x 8: the MoE layer 856 -> 729 us).
template <int TM>
__device__ __forceinline__ bool grouped_tile(const int* __restrict__ offsets, int experts, int R, int tiles_n, int& e,
                                             int& m0, int& m_end, int& nt) {
  constexpr int CH = 4, SPAN = 64 * CH;  // 64-expert chunks in registers
  const int lane = threadIdx.x & 63;
  int lo[CH], hi[CH], cnt[CH];
  auto load = [&](int x0) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int x = x0 + 64 * c + lane;
      lo[c] = hi[c] = 0;
      if (x0 + 64 * c < experts && x < experts) {
        lo[c] = offsets[x];
        hi[c] = offsets[x + 1];
      }
    }
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      lo[c] = min(max(lo[c], 0), R);
      hi[c] = min(max(hi[c], lo[c]), R);
      cnt[c] = (hi[c] - lo[c] + TM - 1) / TM;
    }
  };
  int total = 0;
  for (int x0 = (experts - 1) / SPAN * SPAN; x0 >= 0; x0 -= SPAN) {  // downwards: ends with the first ones in registers
    load(x0);
#pragma unroll
    for (int c = 0; c < CH; ++c) total += cnt[c];
  }
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) total += __shfl_xor(total, d);
  const int tiles = __builtin_amdgcn_readfirstlane(total) * tiles_n;
  const int xcd = (int)blockIdx.x & 7, idx = (int)blockIdx.x >> 3, q = tiles >> 3, rem = tiles & 7;
  if (idx >= q + (xcd < rem ? 1 : 0)) return false;
  const int bid = xcd * q + min(xcd, rem) + idx;
  const int mt = bid / tiles_n;
  nt = bid - mt * tiles_n;
  int seen = 0;
  for (int x0 = 0; x0 < experts; x0 += SPAN) {
    if (x0 > 0) load(x0);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      if (x0 + 64 * c >= experts) break;  // uniform
      int incl = cnt[c];
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(incl, d);
        if (lane >= d) incl += o;
      }
      const int here = __builtin_amdgcn_readfirstlane(__shfl(incl, 63));
      if (mt < seen + here) {
        const unsigned long long hit = __ballot(seen + incl > mt);
        const int l = __builtin_ctzll(hit);
        const int lo_l = __shfl(lo[c], l), hi_l = __shfl(hi[c], l), before = seen + __shfl(incl - cnt[c], l);
        // uniform across the block: scalar registers, so that every address
        // derived from the tile stays scalar
        e = __builtin_amdgcn_readfirstlane(x0 + 64 * c + l);
        m0 = __builtin_amdgcn_readfirstlane(lo_l + (mt - before) * TM);
        m_end = __builtin_amdgcn_readfirstlane(hi_l);
        return true;
      }
      seen += here;
    }
  }
  return false;
}

typedef int v2i __attribute__((ext_vector_type(2)));

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
__device__ __forceinline__ i32x4 rsrc4(const void* p, uint32_t bytes) {
  const uint64_t base = (uint64_t)(uintptr_t)p;
  i32x4 r;
  r[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)base);
  r[1] = __builtin_amdgcn_readfirstlane((int)(uint32_t)(base >> 32) & 0xFFFF);
  r[2] = __builtin_amdgcn_readfirstlane((int)bytes);
  r[3] = (int)RSRC_DW3;
  return r;
}
// (x & mask) | c in one instruction: mask from a scalar register, c from a vector one
__device__ __forceinline__ uint32_t and_or(uint32_t x, uint32_t mask, uint32_t c) {
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "s"(mask), "v"(c));
  return r;
}

// What a tile reads and writes besides the plain product.
enum TileMode {
  T_PLAIN = 0,    // rows m < M of A and Y
  T_GATE_UP = 1,  // MoE gate/up: gathered token rows, SiLU(gate) * up (see tile8 in w4a16_gemm.hip)
  T_DOWN = 2      // MoE down: rows scaled by their routing weight and scattered (see tile8)
};

constexpr int BK = 64;  // K rows per step

}  // namespace w4a16
}  // namespace tb
