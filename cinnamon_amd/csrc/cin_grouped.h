// Expert-range helpers shared by the grouped (MoE) quantizers and GEMMs.
//
// Tokens are sorted by expert; expert e owns rows [starts[e], ends[e]) of a [T, ...]
// operand (reference src/layers.py:141-149: counts -> cumsum -> starts/ends).  The ranges
// are read on the device, so no host synchronisation is needed.  Ranges are clamped to
// [0, T); an empty or inverted range owns no rows.
//
// The backward of the grouped GEMM reduces over each expert's tokens, so its operands are
// quantized in 128-token chunks aligned at the expert's first row (the A7 recipe of the
// reference, src/kernels.py:771-788, applied per expert slice).  Chunk c of expert e holds
// rows [s_e + 128 c, min(s_e + 128 (c + 1), e_e)) and is stored in a padded token axis at
// [p_e + 128 c, p_e + 128 (c + 1)), with p_e = sum over e' < e of 128 * ceil(m_e' / 128).
// The padded length is at most T + 127 E.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cin {

__device__ inline void clamp_range(const int64_t* starts, const int64_t* ends, int64_t e, int64_t T,
                                   int64_t& s0, int64_t& s1) {
  s0 = starts[e];
  s1 = ends[e];
  if (s0 < 0) s0 = 0;
  if (s1 > T) s1 = T;
  if (s1 < s0) s1 = s0;
}

// XCD-aware order: workgroup b runs on XCD b % 8; give each XCD a contiguous run of
// tile ids (n fastest) so its CUs share A row panels and B in their L2.
// Tile index v -> (tm, tn): groups of GM m-tiles swept n by n, m fastest, so the 32 tiles
// an XCD runs at once share GM A row panels and 32 / GM B column panels.  Measured
// alternating in one process: GM = 8 took the config-3 grouped gate/up GEMM 4055 -> 3991
// us and its dgrad 4486 -> 4370 us against GM = 4 (down the same; GM = 16 was 1.5-2%
// slower than 8 on all three); the grouped wgrad and
// the config-4 dgrad keep GM = 4 (8 was 0.6% slower, and the same).  In the one-round
// kernel, GM = 4 took the config-4 wgrad (8 x 28 tiles) 125.5 -> 113.1 us against whole
// m rows per XCD, where every XCD read all of B; config 2 maps the same either way.
template <uint32_t GM>
__device__ inline void raster(uint32_t v, uint32_t tiles_m, uint32_t tiles_n, uint32_t& tm, uint32_t& tn) {
  const uint32_t gsz = GM * tiles_n;
  const uint32_t grp = v / gsz, first = grp * GM;
  const uint32_t gm = tiles_m - first < GM ? tiles_m - first : GM;
  const uint32_t w = v - grp * gsz;
  tm = first + w % gm;
  tn = w / gm;
}

__device__ inline uint32_t xcd_remap(uint32_t b, uint32_t G) {
  const uint32_t Gfull = G & ~7u;
  return b < Gfull ? (b & 7u) * (Gfull >> 3) + (b >> 3) : b;
}

// The tile of this workgroup when every expert's rows are cut into tiles of TM (experts in order)
// against tiles_n column tiles: false for a workgroup past the last one.  The grid holds the
// most tiles that the rows can make; the order over the XCDs is that of the tiles there are, or
// the surplus workgroups, which all come last, leave some XCDs without work (16 Zipf rows, 32
// experts, 7168 x 2048: 42 us over the grid, 12.5 over the tiles; 64 rows 55, 37).  Each wave looks
// at 64 experts at a time.
template <int TM>
__device__ inline bool find_tile(const int64_t* __restrict__ starts, const int64_t* __restrict__ ends, int64_t E,
                                 int64_t Tn, uint32_t tiles_n, int64_t& e, int64_t& row0, int64_t& row_end,
                                 uint32_t& tn) {
  const int lane = threadIdx.x & 63;
  int64_t s0 = 0, s1 = 0;
  int n = 0, incl = 0;  // the lane's expert: its row tiles, and those up to and with it
  auto scan = [&](int64_t base) {
    s0 = s1 = 0;
    if (base + lane < E) clamp_range(starts, ends, base + lane, Tn, s0, s1);
    incl = n = (int)((s1 - s0 + TM - 1) / TM);
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int o = __shfl_up(incl, d, 64);
      if (lane >= d) incl += o;
    }
    return __builtin_amdgcn_readlane(incl, 63);
  };
  int total = scan(0);
  for (int64_t base = 64; base < E; base += 64) total += scan(base);
  if (blockIdx.x >= (uint32_t)total * tiles_n) return false;
  uint32_t tm;
  raster<4>(xcd_remap(blockIdx.x, (uint32_t)total * tiles_n), (uint32_t)total, tiles_n, tm, tn);
  int seen = 0;
  for (int64_t base = 0; base < E; base += 64) {
    const int here = E > 64 ? scan(base) : total;
    if ((int)tm < seen + here) {
      const int l = (int)__builtin_ctzll(__ballot((int)tm < seen + incl));
      e = base + l;
      row0 = __shfl(s0, l, 64) + (int64_t)((int)tm - seen - __builtin_amdgcn_readlane(incl - n, l)) * TM;
      row_end = __shfl(s1, l, 64);
      return true;
    }
    seen += here;
  }
  return false;
}

}  // namespace cin
