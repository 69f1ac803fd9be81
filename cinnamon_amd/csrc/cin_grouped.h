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

// The expert that owns row tile `tile` when every expert's rows are cut into tiles of TM
// (experts in order): false past the last one.  Each wave looks at 64 experts at a time.
template <int TM>
__device__ inline bool find_row_tile(const int64_t* __restrict__ starts, const int64_t* __restrict__ ends, int64_t E,
                                     int64_t Tn, int64_t tile, int64_t& e, int64_t& row0, int64_t& row_end) {
  const int lane = threadIdx.x & 63;
  int64_t seen = 0;
  for (int64_t base = 0; base < E; base += 64) {
    int64_t s0 = 0, s1 = 0;
    if (base + lane < E) clamp_range(starts, ends, base + lane, Tn, s0, s1);
    const int64_t n = (s1 - s0 + TM - 1) / TM;
    int64_t incl = n;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int64_t o = __shfl_up(incl, d, 64);
      if (lane >= d) incl += o;
    }
    const uint64_t past = __ballot(tile < seen + incl);
    if (past) {
      const int l = (int)__builtin_ctzll(past);
      e = base + l;
      row0 = __shfl(s0, l, 64) + (tile - seen - __shfl(incl - n, l, 64)) * TM;
      row_end = __shfl(s1, l, 64);
      return true;
    }
    seen += __shfl(incl, 63, 64);
  }
  return false;
}

}  // namespace cin
