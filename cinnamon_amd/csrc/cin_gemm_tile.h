// Block-scaled FP8 GEMM tile of any size, for the products the 256 x 256 kernels of gemm.hip
// do not take or do not fill the chip with.
//
// A workgroup owns a (16 MT WM) x (16 NT WN) tile.  KS groups of WM x WN waves share its K
// blocks, group g taking blocks g, g + KS, ...: a short, wide or narrow product then has
// enough waves in flight although it has few tiles, and its chain of K blocks is KS times
// shorter.  Operands go global -> LDS by DMA, two stages of KS blocks each, one barrier per
// stage; the groups' fp32 tiles meet in LDS at the end, are added in group order (the result
// does not depend on timing) and leave as whole row segments.
//
// Rows past the operands and bytes past K come from out-of-range DMA lanes, which read as
// zero, so any M, any N and any K % 16 == 0 take the same loop.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "cin_common.h"

namespace cin {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

// 16-byte chunk c of tile row r lives at slot c ^ f(r), f(r) = (r % 8) ^ ((r / 8) % 2):
// the 8 rows a 32-bank LDS serves together, and the 8 same-parity rows a 64-bank LDS
// serves together, all hit distinct banks.
__device__ inline int swz_f(int r) { return (r & 7) ^ ((r >> 3) & 1); }

// DMA of 16 (4) bytes per lane from the buffer to LDS: lane t's bytes land at LDS byte
// address lds + 16 t (4 t).  lds is wave-uniform.
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :: "s"(lds), "v"(voff), "s"(r), "s"(soff) : "memory");
}
__device__ __forceinline__ void dma4(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dword %1, %2, %3 offen lds"
               :: "s"(lds), "v"(voff), "s"(r), "s"(soff) : "memory");
}
// s_waitcnt vmcnt(0) (expcnt and lgkmcnt left at their maxima)
__device__ __forceinline__ void wait_dma() { __builtin_amdgcn_s_waitcnt(0x0F70); }
// s_waitcnt lgkmcnt(0) (vmcnt and expcnt left at their maxima), then a workgroup barrier
// that the compiler may not move LDS accesses across.  No vmcnt wait: operand DMA stays in
// flight across it.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_s_waitcnt(0xC07F);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

namespace gt {

// Rows [0, rows_a) of A against rows [0, rows_b) of B; the tile's columns lie in one
// 128-column block of B scales.
struct Tile {
  const uint8_t* A;
  const float* sa;
  const uint8_t* B;
  const float* sb;
  void* C;  // element (0, 0) of the tile
  int rows_a, rows_b;
};

template <int WM_, int WN_, int MT_, int NT_, int KS_>
struct Cfg {
  static constexpr int WM = WM_, WN = WN_, MT = MT_, NT = NT_, KS = KS_;
  static constexpr int kGroup = 64 * WM * WN;  // threads that share a K block
  static constexpr int kThreads = kGroup * KS;
  static constexpr int TM = 16 * MT * WM, TN = 16 * NT * WN;
  static constexpr int kA = TM * 128, kB = TN * 128;
  static constexpr int kSa = 4 * kGroup;        // one 4-byte DMA per thread; the first TM hold the A scales
  static constexpr int kBlock = kA + kB + kSa;  // one K block's operands
  static constexpr int kStage = kBlock * KS;
  static constexpr int kOpsA = TM * 8 / kGroup, kOpsB = TN * 8 / kGroup;
  // row stride (floats) of the fp32 tile in LDS: the 16 rows of one store pass lie 4 banks apart
  static constexpr int kCStride = TN + 4;
  static constexpr int kCBytes = KS * TM * kCStride * 4;
  static constexpr int kBytes = 2 * kStage > kCBytes ? 2 * kStage : kCBytes;
  static_assert(128 % TN == 0, "one block of B scales");
  static_assert(kGroup >= TM, "one scale per thread");
  static_assert(TM * 8 % kGroup == 0 && TN * 8 % kGroup == 0, "whole DMA operations");
  static_assert(kGroup >= 128, "a DMA operation covers a multiple of 16 rows: one swizzle per thread");
  static_assert(kBytes <= 160 * 1024 && kThreads <= 1024, "one workgroup per CU");
};

// An out-of-range lane offset: the operands end below 2^31 bytes from the tile's first row.
constexpr uint32_t kOut = 0x80000000u;
inline bool offsets_fit(int64_t rows, int64_t lda, int64_t ldb, int64_t K, int64_t ssam, int64_t ssak) {
  const int64_t lim = (int64_t)1 << 31, nk = cdiv(K, 128);
  return K < lim - 4096 && rows * lda + K < lim && rows * ldb + K < lim && (rows * ssam + nk * ssak + 1) * 4 < lim;
}

// Four consecutive columns of C: whole (aligned and inside the tile) or one by one.
__device__ __forceinline__ void store4(void* C, int64_t off, int c_dtype, const float4 v, int valid) {
  const float x[4] = {v.x, v.y, v.z, v.w};
  if (c_dtype == CIN_DT_F32) {
    float* p = static_cast<float*>(C) + off;
    if (valid >= 4 && (((uintptr_t)p) & 15) == 0)
      *reinterpret_cast<float4*>(p) = v;
    else
      for (int r = 0; r < 4; ++r)
        if (r < valid) p[r] = x[r];
  } else {
    uint16_t* p = static_cast<uint16_t*>(C) + off;
    const uint32_t b[4] = {f32_to_half_bits(c_dtype, x[0]), f32_to_half_bits(c_dtype, x[1]),
                           f32_to_half_bits(c_dtype, x[2]), f32_to_half_bits(c_dtype, x[3])};
    if (valid >= 4 && (((uintptr_t)p) & 7) == 0)
      *reinterpret_cast<uint2*>(p) = make_uint2(b[0] | (b[1] << 16), b[2] | (b[3] << 16));
    else
      for (int r = 0; r < 4; ++r)
        if (r < valid) p[r] = (uint16_t)b[r];
  }
}

// TAIL: K % 128 != 0, the last block's chunks past K read as zero.  With one group the sums start at
// K block kb0 and wrap around (see grouped_first_block in gemm.hip).
template <class C, bool TAIL>
__device__ __forceinline__ void tile(const Tile& t, int64_t lda, int64_t ssam, int64_t ssak, int64_t ldb,
                                     int64_t ssbk, int K, int c_dtype, int64_t ldc, uint8_t* smem, int kb0 = 0) {
  constexpr int WN = C::WN, MT = C::MT, NT = C::NT, KS = C::KS;
  const int lane = threadIdx.x & 63;
  const int wave_all = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int grp = wave_all / (C::WM * WN), wave = wave_all % (C::WM * WN);
  const int tid = wave * 64 + lane;  // within the group
  const int wm = wave / WN, wn = wave % WN;
  const int l16 = lane & 15, kq = lane >> 4;
  const int nkb = (K + 127) >> 7, nk = (nkb + KS - 1) / KS;
  const __amdgpu_buffer_rsrc_t ra = make_rsrc(t.A, (int64_t)(t.rows_a - 1) * lda + K);
  const __amdgpu_buffer_rsrc_t rb = make_rsrc(t.B, (int64_t)(t.rows_b - 1) * ldb + K);
  const __amdgpu_buffer_rsrc_t rsa =
      make_rsrc(t.sa, ((int64_t)(t.rows_a - 1) * ssam + (int64_t)(nkb - 1) * ssak + 1) * 4);
  // DMA operation i: thread t covers row i * kGroup / 8 + t / 8, 16-byte chunk (t % 8) ^ f(row)
  const int r0 = tid >> 3, ch = (tid & 7) ^ swz_f(r0);
  const uint32_t offA = (uint32_t)(r0 * lda) + ch * 16, offB = (uint32_t)(r0 * ldb) + ch * 16;
  const uint32_t stepA = (uint32_t)(C::kGroup / 8 * lda), stepB = (uint32_t)(C::kGroup / 8 * ldb);
  const uint32_t offS = tid < t.rows_a ? (uint32_t)(tid * ssam * 4) : kOut;
  const uint32_t ssak4 = (uint32_t)(ssak * 4);
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem + (uint32_t)(grp * C::kBlock + wave * 1024);
  const uint32_t lds0s = (uint32_t)(uintptr_t)smem + (uint32_t)(grp * C::kBlock + C::kA + C::kB + wave * 256);
  auto block = [&](int k) {
    if constexpr (KS > 1) return k * KS + grp;
    return k + kb0 < nkb ? k + kb0 : k + kb0 - nkb;
  };
  // the group's K block of iteration k; past the last block everything reads as zero
  auto dma = [&](int k, int stg) {
    const int kb = block(k);
    const uint32_t so = (uint32_t)kb * 128u;
    uint32_t out = 0;
    if constexpr (TAIL || KS > 1) out = kb * 128 + ch * 16 < K ? 0u : kOut;
    const uint32_t base = lds0 + (uint32_t)(stg * C::kStage);
#pragma unroll
    for (int i = 0; i < C::kOpsA; ++i) dma16(ra, (offA + i * stepA) | out, so, base + i * C::kGroup * 16);
#pragma unroll
    for (int i = 0; i < C::kOpsB; ++i) dma16(rb, (offB + i * stepB) | out, so, base + C::kA + i * C::kGroup * 16);
    dma4(rsa, offS | (kb < nkb ? 0u : kOut), (uint32_t)kb * ssak4, lds0s + (uint32_t)(stg * C::kStage));
  };
  const int fsw = swz_f(l16);
  const uint32_t fbase = (uint32_t)(grp * C::kBlock);
  const uint32_t fa = fbase + (uint32_t)((wm * 16 * MT + l16) * 128 + (((2 * kq) ^ fsw) << 4));
  const uint32_t fb = fbase + (uint32_t)(C::kA + (wn * 16 * NT + l16) * 128 + (((2 * kq) ^ fsw) << 4));
  const uint32_t fs = fbase + (uint32_t)(C::kA + C::kB + (wm * 16 * MT + l16) * 4);
  auto frag = [&](uint32_t o) {
    const uint4 lo = *reinterpret_cast<const uint4*>(smem + o);
    const uint4 hi = *reinterpret_cast<const uint4*>(smem + (o ^ 16u));
    v8i v;
    v[0] = (int)lo.x; v[1] = (int)lo.y; v[2] = (int)lo.z; v[3] = (int)lo.w;
    v[4] = (int)hi.x; v[5] = (int)hi.y; v[6] = (int)hi.z; v[7] = (int)hi.w;
    return v;
  };
  // the B scales of 64 iterations, one per lane (zero past the last block): a scale loaded
  // where it is used would put its latency into every iteration
  auto load_sb = [&](int k) {
    const int kb = block(k + lane);
    return kb < nkb ? t.sb[(int64_t)kb * ssbk] : 0.0f;
  };
  v4f acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
  float sbv = load_sb(0);
  if (nk > 0) dma(0, 0);
  for (int k = 0; k < nk; ++k) {
    if (k != 0 && (k & 63) == 0) sbv = load_sb(k);
    wait_dma();
    lds_barrier();  // block k has landed, and block k - 1's stage has been read
    if (k + 1 < nk) dma(k + 1, (k + 1) & 1);
    const float sb = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(sbv), k & 63));
    const uint32_t so = (uint32_t)((k & 1) * C::kStage);
    v8i bf[NT];
    float cs[MT];
#pragma unroll
    for (int j = 0; j < NT; ++j) bf[j] = frag(fb + so + j * 2048);
#pragma unroll
    for (int i = 0; i < MT; ++i) cs[i] = *reinterpret_cast<const float*>(smem + fs + so + i * 64);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const v8i af = frag(fa + so + i * 2048);
      const float c = cs[i] * sb;
      v4f p[NT];
      const v4f zero = {0.f, 0.f, 0.f, 0.f};
      // D[n][m] = sum_k B[n, k] A[m, k]: the lane holds m = l16, n = 4 kq + r
#pragma unroll
      for (int j = 0; j < NT; ++j)
        p[j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bf[j], af, zero, 0, 0, 0, 0, 0, 0);
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][j][r] = fmaf(p[j][r], c, acc[i][j][r]);
    }
  }
  lds_barrier();  // every fragment has been read: the stages become the groups' fp32 tiles
  float* cl = reinterpret_cast<float*>(smem);
  constexpr int kCTile = C::TM * C::kCStride;
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
      *reinterpret_cast<float4*>(cl + grp * kCTile + (wm * 16 * MT + i * 16 + l16) * C::kCStride + wn * 16 * NT +
                                 j * 16 + kq * 4) =
          make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
  __syncthreads();
  constexpr int kQuads = C::TM * C::TN / 4;
  for (int q = threadIdx.x; q < kQuads; q += C::kThreads) {
    const int m = q / (C::TN / 4), n = (q % (C::TN / 4)) * 4;
    if (m >= t.rows_a || n >= t.rows_b) continue;
    const float* p = cl + m * C::kCStride + n;
    float4 s = *reinterpret_cast<const float4*>(p);
#pragma unroll
    for (int g = 1; g < KS; ++g) {
      const float4 o = *reinterpret_cast<const float4*>(p + g * kCTile);
      s.x += o.x; s.y += o.y; s.z += o.z; s.w += o.w;
    }
    store4(t.C, (int64_t)m * ldc + n, c_dtype, s, t.rows_b - n);
  }
}

}  // namespace gt
}  // namespace cin
