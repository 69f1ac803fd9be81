// Unquantized grouped GEMM for MoE experts on gfx950 fp16 MFMA: the reference's
// moe_grouped_gemm / grouped_gemm_kernel (src/kernels.py:440-581).
//
//   C[r, n] = fp16( sum_k fp16(A[r, k]) * fp16(B_e[n, k]) )   for rows r of expert e
//
// Operands are rounded to fp16 (round-to-nearest-even) as the reference's
// a.to(tl.float16) / b.to(tl.float16) do, the products are summed in fp32 by
// v_mfma_f32_16x16x32_f16, and the result is stored as fp16 (RNE).  One launch covers all
// experts: a workgroup finds its (expert, row tile) from the device-side ranges, so there is
// no host synchronisation and no grid sized by the largest expert.
// Rows outside every expert range are not written (the reference returns torch.empty).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "cin_common.h"
#include "cin_grouped.h"
#include "cin_runtime.h"

using namespace cin;

namespace {

constexpr int BK = 64;                      // K step per LDS stage
constexpr int kRowBytes = BK * 2;           // one fp16 tile row: 8 chunks of 16 bytes

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

// chunk c of tile row r sits at slot c ^ f(r) (the same swizzle as the FP8 GEMM's
// 128-byte rows: conflict-free fragment reads)
__device__ inline int swz_f(int r) { return (r & 7) ^ ((r >> 3) & 1); }

// ---------------------------------------------------------------------------
// Workgroup tiles of 16 MT WM x 16 NT WN, K steps of 64 through two LDS stages.  Each thread
// keeps the next step's operands in flight in registers, in their own dtype, while the current
// step's MFMAs run, then converts them to fp16 on the way into LDS: no converted copy of the
// weights is ever stored.  A wider tile reads fp32 weights less often: with 256 x 256 tiles a
// step's 96 KB of operands (fp32 weights, 16-bit rows) take about 1500 cycles at 64 B / clk and
// its MFMAs 2048, with 128 x 128 tiles 768 and 512.  Rows past an expert or past N and elements
// past K read as zero.  32768 Zipf rows, 16 experts, 2048 x 1024, bf16 rows: 217 us with fp32
// weights, 174 with bf16 (128 x 128 tiles that waited for each step's loads: 400 and 280, the
// same bits): 0.63 and 0.79 PFLOP/s, with 1088 tiles in five rounds of 256.
// ---------------------------------------------------------------------------
typedef unsigned int v4u __attribute__((ext_vector_type(4)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef float f2 __attribute__((ext_vector_type(2)));
constexpr uint32_t kOut = 0x80000000u;  // an out-of-range lane offset

__device__ inline h2 to_h2(float a, float b) { return __builtin_convertvector(f2{a, b}, h2); }

// One operand's share of a K step: ROWS rows x 64 elements over THREADS threads, 16 bytes of
// the source dtype per thread and operation.
// ALIGNED: rows start on 16 bytes, K % 8 == 0 and a tile's rows lie within 2^31 bytes (buffer
// loads, out-of-range lanes read zero).  Otherwise the 16 bytes come from 64-bit addresses and
// any element alignment, and the last ones of a row element by element.
template <int DT, int ROWS, int THREADS, bool ALIGNED>
struct Operand {
  static constexpr int kEs = DT == CIN_DT_F32 ? 4 : 2;
  static constexpr int kPer = 16 / kEs;
  static constexpr int kLanes = 64 * kEs / 16;  // threads of one row
  static constexpr int kOps = ROWS * kLanes / THREADS;
  static constexpr int kRowsPerOp = THREADS / kLanes;
  static_assert(ROWS * kLanes % THREADS == 0 && kRowsPerOp % 16 == 0, "whole operations, one swizzle per thread");
  v4u r[kOps];
  __amdgpu_buffer_rsrc_t rsrc;
  uint32_t off, step;
  const uint8_t* p;  // !ALIGNED: the thread's first element of operation 0
  int64_t stride;    // bytes between operations
  int row, rows;
  uint32_t lds;  // byte offset of operation 0 in a stage
  int k;         // first element of the thread's 16 bytes within a step

  __device__ __forceinline__ void init(const void* base, int64_t ld, int rows_, int64_t K, int tid) {
    row = tid / kLanes;
    rows = rows_;
    const int c = tid % kLanes;
    k = c * kPer;
    if constexpr (ALIGNED) {
      rsrc = make_rsrc(base, ((int64_t)(rows - 1) * ld + K) * kEs);
      off = (uint32_t)(row * ld * kEs) + c * 16;
      step = (uint32_t)(kRowsPerOp * ld * kEs);
    } else {
      p = static_cast<const uint8_t*>(base) + (row * ld + k) * kEs;
      stride = kRowsPerOp * ld * kEs;
    }
    const int chunk = DT == CIN_DT_F32 ? c >> 1 : c;
    lds = (uint32_t)(row * kRowBytes + ((chunk ^ swz_f(row)) << 4) + (DT == CIN_DT_F32 ? (c & 1) * 8 : 0));
  }
  __device__ __forceinline__ void fetch(int64_t k0, int64_t K) {
    if constexpr (ALIGNED) {
      const uint32_t out = k0 + k < K ? 0u : kOut;
#pragma unroll
      for (int i = 0; i < kOps; ++i)
        r[i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (off + i * step) | out, (uint32_t)(k0 * kEs), 0);
    } else {
      const int64_t left = K - k0 - k;  // elements of the row from the thread's first one on
      if (left >= kPer) {
#pragma unroll
        for (int i = 0; i < kOps; ++i) {
          r[i] = v4u{0u, 0u, 0u, 0u};
          if (row + i * kRowsPerOp < rows) __builtin_memcpy(&r[i], p + i * stride + k0 * kEs, 16);
        }
      } else {
#pragma unroll
        for (int i = 0; i < kOps; ++i) {
          r[i] = v4u{0u, 0u, 0u, 0u};
#pragma unroll
          for (int e = 0; e < kPer; ++e) {
            if (e >= left || row + i * kRowsPerOp >= rows) continue;
            const uint8_t* q = p + i * stride + (k0 + e) * kEs;
            if constexpr (kEs == 4)
              r[i][e] = *reinterpret_cast<const uint32_t*>(q);
            else
              r[i][e >> 1] |= (uint32_t)*reinterpret_cast<const uint16_t*>(q) << (16 * (e & 1));
          }
        }
      }
    }
  }
  __device__ __forceinline__ void store(uint8_t* stage) const {
#pragma unroll
    for (int i = 0; i < kOps; ++i) {
      uint8_t* d = stage + lds + i * kRowsPerOp * kRowBytes;
      if constexpr (DT == CIN_DT_F32) {
        const h2 a = to_h2(__uint_as_float(r[i][0]), __uint_as_float(r[i][1]));
        const h2 b = to_h2(__uint_as_float(r[i][2]), __uint_as_float(r[i][3]));
        *reinterpret_cast<h4*>(d) = h4{a[0], a[1], b[0], b[1]};
      } else if constexpr (DT == CIN_DT_F16) {
        *reinterpret_cast<v4u*>(d) = r[i];
      } else {
        h8 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const h2 a = to_h2(bf16_lo(r[i][e]), bf16_hi(r[i][e]));
          o[2 * e] = a[0];
          o[2 * e + 1] = a[1];
        }
        *reinterpret_cast<h8*>(d) = o;
      }
    }
  }
};

template <int WM_, int WN_, int MT_, int NT_>
struct Cfg16 {
  static constexpr int WM = WM_, WN = WN_, MT = MT_, NT = NT_;
  static constexpr int kThreads = 64 * WM * WN, TM = 16 * MT * WM, TN = 16 * NT * WN;
  static constexpr int kStage = (TM + TN) * kRowBytes;
  static constexpr int kCStride = TN * 2 + 16;  // bytes; rows 4 banks apart
  static constexpr int kBytes = 2 * kStage > TM * kCStride ? 2 * kStage : TM * kCStride;
};
using W256 = Cfg16<2, 4, 8, 4>;    // 8 waves of 128 x 64
using W128 = Cfg16<4, 2, 2, 4>;    // 8 waves of 32 x 64, two workgroups a CU
using W64x128 = Cfg16<2, 2, 2, 4>; // 4 waves of 32 x 64, three workgroups a CU

template <class C, int ADT, int BDT, bool ALIGNED>
__global__ __launch_bounds__(C::kThreads, 2) void k_grouped_gemm_f16_tile(
    const void* __restrict__ A, int64_t lda, const void* __restrict__ B, int64_t sbe, int64_t ldb,
    const int64_t* __restrict__ starts, const int64_t* __restrict__ ends, int64_t E, int64_t T,
    int64_t N, int64_t K, _Float16* __restrict__ Cp, int64_t ldc, uint32_t tiles_n) {
  __shared__ __attribute__((aligned(128))) uint8_t smem[C::kBytes];
  constexpr int MT = C::MT, NT = C::NT;
  uint32_t tn;
  int64_t e, r0, r1;
  if (!find_tile<C::TM>(starts, ends, E, T, tiles_n, e, r0, r1, tn)) return;  // the whole workgroup
  const int nr = __builtin_amdgcn_readfirstlane((int)(r1 - r0 < C::TM ? r1 - r0 : C::TM));
  const int64_t n0 = (int64_t)tn * C::TN;
  const int nc = (int)(N - n0 < C::TN ? N - n0 : C::TN);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / C::WN, wn = wave % C::WN;
  const int l16 = lane & 15, kq = lane >> 4;
  Operand<ADT, C::TM, C::kThreads, ALIGNED> oa;
  Operand<BDT, C::TN, C::kThreads, ALIGNED> ob;
  oa.init(static_cast<const uint8_t*>(A) + r0 * lda * oa.kEs, lda, nr, K, tid);
  ob.init(static_cast<const uint8_t*>(B) + (e * sbe + n0 * ldb) * ob.kEs, ldb, nc, K, tid);
  const int fsw = swz_f(l16);
  const uint32_t fa = (uint32_t)((wm * 16 * MT + l16) * kRowBytes);
  const uint32_t fb = (uint32_t)((C::TM + wn * 16 * NT + l16) * kRowBytes);

  v4f acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
  const int nkt = (int)((K + BK - 1) / BK);
  // half of a K step: 32 elements
  auto half = [&](const uint8_t* st, int ks) {
    const uint32_t ck = (uint32_t)(((4 * ks + kq) ^ fsw) << 4);
    h8 bfr[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) bfr[j] = *reinterpret_cast<const h8*>(st + fb + j * 16 * kRowBytes + ck);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const h8 afr = *reinterpret_cast<const h8*>(st + fa + i * 16 * kRowBytes + ck);
#pragma unroll
      for (int j = 0; j < NT; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bfr[j], afr, acc[i][j], 0, 0, 0);
    }
  };
  oa.fetch(0, K);
  ob.fetch(0, K);
  oa.store(smem);
  ob.store(smem + C::TM * kRowBytes);
  if (nkt > 1) {
    oa.fetch(BK, K);
    ob.fetch(BK, K);
  }
  __syncthreads();
  for (int kt = 0; kt < nkt; ++kt) {
    const uint8_t* st = smem + (kt & 1) * C::kStage;
    half(st, 0);
    if (kt + 1 < nkt) {
      // step kt + 1, in flight since step kt - 1, into the stage read last in that step
      uint8_t* nx = smem + ((kt + 1) & 1) * C::kStage;
      oa.store(nx);
      ob.store(nx + C::TM * kRowBytes);
      if (kt + 2 < nkt) {
        oa.fetch((int64_t)(kt + 2) * BK, K);
        ob.fetch((int64_t)(kt + 2) * BK, K);
      }
    }
    half(st, 1);
    __syncthreads();
  }
  // fp16 rows through LDS: a lane holds C[m = l16][n = 4 kq .. + 3]
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const h2 a = to_h2(acc[i][j][0], acc[i][j][1]), c = to_h2(acc[i][j][2], acc[i][j][3]);
      *reinterpret_cast<h4*>(smem + (wm * 16 * MT + i * 16 + l16) * C::kCStride + (wn * 16 * NT + j * 16 + kq * 4) * 2) =
          h4{a[0], a[1], c[0], c[1]};
    }
  __syncthreads();
  constexpr int kChunks = C::TN / 8;
  for (int q = tid; q < C::TM * kChunks; q += C::kThreads) {
    const int m = q / kChunks, n = (q % kChunks) * 8;
    if (m >= nr || n >= nc) continue;
    _Float16* cp = Cp + (r0 + m) * ldc + n0 + n;
    const h8 v = *reinterpret_cast<const h8*>(smem + m * C::kCStride + n * 2);
    if (n + 8 <= nc && (((uintptr_t)cp) & 15) == 0)
      *reinterpret_cast<h8*>(cp) = v;
    else
      for (int r = 0; r < 8; ++r)
        if (n + r < nc) cp[r] = v[r];
  }
}

inline bool valid_dtype(int dt) { return dt == CIN_DT_BF16 || dt == CIN_DT_F32 || dt == CIN_DT_F16; }
inline int elem_size(int dt) { return dt == CIN_DT_F32 ? 4 : 2; }

struct Args {
  const void* A;
  int64_t lda;
  const void* B;
  int64_t sbe, ldb;
  const int64_t *starts, *ends;
  int64_t E, T, N, K;
  _Float16* C;
  int64_t ldc;
};

template <class C, int ADT, int BDT, bool ALIGNED>
void launch_tile(const Args& a, hipStream_t s) {
  const int64_t tm = cdiv(a.T, C::TM) + a.E - 1, tn = cdiv(a.N, C::TN);
  hipLaunchKernelGGL((k_grouped_gemm_f16_tile<C, ADT, BDT, ALIGNED>), (unsigned)(tm * tn), C::kThreads, 0, s, a.A,
                     a.lda, a.B, a.sbe, a.ldb, a.starts, a.ends, a.E, a.T, a.N, a.K, a.C, a.ldc, (uint32_t)tn);
}

template <int ADT, int BDT>
void launch(const Args& a, hipStream_t s) {
  const int ea = elem_size(ADT), eb = elem_size(BDT);
  const bool rows16 = ((uintptr_t)a.A % 16) == 0 && ((uintptr_t)a.B % 16) == 0 && (a.lda * ea) % 16 == 0 &&
                      (a.ldb * eb) % 16 == 0 && (a.sbe * eb) % 16 == 0;
  const int64_t lim = (int64_t)1 << 31;  // lane offsets from a tile's first row
  const bool few = a.T <= 64 * a.E && (cdiv(a.T, 64) + a.E) * cdiv(a.N, 128) < lim;
  if (rows16 && a.K % 8 == 0 && (256 * a.lda + a.K) * ea < lim && (256 * a.ldb + a.K) * eb < lim) {
    // us, 256 x 256 / 128 x 128 / 64 x 128 tiles, fp32 and bf16 weights, T, E, N, K: 32768, 16, 2048,
    // 1024 (four rounds of 256 x 256): 217, 174 / 236, 208 / 297, 240; 16384 (two): 120, 109 / 120,
    // 105 / 151, 123; 8192 (one): 76, 67 / 69, 60 / 86, 69; 1024 (64 rows an expert): 37, 34 / 31, 24 /
    // 33, 19; 64: 37, 34 / 22, 17 / 22, 15.
    if (a.T / 256 * cdiv(a.N, 256) >= 2 * (int64_t)cin_device_cus())
      launch_tile<W256, ADT, BDT, true>(a, s);
    else if (few)
      launch_tile<W64x128, ADT, BDT, true>(a, s);
    else
      launch_tile<W128, ADT, BDT, true>(a, s);
  } else if (few) {
    // (31899, 16, 256, 1315, bf16: 842 us element by element, 65 so; 696, 32, 368, 541: 149, 16)
    launch_tile<W64x128, ADT, BDT, false>(a, s);
  } else {
    launch_tile<W128, ADT, BDT, false>(a, s);
  }
}

template <int ADT>
void launch_b(int b_dtype, const Args& a, hipStream_t s) {
  if (b_dtype == CIN_DT_BF16)
    launch<ADT, CIN_DT_BF16>(a, s);
  else if (b_dtype == CIN_DT_F16)
    launch<ADT, CIN_DT_F16>(a, s);
  else
    launch<ADT, CIN_DT_F32>(a, s);
}

}  // namespace

extern "C" {

int cin_grouped_gemm_f16(const void* A, int a_dtype, int64_t lda, const void* B, int b_dtype,
                         int64_t sbe, int64_t ldb, const int64_t* starts, const int64_t* ends,
                         int64_t E, int64_t T, int64_t N, int64_t K, void* C, int64_t ldc,
                         void* stream) {
  CIN_CHECK_ARG(valid_dtype(a_dtype) && valid_dtype(b_dtype), "grouped_gemm_f16: unsupported dtype");
  CIN_CHECK_ARG(E >= 0 && T >= 0 && N >= 0 && K >= 0, "grouped_gemm_f16: negative shape");
  if (E == 0 || T == 0 || N == 0) return CIN_OK;
  CIN_CHECK_ARG(A && B && starts && ends && C, "grouped_gemm_f16: null pointer");
  CIN_CHECK_ARG(lda >= K && ldb >= K && ldc >= N && sbe >= 0, "grouped_gemm_f16: bad strides");
  CIN_CHECK_ARG((cdiv(T, 128) + E) * cdiv(N, 128) < ((int64_t)1 << 31), "grouped_gemm_f16: grid too large");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const Args a = {A, lda, B, sbe, ldb, starts, ends, E, T, N, K, static_cast<_Float16*>(C), ldc};
  if (a_dtype == CIN_DT_BF16)
    launch_b<CIN_DT_BF16>(b_dtype, a, s);
  else if (a_dtype == CIN_DT_F16)
    launch_b<CIN_DT_F16>(b_dtype, a, s);
  else
    launch_b<CIN_DT_F32>(b_dtype, a, s);
  return cin_check_launch("grouped_gemm_f16");
}

}  // extern "C"
