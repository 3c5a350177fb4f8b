// On-device cross-check kernels (SIMT, no matrix cores).
//
//  * fp32 mode: the reference's GEMM_Naive (mmm.cpp:52-62) -- one fp32 accumulator per output,
//    k ascending, acc += float(a) * float(b).  The product of two fp16 values is exact in fp32,
//    so fused and unfused multiply-add round identically and the result is bit-reproducible
//    on the CPU with the same loop.
//  * fp64 mode: T = sum_k a*b and S = sum_k |a*b| in fp64, k ascending (products exact in
//    fp64).  T is the ground truth and S the scale of the tolerance |C - T| <= rel * S,
//    for every element of a full-size output instead of a sampled sub-grid.
//
// Both take any two-level fold per axis (a plain GEMM is the fold with high extents of 1), so
// they check the tensor contractions at their own layouts as well.  The order of the additions per
// output is the plain ascending-k loop whatever the tiling.
//
// Bound by the vector FMA rate (fp64: two FMAs per term with S; 65 TFLOP/s measured in a loop of
// independent v_fma_f64, v_mfma_f64_16x16x4 47).  fp16 products are exact in either type, so one FMA
// is the multiply and the add.  A thread holds RM x RN outputs (T and S), so a k costs RM + RN LDS
// values for 2 RM RN FMAs; operands are converted once, when they are staged, and lie in LDS in the
// accumulator's type, so the loop is LDS reads and FMAs only.  K stages are double-buffered through
// registers, deeper with fewer outputs per thread (a stage has to cover the next one's loads: 64 x 64
// x 2048 119 us with 16 k a stage, 98 with 64).  Measured on MI355X, T and S, against the kernel before
// (4x4 outputs, converted per use, multiply, add and |.| apart): 2048^3 1939 -> 660 us (52 TFLOP/s),
// 4096 x 4096 x 1024 3559 -> 1231, 1000^3 366 -> 142, 512 x 512 x 2048 647 -> 106, 64 x 64 x 2048 642 ->
// 98; T alone 2048^3 1931 -> 458, the fp32 mode 562 -> 307.  Few outputs are bound by one k after the
// other per output, which the defined order asks for.
#include <type_traits>

#include "mmm_kernels.h"

namespace mmm {
namespace {

__device__ __forceinline__ int64_t fold_index(int x, int lo, const int64_t* s) {
  if (x < lo) return (int64_t)x * s[1];
  return (int64_t)(x / lo) * s[0] + (int64_t)(x % lo) * s[1];
}

enum CheckMode { kNaiveF32, kTruth, kTruthScale };

// 256 threads, tile 16 RM x 16 RN; thread (tr, tc) holds rows 2 tr + e + 32 h and columns 2 tc + e +
// 32 h (pairs: one 2-element LDS read each, neighbouring threads on neighbouring pairs); K in stages
// of KD.
template <int MODE, int RM, int RN, int KD>
__global__ __launch_bounds__(256) void check_fold_kernel(FoldProblem p, double* T, double* S, int tiles_n) {
  using Acc = std::conditional_t<MODE == kNaiveF32, float, double>;
  typedef Acc Acc2 __attribute__((ext_vector_type(2)));
  constexpr int BM = 16 * RM, BN = 16 * RN;
  // rows padded by 4 against bank conflicts of the stores along k
  __shared__ __attribute__((aligned(16))) Acc As[2][KD][BM + 4];  // [k][m]
  __shared__ __attribute__((aligned(16))) Acc Bs[2][KD][BN + 4];  // [k][n]
  const int t = threadIdx.x;
  const int m0 = (int)(blockIdx.x / tiles_n) * BM, n0 = (int)(blockIdx.x % tiles_n) * BN;

  // Staging: A with lanes along k (k-contiguous operands coalesce), B with lanes along n.
  const int a_k = t % KD, a_m = t / KD;  // rows a_m + 256 / KD * i
  const int b_n = t % BN, b_k = t / BN;    // k rows b_k + 256 / BN * i
  constexpr int LA = BM * KD / 256, LB = BN * KD / 256;  // elements per thread and stage
  int64_t a_row[LA];
#pragma unroll
  for (int i = 0; i < LA; ++i) {
    const int m = m0 + a_m + 256 / KD * i;
    a_row[i] = m < p.M ? fold_index(m, p.m_lo, p.am) : -1;
  }
  const int gn = n0 + b_n;
  const int64_t b_col = gn < p.N ? fold_index(gn, p.n_lo, p.bn) : -1;

  const int tr = t / 16, tc = t % 16;
  Acc acc[RM][RN], sab[MODE == kTruthScale ? RM : 1][RN];
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < RN; ++j) {
      acc[i][j] = 0;
      if constexpr (MODE == kTruthScale) sab[i][j] = 0;
    }

  // elements past M, N or K are zero: their terms add nothing (fma(0, 0, x) is x)
  mmm_half ra[LA], rb[LB];
  auto load = [&](int k0) {
    const int k = k0 + a_k;
    const int64_t ko = k < p.K ? fold_index(k, p.k_lo, p.ak) : -1;
#pragma unroll
    for (int i = 0; i < LA; ++i) ra[i] = ko >= 0 && a_row[i] >= 0 ? p.A[a_row[i] + ko] : (mmm_half)0;
#pragma unroll
    for (int i = 0; i < LB; ++i) {
      int kb = k0 + b_k + 256 / BN * i;
      if constexpr (BN >= 64) kb = __builtin_amdgcn_readfirstlane(kb);
      rb[i] = kb < p.K && b_col >= 0 ? p.B[fold_index(kb, p.k_lo, p.bk) + b_col] : (mmm_half)0;
    }
  };
  auto value = [](mmm_half h) { return (Acc)(float)__builtin_bit_cast(_Float16, h); };
  auto store = [&](int st) {
#pragma unroll
    for (int i = 0; i < LA; ++i) As[st][a_k][a_m + 256 / KD * i] = value(ra[i]);
#pragma unroll
    for (int i = 0; i < LB; ++i) Bs[st][b_k + 256 / BN * i][b_n] = value(rb[i]);
  };

  if (p.K > 0) {
    load(0);
    store(0);
  }
  __syncthreads();
  for (int k0 = 0, st = 0; k0 < p.K; k0 += KD, st ^= 1) {
    const bool more = k0 + KD < p.K;
    if (more) load(k0 + KD);
#pragma unroll 4
    for (int kk = 0; kk < KD; ++kk) {
      Acc2 a[RM / 2], b[RN / 2];
#pragma unroll
      for (int h = 0; h < RM / 2; ++h) a[h] = *(const Acc2*)&As[st][kk][2 * tr + 32 * h];
#pragma unroll
      for (int h = 0; h < RN / 2; ++h) b[h] = *(const Acc2*)&Bs[st][kk][2 * tc + 32 * h];
#pragma unroll
      for (int i = 0; i < RM; ++i)
#pragma unroll
        for (int j = 0; j < RN; ++j) {
          const Acc x = a[i / 2][i % 2], y = b[j / 2][j % 2];
          if constexpr (MODE == kNaiveF32) {
            acc[i][j] = __builtin_fmaf(x, y, acc[i][j]);
          } else {
            acc[i][j] = __builtin_fma(x, y, acc[i][j]);
            if constexpr (MODE == kTruthScale)
              sab[i][j] = __builtin_fma(__builtin_fabs(x), __builtin_fabs(y), sab[i][j]);
          }
        }
    }
    if (more) store(st ^ 1);
    __syncthreads();
  }

#pragma unroll
  for (int i = 0; i < RM; ++i) {
    const int m = m0 + 2 * tr + i % 2 + 32 * (i / 2);
    if (m >= p.M) continue;
    const int64_t row = fold_index(m, p.m_lo, p.cm);
#pragma unroll
    for (int j = 0; j < RN; ++j) {
      const int n = n0 + 2 * tc + j % 2 + 32 * (j / 2);
      if (n >= p.N) continue;
      const int64_t o = row + fold_index(n, p.n_lo, p.cn);
      if constexpr (MODE == kNaiveF32) {
        p.C[o] = acc[i][j];
      } else {
        T[o] = acc[i][j];
        if constexpr (MODE == kTruthScale) S[o] = sab[i][j];
      }
    }
  }
}

template <int MODE, int RM, int RN, int KD>
hipError_t launch_tiles(const FoldProblem& p, double* T, double* S, hipStream_t stream) {
  const int64_t tiles_m = (p.M + 16 * RM - 1) / (16 * RM), tiles_n = (p.N + 16 * RN - 1) / (16 * RN);
  if (tiles_m * tiles_n > 0x7fffffff) return hipErrorInvalidValue;
  check_fold_kernel<MODE, RM, RN, KD>
      <<<dim3((unsigned)(tiles_m * tiles_n)), dim3(256), 0, stream>>>(p, T, S, (int)tiles_n);
  return hipGetLastError();
}

// The largest outputs per thread that still give every CU a workgroup (K cannot be split: the sum's
// order is the result).
template <int MODE>
hipError_t launch_mode(const FoldProblem& p, double* T, double* S, hipStream_t stream) {
  const double outputs = (double)p.M * p.N;
  if (outputs >= 256.0 * 128 * 64) return launch_tiles<MODE, 8, 4, 16>(p, T, S, stream);
  if (outputs >= 256.0 * 64 * 64) return launch_tiles<MODE, 4, 4, 32>(p, T, S, stream);
  return launch_tiles<MODE, 2, 2, 64>(p, T, S, stream);
}

}  // namespace

hipError_t launch_check_fold(const FoldProblem& p, double* T, double* S, hipStream_t stream) {
  if (!T) return launch_mode<kNaiveF32>(p, nullptr, nullptr, stream);
  return S ? launch_mode<kTruthScale>(p, T, S, stream) : launch_mode<kTruth>(p, T, S, stream);
}

}  // namespace mmm
