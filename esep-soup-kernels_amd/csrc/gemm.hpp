// MFMA GEMM (kernels in gemm.hip): C[M, N] = A[M, K] . B, B given as [N, K] or as [K, N].
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace esep {

struct GemmArgs {
  const void* a;
  int64_t lda;
  const void* b;
  int64_t ldb;
  const void* bias;  // [N] of the operands' type, or null
  void* c;
  int64_t ldc;
  float* part;  // [splits][M][N] fp32 partial sums (splits > 1)
  int64_t M, N, K;
  int tiles_m, tiles_n;
  int splits;
  int steps;  // 64-deep steps per split (the last split takes what is left)
};

// The tile shapes a launch may take (rows x columns of C per block).
constexpr int kGemm256x256 = 0, kGemm128x256 = 1, kGemm256x128 = 2, kGemm128x128 = 3,
              kGemm64x128 = 4;

struct GemmPlan {
  int shape, splits;
  double us;  // expected
};

// Tile shape and splits of the contraction for a product of this size (K a multiple of 64).
GemmPlan gemm_plan(int64_t M, int64_t N, int64_t K);
// Whether it is expected to beat the vendor BLAS there.
bool gemm_pays(int64_t M, int64_t N, int64_t K, bool b_kn);

// out_dt 0: fp32, else the operands' type
hipError_t launch_gemm(const GemmArgs& a, int shape, int b_kn, int dt, int out_dt, hipStream_t s,
                       bool* sup);

}  // namespace esep
