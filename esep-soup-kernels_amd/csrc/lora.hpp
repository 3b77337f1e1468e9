// Fused LoRA products (kernels in lora.hip): the skinny GEMMs of a LoRA term with the dropout
// mask regenerated inside them.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace esep {

constexpr int kLoraMaxRank = 64;
constexpr int kLoraMaxRows = 1 << 22;  // k_lora_up's grid: 64 rows per y block

// out[T, r] = scale * drop(x)[T, K] . W^T, W given as [r, K], or as [K, r] with w_kr.
struct LoraDownArgs {
  const void* x;
  int64_t ld_x;
  const void* w;
  const int64_t* key;  // null: no dropout
  float p, inv_keep, scale;
  void* out;
  int64_t T, K;
  int r;
};

// out[T, N] = [base +] scale * xa[T, r] . B[N, r]^T.
struct LoraUpArgs {
  const void* xa;
  const void* b;
  const void* base;  // null: none
  int64_t ld_base;
  void* out;
  int64_t ld_out;
  float scale;
  int64_t T, N;
  int r;
};

// dx[T, K] = [dx +] (dxa . A) * keep / (1 - p), dA[r, K] = dxa^T . drop(x) and
// dB[N, r] = scale * dterm^T . xa. Either half may be absent (x or dterm null).
struct LoraGradArgs {
  const void* x;
  const void* a;
  const void* dxa;
  const int64_t* key;
  float p, inv_keep, scale;
  void* dx;  // null: not wanted
  int accumulate;
  const void* dterm;
  int64_t ld_dterm;
  const void* xa;
  float* da;
  float* db;
  float* part;  // [chunks][r K] then [chunks][N r]
  int64_t T, K, N;
  int r;
  int64_t rows;  // rows per chunk (a multiple of 32)
  int chunks;
};

int64_t lora_chunk_rows(int64_t T, int64_t K, int64_t N, int r);

hipError_t launch_lora_down(const LoraDownArgs& a, int w_kr, int dt, hipStream_t s, bool* sup);
hipError_t launch_lora_up(const LoraUpArgs& a, int dt, hipStream_t s, bool* sup);
hipError_t launch_lora_grads(const LoraGradArgs& a, int dt, hipStream_t s, bool* sup);

}  // namespace esep
