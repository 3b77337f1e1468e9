// LM-head row kernel launch helper (kernel in head.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace esep {

struct HeadArgs {
  void* z;                // [rows, ld] logits chunk (fp16 / bf16); rows with g get overwritten
  const int64_t* target;  // [rows] vocabulary id; outside [0, V) = no target
  const float* cew;       // [rows] CE weight: pass 2 runs on rows where it is != 0
  float* lse;             // [rows] log-sum-exp
  float* tlogit;          // [rows] target logit (0 without a target)
  float* ent;             // [rows] entropy of softmax(z)
  int32_t* amax;          // [rows] first index of the row maximum
  int64_t rows, ld, V;
  float g_scale;
  int write_g;
  // with ce: [rows] lse - tlogit (0 without a target), the argmax in 64 bits instead of amax, and
  // pass 2 only on rows that have a target
  float* ce;
  int64_t* amax64;
  const int32_t* perm;  // null, or: row i of the chunk is row perm[i] of every [rows] array
};

// vec: z is 16-byte aligned and ld and V are multiples of 8 (whole 16-byte chunks).
hipError_t launch_head_row(const HeadArgs& a, int dt, bool vec, hipStream_t s, bool* supported);

// The rows with a target in [0, V) and cew != 0 first (stable), then the rest.
hipError_t launch_head_partition(const int64_t* target, const float* cew, int64_t N, int64_t V,
                                 int32_t* perm, int32_t* inv, int32_t* n_live, hipStream_t s);
// *loss = sum of cew * ce over the rows with a target in [0, V).
hipError_t launch_head_loss(const int64_t* target, const float* cew, const float* ce, int64_t N,
                            int64_t V, float* loss, hipStream_t s);
// dx[i] = prod[inv[i]] * (cew[i] * inv_scale) * *dloss where inv[i] < n_live, else 0 * *dloss.
hipError_t launch_head_dx(const float* prod, int64_t n_live, const int32_t* inv, const float* cew,
                          const float* dloss, float inv_scale, void* dx, int dx_dt, int64_t N,
                          int64_t H, hipStream_t s);

}  // namespace esep
