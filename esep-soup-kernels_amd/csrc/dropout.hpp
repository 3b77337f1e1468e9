// LoRA-dropout launch helpers (kernels in dropout.hip) and the mask generator its kernels share
// with the fused LoRA products (lora.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace esep {

hipError_t launch_dropout_fwd(const void* x, const int64_t* key, void* xd, int64_t n, float p,
                              int dt, hipStream_t s, bool* supported);
hipError_t launch_dropout_bwd(const void* x, const void* g, const int64_t* key, void* xd, void* dx,
                              int64_t n, float p, int accumulate, int dt, hipStream_t s,
                              bool* supported);

struct U4 {
  uint32_t w[4];
};

__device__ __forceinline__ U4 philox4x32_10(uint64_t ctr, uint32_t k0, uint32_t k1) {
  uint32_t c0 = (uint32_t)ctr, c1 = (uint32_t)(ctr >> 32), c2 = 0u, c3 = 0u;
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    if (r) {
      k0 += 0x9E3779B9u;
      k1 += 0xBB67AE85u;
    }
    // one 32 x 32 -> 64-bit product per multiplier (v_mad_u64_u32) instead of a low and a
    // high half (v_mul_lo_u32 + v_mul_hi_u32, each quarter rate)
    const uint64_t p0 = (uint64_t)0xD2511F53u * c0, p1 = (uint64_t)0xCD9E8D57u * c2;
    const uint32_t lo0 = (uint32_t)p0, hi0 = (uint32_t)(p0 >> 32);
    const uint32_t lo1 = (uint32_t)p1, hi1 = (uint32_t)(p1 >> 32);
    const uint32_t n0 = hi1 ^ c1 ^ k0, n2 = hi0 ^ c3 ^ k1;
    c0 = n0;
    c1 = lo1;
    c2 = n2;
    c3 = lo0;
  }
  return U4{{c0, c1, c2, c3}};
}

__device__ __forceinline__ bool keep_of(uint32_t word, float p) {
  return (float)(word >> 8) * 5.9604644775390625e-8f >= p;  // 2^-24
}

}  // namespace esep
