// NF4 (double-quant) weight dequantization for gfx950. Restates the reference's kernel
// (solution/nf4/dequant.py:35-57, nf4_dequant_kernel; the QLoRA / bitsandbytes Linear4bit format
// of its docstring, dequant.py:1-22):
//   scale[b] = fp32(fp32(code2[absmax[b]] * absmax2[b / 256]) + offset)
//   W[e]     = round(fp32(nf4[nibble(e)] * scale[e / 64]))     element 2i: high nibble of byte i
// Every step is rounded separately (contraction into fused multiply-adds is switched off in the
// kernel), which is what makes the result bit-exact with the format's reference decoder.
//
// Bound by bytes: 0.5 read and 2 (fp32: 4) written per element. A thread decodes units of 4 packed
// bytes (8 elements), consecutive threads consecutive units, so that a wavefront's loads (256
// bytes) and its 16-byte stores (1 KiB) are each one contiguous run, and takes several units 256
// apart, all requested before any is decoded. The 16-entry NF4 tables sit in LDS. 16 elements per
// thread left every store of a wavefront a stride of 32 bytes (fp32: 64) apart. Before -> now in us:
// 17920 x 1536 in fp32 86 -> 35 by k_nf4_dequant_one; in fp16 20 -> 19.5 by it, two weights of half that size
// 19.7 -> 18 by k_nf4_dequant_multi (69 MB: 3.8 TB/s). Stores: see kNf4Stream.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "common.hpp"
#include "nf4.hpp"

namespace esep {
namespace {

constexpr int kNf4Threads = 256;
// Units from which a block of k_nf4_dequant_multi takes 4 runs of units instead of 2: 1024 blocks,
// 4 per CU. Below, fewer blocks leave CUs idle (2 runs against 4 in us: 5.6 / 6.9 at 295 k units,
// 7.4 / 8.3 at 688 k; 14.4 / 12.1 at 1.7 M, 26.8 / 23.2 at 3.4 M).
constexpr int64_t kNf4Wide = 1 << 20;

// Output bytes of 16-bit types from which the stores go past the caches (non-temporal). Below, the GEMM
// that reads the weight next finds it there: decode + product of 256 rows, plain / non-temporal in us,
// 32 / 36 at 28 MiB, 60 / 68 at 84, 88 / 96 at 168 MiB (the decode alone 8.7 / 6.5, 21 / 16, 36 / 35). What
// the 256 MiB Infinity Cache cannot hold is written back all the same: 147 / 118 at 224 MiB (alone
// 77 / 45), 175 / 146 at 259, 355 / 315 at 518 MiB; at 4096 rows within 2% either way. In fp32 the plain
// stores are the faster ones at every size (168 MiB 36 / 69, 1036 MiB 311 / 416).
constexpr int64_t kNf4Stream = int64_t{192} << 20;

// Decode one unit (4 packed bytes, 8 elements, low byte first) with its block's scale into o;
// tab = the weight's NF4 table (LDS).
template <typename TO, bool NT>
__device__ __forceinline__ void nf4_decode(uint32_t raw, float scale, const float* tab,
                                           TO* __restrict__ o) {
#pragma clang fp contract(off)
  float v[8];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t byte = (raw >> (8 * j)) & 0xffu;
    v[2 * j] = tab[byte >> 4] * scale;
    v[2 * j + 1] = tab[byte & 15u] * scale;
  }
  if constexpr (sizeof(TO) == 2) {
    typedef TO v8t __attribute__((ext_vector_type(8)));
    v8t e;
#pragma unroll
    for (int k = 0; k < 8; ++k) e[k] = Elt<TO>::from_f(v[k]);
    if constexpr (NT)
      __builtin_nontemporal_store(__builtin_bit_cast(u32x4, e), reinterpret_cast<u32x4*>(o));
    else
      *reinterpret_cast<v8t*>(o) = e;
  } else {
#pragma unroll
    for (int h = 0; h < 2; ++h)
      reinterpret_cast<f32x4*>(o)[h] = f32x4{v[4 * h], v[4 * h + 1], v[4 * h + 2], v[4 * h + 3]};
  }
}

// Scale of block b: two roundings (without the pragma the compiler contracts the multiply and
// the add into one fused multiply-add, one rounding, which differs from the format's decoder;
// HIP's __fmul_rn is a plain multiply in a header, outside this pragma, and does not prevent
// it).
__device__ __forceinline__ float nf4_scale(const uint8_t* __restrict__ absmax,
                                           const float* __restrict__ absmax2,
                                           const float* __restrict__ code2, float off, int64_t b) {
#pragma clang fp contract(off)
  const float prod = code2[absmax[b]] * absmax2[b >> 8];
  return prod + off;
}

// A grid dimension counts its threads in 32 bits, silently: of 2^24 blocks and more only the
// remainder would run. Grids past kNf4Fold blocks have rows of that many.
constexpr int64_t kNf4Fold = 1 << 22;
__device__ __forceinline__ int64_t nf4_block() {
  return (int64_t)blockIdx.y * gridDim.x + blockIdx.x;
}

// Several weights, their units laid end to end (weight w: units [u0[w], u0[w + 1]), whole scale
// blocks). A block takes U runs of 256 units. While the packed bytes are on their way, one thread per
// scale block resolves its scale (absmax -> code2 is a dependent pair of loads) into LDS, so the
// search for the weight and that chain are paid once per 8 units.
template <typename TO, int U, bool NT>
__global__ __launch_bounds__(kNf4Threads) void k_nf4_dequant_multi(const Nf4Multi m) {
  constexpr int kScales = kNf4Threads * U / 8;
  __shared__ float tab[kNf4MultiMax][16];
  __shared__ float scl[kScales];
  const int tid = threadIdx.x;
  const int64_t g0 = nf4_block() * (kNf4Threads * U);
  const int64_t total = m.u0[m.n];
  auto weight_of = [&](int64_t u) {
    int wi = 0;
#pragma unroll
    for (int k = 1; k < kNf4MultiMax; ++k)
      if (k < m.n && u >= m.u0[k]) wi = k;
    return wi;
  };
  uint32_t raw[U];
  int wi[U];
#pragma unroll
  for (int t = 0; t < U; ++t) {
    const int64_t g = g0 + t * kNf4Threads + tid;
    wi[t] = g < total ? weight_of(g) : 0;
    raw[t] = g < total ? static_cast<const uint32_t*>(m.w[wi[t]].packed)[g - m.u0[wi[t]]] : 0u;
  }
  if (tid < 16 * m.n) tab[tid >> 4][tid & 15] = m.w[tid >> 4].nf4[tid & 15];
  if (tid < kScales) {
    const int64_t gs = g0 + 8 * tid;  // first unit of this scale block
    if (gs < total) {
      const int ws = weight_of(gs);
      const Nf4Args& w = m.w[ws];
      scl[tid] = nf4_scale(w.absmax, w.absmax2, w.code2, *w.offset, (gs - m.u0[ws]) >> 3);
    }
  }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < U; ++t) {
    const int64_t g = g0 + t * kNf4Threads + tid;
    if (g < total)
      nf4_decode<TO, NT>(raw[t], scl[(t * kNf4Threads + tid) >> 3], tab[wi[t]],
                     static_cast<TO*>(m.w[wi[t]].out) + 8 * (g - m.u0[wi[t]]));
  }
}

// One weight: every thread reads its own scales (8 threads the same ones), no wait between them and the
// packed bytes: 5.2 us at 1536 x 1536 against 5.6 through LDS, 10.7 against 14.4 at 1536 x 8960. Two
// runs of units per block: four take 10.3 there but 5.8 at 1536 x 1536, one 12.5 and 5.2.
template <typename TO, int U, bool NT>
__global__ __launch_bounds__(kNf4Threads) void k_nf4_dequant_one(const Nf4Args w) {
  __shared__ float tab[16];
  const int tid = threadIdx.x;
  const int64_t g0 = nf4_block() * (kNf4Threads * U) + tid;
  const int64_t total = 8 * w.n_blocks;
  uint32_t raw[U];
  float scale[U];
  const float off = *w.offset;
#pragma unroll
  for (int t = 0; t < U; ++t) {
    const int64_t g = g0 + t * kNf4Threads;
    const bool live = g < total;
    raw[t] = live ? static_cast<const uint32_t*>(w.packed)[g] : 0u;
    scale[t] = live ? nf4_scale(w.absmax, w.absmax2, w.code2, off, g >> 3) : 0.f;
  }
  if (tid < 16) tab[tid] = w.nf4[tid];
  __syncthreads();
#pragma unroll
  for (int t = 0; t < U; ++t) {
    const int64_t g = g0 + t * kNf4Threads;
    if (g < total) nf4_decode<TO, NT>(raw[t], scale[t], tab, static_cast<TO*>(w.out) + 8 * g);
  }
}

template <typename TO, bool NT>
void launch_nt(const Nf4Multi& m, hipStream_t s) {
  const int64_t units = m.u0[m.n];
  auto grid = [&](int u) {
    const int64_t per = (int64_t)kNf4Threads * u, blocks = (units + per - 1) / per;
    return blocks <= kNf4Fold ? dim3((unsigned)blocks)
                              : dim3((unsigned)kNf4Fold, (unsigned)((blocks + kNf4Fold - 1) / kNf4Fold));
  };
  const dim3 block(kNf4Threads);
  if (m.n == 1)
    hipLaunchKernelGGL((k_nf4_dequant_one<TO, 2, NT>), grid(2), block, 0, s, m.w[0]);
  else if (units < kNf4Wide)
    hipLaunchKernelGGL((k_nf4_dequant_multi<TO, 2, NT>), grid(2), block, 0, s, m);
  else
    hipLaunchKernelGGL((k_nf4_dequant_multi<TO, 4, NT>), grid(4), block, 0, s, m);
}

template <typename TO>
void launch(const Nf4Multi& m, hipStream_t s) {
  if constexpr (sizeof(TO) == 2)
    if (m.u0[m.n] * 16 >= kNf4Stream) return launch_nt<TO, true>(m, s);  // 8 elements per unit
  launch_nt<TO, false>(m, s);
}

}  // namespace

hipError_t launch_nf4_dequant(const Nf4Multi& m, int out_dt, hipStream_t s, bool* sup) {
  *sup = true;
  if (m.u0[m.n] == 0) return hipSuccess;
  if (out_dt == 0)
    launch<float>(m, s);
  else if (out_dt == 1)
    launch<_Float16>(m, s);
  else if (out_dt == 2)
    launch<__bf16>(m, s);
  else {
    *sup = false;
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace esep
