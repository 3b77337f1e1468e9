// The LoRA term's products on MFMA with the dropout mask regenerated inside them (the
// reference runs a dropout kernel and library products, solution/body/lora.py:140-245):
//
//   k_lora_down   xa = drop(x) A^T (forward), dxa = scaling * dterm B (backward)
//   k_lora_up     term = scaling * xa B^T, or added into the base projection's output
//   k_lora_grads  dx = (dxa A) * keep / (1 - p), dA = dxa^T drop(x), dB = scaling * dterm^T xa
//   k_lora_reduce the fixed-order sum of dA's and dB's partials
//
// Every product here has one side of at most 64 (the rank), so all are bound by streaming the
// [T, in] or [T, out] operand once (and, with dropout, by the ten Philox rounds per four
// elements). As separate passes the dropped input was written and read again in both
// directions and the library ran the products at 4-30 us each on 16-wide tiles: the q_proj term
// at T = 5933, 1536 -> 1536, r = 16, p = 0.05, fp16 took 145 us of kernels in 18 launches; here it
// takes 65 us in 8 (k_lora_down 13.6 us with dropout, of which the Philox rounds alone are about
// 8, and 8.4 us for dxa; k_lora_up 6.6; k_lora_grads 22; k_lora_reduce 4.6; key and casts 9). With
// 32 consecutive bytes per lane (16-byte accesses that leave half of every line to the next one)
// k_lora_up took 11.3 us.
//
// MFMA 16x16x32: A[i][k] in lane i + 16 (k / 8), element k % 8; B[k][j] in lane j + 16 (k / 8);
// D[i][j] in lane j + 16 (i / 4), element i % 4. A streamed row tile is 16 rows x 64 columns:
// lane (t = lane % 16, g = lane / 16) holds columns 8 g .. 8 g + 7 and 32 + 8 g .. of row t, so
// each 16-byte access of the wavefront covers 64 consecutive bytes of every row, and the two
// chunks are the k order of two MFMAs over the columns. Products whose result is such a tile
// compute it transposed, index i of tile m being column 32 (m / 2) + 8 (i / 4) + 4 (m % 2) + i % 4,
// so that a lane's results over m = 0..3 are its two chunks.
// Contractions over the rows read both operands transposed out of LDS (ds_read_b64_tr_b16:
// within a 16-lane group, lane j, slot k gets element j % 4 of the 8 bytes addressed by lane
// 4 k + j / 4).
#include <hip/hip_runtime.h>

#include <cstdint>

#include "common.hpp"
#include "dropout.hpp"
#include "lora.hpp"

namespace esep {
namespace {

template <typename T>
struct Mfma16;
template <>
struct Mfma16<__bf16> {
  typedef __bf16 v8 __attribute__((ext_vector_type(8)));
  static __device__ __forceinline__ f32x4 run(v8 a, v8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};
template <>
struct Mfma16<_Float16> {
  typedef _Float16 v8 __attribute__((ext_vector_type(8)));
  static __device__ __forceinline__ f32x4 run(v8 a, v8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

template <typename V>
__device__ __forceinline__ V ldv8(const void* p, bool ok) {
  return ok ? __builtin_bit_cast(V, *static_cast<const u32x4*>(p)) : V{};
}
// a tensor that the kernel reads once
template <typename V>
__device__ __forceinline__ V ldv8_nt(const void* p, bool ok) {
  return ok ? __builtin_bit_cast(V, __builtin_nontemporal_load(static_cast<const u32x4*>(p))) : V{};
}

typedef short s16x4l __attribute__((ext_vector_type(4)));

// Eight rows k0 .. k0 + 7 of one column per lane out of a row-major LDS matrix of pitch `pitch`
// elements: lane j of its 16-lane group gets column cseg(j / 4) + j % 4, where this lane (4 k +
// m) passes `p` = the address of row k0 + k, column cseg(m).
template <typename V, typename T>
__device__ __forceinline__ V ld_tr8(const T* p, int pitch) {
  typedef __attribute__((address_space(3))) s16x4l* lds_ptr;
  T* q = const_cast<T*>(p);
  const s16x4l lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(q));
  const s16x4l up = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(q + 4 * pitch));
  return __builtin_bit_cast(V, __builtin_shufflevector(lo, up, 0, 1, 2, 3, 4, 5, 6, 7));
}

// v * keep / (1 - p) of the 8 elements at `e` (a multiple of 4), rounded to T
template <typename T>
__device__ __forceinline__ void keep_mask8(int64_t e, uint32_t k0, uint32_t k1, float p,
                                           bool (&k)[8]) {
  const U4 a = philox4x32_10((uint64_t)(e / 4), k0, k1);
  const U4 b = philox4x32_10((uint64_t)(e / 4 + 1), k0, k1);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    k[i] = keep_of(a.w[i], p);
    k[4 + i] = keep_of(b.w[i], p);
  }
}

constexpr int kDownWaves = 8;

// A block owns 16 RT rows and all of K, its 8 wavefronts taking 64-column steps in turn; the
// partial sums meet in LDS and are added in wavefront order. RT grows with the rank (launch):
// every block reads all of W, r / (16 RT) of its x bytes.
template <typename T, int NR, int RT, bool WKR, bool DROP>
__global__ __launch_bounds__(64 * kDownWaves) void k_lora_down(const LoraDownArgs a) {
  using V8 = typename Mfma16<T>::v8;
  constexpr int WP = 16 * NR + 8;  // pitch of a wavefront's [64][16 NR] slice of W (WKR)
  constexpr int RP = 16 * RT + 4;  // pitch of the partial sums [16 NR][16 RT]
  constexpr int kStage = WKR ? 64 * WP * 2 : 0, kRed = 16 * NR * RP * 4;
  constexpr int kBytes = kDownWaves * (kStage > kRed ? kStage : kRed);
  __shared__ __align__(16) char sm[kBytes];
  const int lane = threadIdx.x & 63, w = wave_id();
  const int t = lane & 15, g = lane >> 4;
  const int64_t row0 = (int64_t)blockIdx.x * (16 * RT);
  const int r = a.r;
  uint32_t k0 = 0, k1 = 0;
  if constexpr (DROP) {
    const uint64_t kk = (uint64_t)*a.key;
    k0 = (uint32_t)kk;
    k1 = (uint32_t)(kk >> 32);
  }
  const T* W = static_cast<const T*>(a.w);
  T* stage = reinterpret_cast<T*>(sm) + (kStage / 2) * w;
  f32x4 acc[RT][NR];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int q = 0; q < NR; ++q) acc[i][q] = f32x4{0.f, 0.f, 0.f, 0.f};

  V8 xv[RT][2];
  auto load = [&](int64_t c) {  // columns c .. c + 63 of the block's rows
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const int64_t row = row0 + 16 * i + t;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int64_t col = c + 32 * h + 8 * g;
        xv[i][h] = ldv8<V8>(static_cast<const T*>(a.x) + row * a.ld_x + col,
                            row < a.T && col < a.K);
      }
    }
  };
  int64_t c = 64 * w;
  if (c < a.K) load(c);
  for (; c < a.K; c += 64 * kDownWaves) {
    V8 wv[2][NR];
    if constexpr (WKR) {
      constexpr int kChunks = 2 * NR;  // 16-byte chunks per row of the slice
#pragma unroll
      for (int j = 0; j < kChunks; ++j) {
        const int idx = lane + 64 * j, row = idx / kChunks, ch = idx % kChunks;
        const V8 v = ldv8<V8>(W + (c + row) * r + 8 * ch, c + row < a.K && 8 * ch < r);
        *reinterpret_cast<u32x4*>(stage + row * WP + 8 * ch) = __builtin_bit_cast(u32x4, v);
      }
      wave_lds_sync();
      const T* p = stage + (8 * g + ((lane >> 2) & 3)) * WP + 4 * (lane & 3);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int q = 0; q < NR; ++q) wv[h][q] = ld_tr8<V8>(p + 32 * h * WP + 16 * q, WP);
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int q = 0; q < NR; ++q) {
          const int64_t col = c + 32 * h + 8 * g;
          const int row = 16 * q + t;
          wv[h][q] = ldv8<V8>(W + (int64_t)row * a.K + col, row < r && col < a.K);
        }
    }
    V8 cur[RT][2];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) cur[i][h] = xv[i][h];
    if (c + 64 * kDownWaves < a.K) load(c + 64 * kDownWaves);
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if constexpr (DROP) {
          bool k[8];
          keep_mask8<T>((row0 + 16 * i + t) * a.K + c + 32 * h + 8 * g, k0, k1, a.p, k);
#pragma unroll
          for (int e = 0; e < 8; ++e)
            cur[i][h][e] = k[e] ? Elt<T>::from_f(Elt<T>::to_f(cur[i][h][e]) * a.inv_keep) : (T)0.f;
        }
#pragma unroll
        for (int q = 0; q < NR; ++q) acc[i][q] = Mfma16<T>::run(wv[h][q], cur[i][h], acc[i][q]);
      }
    if constexpr (WKR) wave_lds_sync();
  }
  // acc[i][q] element e is rank 16 q + 4 g + e of row 16 i + t
  __syncthreads();
  float* red = reinterpret_cast<float*>(sm);
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int q = 0; q < NR; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        red[(w * 16 * NR + 16 * q + 4 * g + e) * RP + 16 * i + t] = acc[i][q][e];
  __syncthreads();
  for (int idx = threadIdx.x; idx < 16 * RT * r; idx += 64 * kDownWaves) {
    const int row = idx / r, rank = idx % r;
    float s = 0.f;
#pragma unroll
    for (int v = 0; v < kDownWaves; ++v) s += red[(v * 16 * NR + rank) * RP + row];
    if (row0 + row < a.T)
      static_cast<T*>(a.out)[(row0 + row) * r + rank] = Elt<T>::from_f(s * a.scale);
  }
}

constexpr int kUpRows = 64;  // rows per k_lora_up block

// A wavefront owns 64 columns (B's operands stay in registers) and walks the block's rows 16 at
// a time; bound by the [T, N] store (and the base's read).
template <typename T, int NR>
__global__ __launch_bounds__(256) void k_lora_up(const LoraUpArgs a) {
  using V8 = typename Mfma16<T>::v8;
  constexpr int KR = (NR + 1) / 2;
  const int lane = threadIdx.x & 63, w = wave_id();
  const int t = lane & 15, g = lane >> 4;
  const int64_t n0 = (int64_t)blockIdx.x * 256 + 64 * w;
  if (n0 >= a.N) return;
  V8 bv[4][KR];
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int k = 0; k < KR; ++k) {
      const int64_t n = n0 + 32 * (m / 2) + 8 * (t >> 2) + 4 * (m % 2) + (t & 3);
      const int rank = 32 * k + 8 * g;
      bv[m][k] = ldv8<V8>(static_cast<const T*>(a.b) + n * a.r + rank, n < a.N && rank < a.r);
    }
  const int64_t r1 = (int64_t)(blockIdx.y + 1) * kUpRows < a.T ? (int64_t)(blockIdx.y + 1) * kUpRows
                                                               : a.T;
  for (int64_t row0 = (int64_t)blockIdx.y * kUpRows; row0 < r1; row0 += 16) {
    const int64_t row = row0 + t;
    V8 xv[KR];
#pragma unroll
    for (int k = 0; k < KR; ++k) {
      const int rank = 32 * k + 8 * g;
      xv[k] = ldv8<V8>(static_cast<const T*>(a.xa) + row * a.r + rank, row < a.T && rank < a.r);
    }
    V8 o[2];
    const int64_t n = n0 + 8 * g;
    if (a.base != nullptr) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
        o[h] = ldv8_nt<V8>(static_cast<const T*>(a.base) + row * a.ld_base + n + 32 * h,
                           row < a.T && n + 32 * h < a.N);
    } else {
      o[0] = o[1] = V8{};
    }
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < KR; ++k) acc = Mfma16<T>::run(bv[m][k], xv[k], acc);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int h = m / 2, i = 4 * (m % 2) + e;
        o[h][i] = Elt<T>::from_f(fmaf(acc[e], a.scale, Elt<T>::to_f(o[h][i])));
      }
    }
    if (row < a.T) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
        if (n + 32 * h < a.N)
          __builtin_nontemporal_store(
              __builtin_bit_cast(u32x4, o[h]),
              reinterpret_cast<u32x4*>(static_cast<T*>(a.out) + row * a.ld_out + n + 32 * h));
    }
  }
}

// One wavefront's part of k_lora_grads: 64 columns of x (DX: with dx) or of dterm, the rows of
// one chunk 32 at a time. Everything it shares through LDS stays within the wavefront.
template <typename T, int NR, bool DA, bool DROP>
__device__ __forceinline__ void grads_wave(const LoraGradArgs& a, int64_t c0, int chunk, T* xs,
                                           T* vs) {
  using V8 = typename Mfma16<T>::v8;
  constexpr int KR = (NR + 1) / 2;
  constexpr int XP = 64 + 8;        // pitch of the column tile [32][64]
  constexpr int VP = 32 * KR + 8;   // pitch of the rank tile [32][32 KR]
  const int lane = threadIdx.x & 63;
  const int t = lane & 15, g = lane >> 4, k4 = (lane >> 2) & 3, m4 = lane & 3;
  const int r = a.r;
  const int64_t C = DA ? a.K : a.N;
  const T* M = static_cast<const T*>(DA ? a.x : a.dterm);
  const int64_t ld = DA ? a.K : a.ld_dterm;
  const T* V = static_cast<const T*>(DA ? a.dxa : a.xa);
  uint32_t k0 = 0, k1 = 0;
  if constexpr (DROP) {
    const uint64_t kk = (uint64_t)*a.key;
    k0 = (uint32_t)kk;
    k1 = (uint32_t)(kk >> 32);
  }
  // A^T as the A operand of dx^T: lane i holds ranks 32 k + 8 g .. + 7 of its column of tile m.
  // A's 64 columns pass through the column tile 32 ranks at a time.
  V8 at[4][KR];
  if (DA && a.dx != nullptr) {
#pragma unroll
    for (int k = 0; k < KR; ++k) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int rank = 32 * k + 8 * j + (lane >> 3);
        const int64_t col = c0 + 8 * (lane & 7);
        const V8 v = ldv8<V8>(static_cast<const T*>(a.a) + (int64_t)rank * a.K + col,
                              rank < r && col < C);
        *reinterpret_cast<u32x4*>(xs + (8 * j + (lane >> 3)) * XP + 8 * (lane & 7)) =
            __builtin_bit_cast(u32x4, v);
      }
      wave_lds_sync();
#pragma unroll
      for (int m = 0; m < 4; ++m)
        at[m][k] = ld_tr8<V8>(xs + (8 * g + k4) * XP + 32 * (m / 2) + 8 * m4 + 4 * (m % 2), XP);
      wave_lds_sync();
    }
  }
  f32x4 acc[4][NR];
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int q = 0; q < NR; ++q) acc[m][q] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int64_t rbeg = (int64_t)chunk * a.rows;
  const int64_t rend = rbeg + a.rows < a.T ? rbeg + a.rows : a.T;

  V8 xv[2][2], vv[2 * KR];
  auto load = [&](int64_t row0) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int64_t row = row0 + 16 * s + t, col = c0 + 32 * h + 8 * g;
        xv[s][h] = ldv8_nt<V8>(M + row * ld + col, row < rend && col < C);
      }
#pragma unroll
    for (int j = 0; j < 2 * KR; ++j) {  // [32][32 KR] of the rank side, zero past r and rend
      const int idx = lane + 64 * j, row = idx / (4 * KR), ch = idx % (4 * KR);
      vv[j] = ldv8<V8>(V + (row0 + row) * r + 8 * ch, row0 + row < rend && 8 * ch < r);
    }
  };
  if (rbeg < rend) load(rbeg);
  for (int64_t row0 = rbeg; row0 < rend; row0 += 32) {
    V8 cur[2][2];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int h = 0; h < 2; ++h) cur[s][h] = xv[s][h];
#pragma unroll
    for (int j = 0; j < 2 * KR; ++j) {
      const int idx = lane + 64 * j, row = idx / (4 * KR), ch = idx % (4 * KR);
      *reinterpret_cast<u32x4*>(vs + row * VP + 8 * ch) = __builtin_bit_cast(u32x4, vv[j]);
    }
    if (row0 + 32 < rend) load(row0 + 32);
    wave_lds_sync();
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int64_t row = row0 + 16 * s + t, col = c0 + 8 * g;
      bool keep[2][8];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if constexpr (DROP) {
          keep_mask8<T>(row * C + col + 32 * h, k0, k1, a.p, keep[h]);
#pragma unroll
          for (int e = 0; e < 8; ++e)
            cur[s][h][e] =
                keep[h][e] ? Elt<T>::from_f(Elt<T>::to_f(cur[s][h][e]) * a.inv_keep) : (T)0.f;
        }
        *reinterpret_cast<u32x4*>(xs + (16 * s + t) * XP + 32 * h + 8 * g) =
            __builtin_bit_cast(u32x4, cur[s][h]);
      }
      if (DA && a.dx != nullptr) {
        V8 o[2] = {V8{}, V8{}};
        T* dst = static_cast<T*>(a.dx) + row * C + col;
        if (a.accumulate) {
#pragma unroll
          for (int h = 0; h < 2; ++h)
            o[h] = ldv8_nt<V8>(dst + 32 * h, row < rend && col + 32 * h < C);
        }
        V8 dv[KR];
#pragma unroll
        for (int k = 0; k < KR; ++k)
          dv[k] = __builtin_bit_cast(
              V8, *reinterpret_cast<const u32x4*>(vs + (16 * s + t) * VP + 32 * k + 8 * g));
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          f32x4 d = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int k = 0; k < KR; ++k) d = Mfma16<T>::run(at[m][k], dv[k], d);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int h = m / 2, i = 4 * (m % 2) + e;
            float v = d[e];
            if constexpr (DROP) v = keep[h][i] ? v * a.inv_keep : 0.f;
            o[h][i] = Elt<T>::from_f(Elt<T>::to_f(o[h][i]) + v);
          }
        }
        if (row < rend) {
#pragma unroll
          for (int h = 0; h < 2; ++h)
            if (col + 32 * h < C)
              __builtin_nontemporal_store(__builtin_bit_cast(u32x4, o[h]),
                                          reinterpret_cast<u32x4*>(dst + 32 * h));
        }
      }
    }
    wave_lds_sync();
    V8 vt[NR];
#pragma unroll
    for (int q = 0; q < NR; ++q) vt[q] = ld_tr8<V8>(vs + (8 * g + k4) * VP + 16 * q + 4 * m4, VP);
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const V8 xt = ld_tr8<V8>(xs + (8 * g + k4) * XP + 16 * m + 4 * m4, XP);
#pragma unroll
      for (int q = 0; q < NR; ++q)  // dA: columns x ranks; dB: ranks x columns
        acc[m][q] = DA ? Mfma16<T>::run(xt, vt[q], acc[m][q]) : Mfma16<T>::run(vt[q], xt, acc[m][q]);
    }
    wave_lds_sync();
  }
  float* part = a.part;
  if (DA) {
    part += (int64_t)chunk * r * a.K;  // [r][K]: four consecutive columns of one rank
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int q = 0; q < NR; ++q) {
        const int rank = 16 * q + t;
        const int64_t col = c0 + 16 * m + 4 * g;
        if (rank < r && col < C) *reinterpret_cast<f32x4*>(part + rank * a.K + col) = acc[m][q];
      }
  } else {
    if (a.x != nullptr) part += (int64_t)a.chunks * r * a.K;
    part += (int64_t)chunk * r * a.N;  // [N][r]: four consecutive ranks of one column
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int q = 0; q < NR; ++q) {
        const int64_t col = c0 + 16 * m + t;
        const int rank = 16 * q + 4 * g;
        if (rank < r && col < C) *reinterpret_cast<f32x4*>(part + col * r + rank) = acc[m][q];
      }
  }
}

// Blocks of 4 wavefronts x 64 columns: first the column groups of x (cgx of them), then those of
// dterm, times the row chunks. dx and dA take x's mask and dA's operand from one read of x.
template <typename T, int NR, bool DROP>
__global__ __launch_bounds__(256) void k_lora_grads(const LoraGradArgs a, int cgx) {
  constexpr int KR = (NR + 1) / 2;
  __shared__ __align__(16) T xs[4][32 * (64 + 8)];
  __shared__ __align__(16) T vs[4][32 * (32 * KR + 8)];
  const int w = wave_id(), cg = blockIdx.x, chunk = blockIdx.y;
  if (cg < cgx) {
    const int64_t c0 = 256 * (int64_t)cg + 64 * w;
    if (c0 < a.K) grads_wave<T, NR, true, DROP>(a, c0, chunk, xs[w], vs[w]);
  } else {
    const int64_t c0 = 256 * (int64_t)(cg - cgx) + 64 * w;
    if (c0 < a.N) grads_wave<T, NR, false, false>(a, c0, chunk, xs[w], vs[w]);
  }
}

// Sums the chunks' partials: four threads per 4 elements, each a quarter of the chunks, added in
// order.
__global__ __launch_bounds__(256) void k_lora_reduce(const float* part, int chunks, int64_t na,
                                                     int64_t nb, float scale, float* da,
                                                     float* db) {
  __shared__ f32x4 sm[4][64];
  const int64_t quad = (int64_t)blockIdx.x * 64 + (threadIdx.x & 63);
  const int s = threadIdx.x >> 6;
  const int64_t e = 4 * quad;
  const bool first = e < na, live = e < na + nb;
  const float* src = first ? part + e : part + (int64_t)chunks * na + (e - na);
  const int64_t step = first ? na : nb;
  const int per = (chunks + 3) / 4, c1 = per * (s + 1) < chunks ? per * (s + 1) : chunks;
  f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
  if (live) {
#pragma unroll 8
    for (int c = per * s; c < c1; ++c) v += *reinterpret_cast<const f32x4*>(src + c * step);
  }
  sm[s][threadIdx.x & 63] = v;
  __syncthreads();
  if (s == 0 && live) {
    const int l = threadIdx.x & 63;
    v = (sm[0][l] + sm[1][l]) + (sm[2][l] + sm[3][l]);
    if (first)
      *reinterpret_cast<f32x4*>(da + e) = v;
    else
      *reinterpret_cast<f32x4*>(db + (e - na)) = v * scale;
  }
}

template <typename T, int NR, int RT>
hipError_t down_run(const LoraDownArgs& a, int w_kr, hipStream_t s) {
  const dim3 grid((unsigned)((a.T + 16 * RT - 1) / (16 * RT))), block(64 * kDownWaves);
  if (w_kr)  // the backward's product: no dropout on dterm
    hipLaunchKernelGGL((k_lora_down<T, NR, RT, true, false>), grid, block, 0, s, a);
  else if (a.key != nullptr)
    hipLaunchKernelGGL((k_lora_down<T, NR, RT, false, true>), grid, block, 0, s, a);
  else
    hipLaunchKernelGGL((k_lora_down<T, NR, RT, false, false>), grid, block, 0, s, a);
  return hipGetLastError();
}

// Rows per block: as many 16-row tiles as rank tiles (W's reads then equal x's), as long as that
// leaves a block for every CU.
template <typename T, int NR>
hipError_t down_nr(const LoraDownArgs& a, int w_kr, hipStream_t s) {
  if constexpr (NR >= 4)
    if (a.T >= 64 * 256) return down_run<T, NR, 4>(a, w_kr, s);
  if constexpr (NR >= 2)
    if (a.T >= 32 * 256) return down_run<T, NR, 2>(a, w_kr, s);
  return down_run<T, NR, 1>(a, w_kr, s);
}

template <typename T, int NR>
hipError_t grads_nr(const LoraGradArgs& a, hipStream_t s) {
  const int cgx = a.x != nullptr ? (int)((a.K + 255) / 256) : 0;
  const int cgn = a.dterm != nullptr ? (int)((a.N + 255) / 256) : 0;
  const dim3 grid(cgx + cgn, a.chunks);
  if (a.key != nullptr)
    hipLaunchKernelGGL((k_lora_grads<T, NR, true>), grid, dim3(256), 0, s, a, cgx);
  else
    hipLaunchKernelGGL((k_lora_grads<T, NR, false>), grid, dim3(256), 0, s, a, cgx);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int64_t na = a.x != nullptr ? (int64_t)a.r * a.K : 0;
  const int64_t nb = a.dterm != nullptr ? (int64_t)a.r * a.N : 0;
  hipLaunchKernelGGL(k_lora_reduce, dim3((unsigned)((na + nb + 255) / 256)), dim3(256), 0, s,
                     a.part, a.chunks, na, nb, a.scale, a.da, a.db);
  return hipGetLastError();
}

// f(rank tiles of 16 as a constant)
template <typename F>
hipError_t by_rank(int r, F f) {
  if (r <= 16) return f(std::integral_constant<int, 1>{});
  if (r <= 32) return f(std::integral_constant<int, 2>{});
  return f(std::integral_constant<int, 4>{});
}

template <typename F>
hipError_t by_type(int dt, bool* sup, F f) {
  *sup = true;
  if (dt == 1) return f(_Float16{});
  if (dt == 2) return f(__bf16{});
  *sup = false;
  return hipErrorInvalidValue;
}

}  // namespace

// Rows per chunk of k_lora_grads: about 768 blocks (three per CU), but at least 2 r rows, which
// keeps the fp32 partials within the bytes of the operand they sum over, and at most 65535
// chunks (the grid's y limit).
int64_t lora_chunk_rows(int64_t T, int64_t K, int64_t N, int r) {
  const int64_t groups = (K + 255) / 256 + (N + 255) / 256;
  const int64_t chunks = 768 / groups > 0 ? 768 / groups : 1;
  int64_t rows = (T + chunks - 1) / chunks;
  if (rows < 2 * r) rows = 2 * r;
  if (rows < (T + 65534) / 65535) rows = (T + 65534) / 65535;
  return (rows + 31) / 32 * 32;
}

hipError_t launch_lora_down(const LoraDownArgs& a, int w_kr, int dt, hipStream_t s, bool* sup) {
  return by_type(dt, sup, [&](auto tag) {
    return by_rank(a.r, [&](auto nr) { return down_nr<decltype(tag), decltype(nr)::value>(a, w_kr, s); });
  });
}

hipError_t launch_lora_up(const LoraUpArgs& a, int dt, hipStream_t s, bool* sup) {
  return by_type(dt, sup, [&](auto tag) {
    return by_rank(a.r, [&](auto nr) {
      using T = decltype(tag);
      constexpr int NR = decltype(nr)::value;
      const dim3 grid((unsigned)((a.N + 255) / 256), (unsigned)((a.T + kUpRows - 1) / kUpRows));
      hipLaunchKernelGGL((k_lora_up<T, NR>), grid, dim3(256), 0, s, a);
      return hipGetLastError();
    });
  });
}

hipError_t launch_lora_grads(const LoraGradArgs& a, int dt, hipStream_t s, bool* sup) {
  return by_type(dt, sup, [&](auto tag) {
    return by_rank(a.r, [&](auto nr) { return grads_nr<decltype(tag), decltype(nr)::value>(a, s); });
  });
}

}  // namespace esep
