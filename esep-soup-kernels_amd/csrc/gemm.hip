// C[M, N] = A[M, K] . B (+ bias) on MFMA for 16-bit operands with fp32 accumulation, B given as
// [N, K] (a weight as it is stored: the forward's x W^T) or as [K, N] (the same weight in the
// backward's dy W). Used where it beats hipBLASLt (gemm_pays): few output tiles under a long
// contraction, where the library leaves most CUs idle (fp16, 1031 x 1536 x 17920, B [K, N]:
// 199 us against 74 here on four splits of the contraction).
//
// A block of WM x WN wavefronts owns a tile of C, each wavefront 32 TM x 32 TN of it in fp32
// accumulators. A and B move in 64-deep tiles by dwordx4 LDS DMA through two buffers: rows of
// 128 bytes, chunk c of row r at position c ^ ((r >> 1) & 7), so that the 16 rows a 16-byte
// operand read touches in one pass lie in 16 different bank groups; B as [K, N] in rows of the
// tile's width, 32-byte unit u of row r at u ^ (r & 3), read with ds_read_b64_tr_b16. The 16-deep
// contraction steps are software-pipelined in registers: a step's MFMAs have the next step's
// operand reads between them, and the last step of a tile has the barrier, the refill of the
// buffer just consumed and the first reads of the next tile between its MFMAs (8192^3 with B
// [K, N]: 1193 -> 1253 TFLOP/s against reads and refills issued in blocks ahead of the MFMAs, same
// box; hipBLASLt 1113). A timing-only copy without the refills runs at 1455 TFLOP/s, one with every
// block on the same (L2-resident) tiles at 1270; MFMAs alone on random register data at 1720,
// the power limit. Four wavefronts of 128 x 128 instead of eight of 128 x 64: 1177.
//
// Outputs with fewer tiles than CUs split the contraction over blocks; the fp32 partial sums are
// added in split order by k_gemm_reduce.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "attention.hpp"
#include "common.hpp"
#include "gemm.hpp"

namespace esep {
namespace {

constexpr int kBK = 64;  // contraction depth of one LDS tile: 128-byte rows

// s_waitcnt vmcnt(0) lgkmcnt(0)
constexpr int kWaitVmLgkm0 = 0x0070;

// lds_dma_x4_s from any wavefront-uniform base, also one that the compiler holds in VGPRs.
__device__ __forceinline__ void lds_dma(const char* base, uint32_t voff, const void* lds) {
  const uint64_t v = reinterpret_cast<uint64_t>(base);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t up = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  lds_dma_x4_s(reinterpret_cast<const void*>(((uint64_t)up << 32) | lo), voff, lds);
}

template <int WM, int WN, int TM, int TN>
struct Shape {
  static constexpr int NW = WM * WN, NT = 64 * NW;
  static constexpr int BM = 32 * WM * TM, BN = 32 * WN * TN;
  static constexpr int ABYTES = BM * 128, BBYTES = BN * 128;
  static constexpr int AI = BM / 8 / NW, BI = BN / 8 / NW;  // DMA instructions per wavefront
  static_assert(AI >= 1 && BI >= 1, "one DMA instruction per wavefront at least");
};

template <typename T, typename O, bool KN, int WM, int WN, int TM, int TN>
__global__ __launch_bounds__(64 * WM * WN, 2) void k_gemm(const GemmArgs g) {
  using S = Shape<WM, WN, TM, TN>;
  using V8 = typename Mfma<T>::v8;
  constexpr int BUF = S::ABYTES + S::BBYTES;
  __shared__ __align__(1024) char sm[2 * BUF];  // [2][A tile | B tile]
  const int lane = threadIdx.x & 63;
  const int w = wave_id();
  const int wm = w / WN, wn = w % WN;
  const int lq = lane & 31, hi = lane >> 5;

  // tile of this block: XCD x takes a contiguous run of the tile list, which walks 4 row tiles by
  // all column tiles before the next 4 (the blocks of an XCD then share A and B rows in its L2)
  const int ntile = g.tiles_m * g.tiles_n;
  const int nblk = ntile * g.splits;
  int lin;
  {
    const int b = blockIdx.x, q = nblk / 8, r = nblk % 8, x = b % 8;
    lin = x * q + (x < r ? x : r) + b / 8;
  }
  const int split = lin / ntile;
  int tm, tn;
  {
    constexpr int G = 4;
    const int t = lin % ntile;
    const int per = G * g.tiles_n, grp = t / per, in = t % per;
    const int rows = g.tiles_m - grp * G < G ? g.tiles_m - grp * G : G;
    tm = grp * G + in % rows;
    tn = in / rows;
  }
  const int64_t m0 = (int64_t)tm * S::BM, n0 = (int64_t)tn * S::BN;
  const int total = (int)(g.K / kBK);
  const int s0 = split * g.steps;
  const int steps = total - s0 < g.steps ? total - s0 : g.steps;

  // DMA: instruction i of this wavefront fills 1 KiB: 8 rows of a 128-byte-row tile (chunk c of row
  // r at position c ^ ((r >> 1) & 7)); rows past the matrix repeat its last row
  const char* acur = static_cast<const char*>(g.a) + 2 * (int64_t)s0 * kBK;
  const char* bcur = static_cast<const char*>(g.b) +
                     (KN ? 2 * (int64_t)s0 * kBK * g.ldb : 2 * (int64_t)s0 * kBK);
  const int64_t bstep = KN ? 2 * (int64_t)kBK * g.ldb : 2 * kBK;
  uint32_t avo[S::AI], bvo[S::BI];
#pragma unroll
  for (int i = 0; i < S::AI; ++i) {
    const int r = 8 * (w + S::NW * i) + (lane >> 3);
    const int64_t row = m0 + r < g.M ? r : g.M - 1 - m0;
    avo[i] = (uint32_t)(2 * row * g.lda) + 16u * ((lane & 7) ^ ((r >> 1) & 7));
  }
  acur += 2 * m0 * g.lda;
  if constexpr (KN) {
    // [64][BN]: rows of 2 BN bytes, the 32-byte unit u of row r at position u ^ (r & 3)
    constexpr int CPR = S::BN / 8;  // chunks per row
    bcur += 2 * n0;
#pragma unroll
    for (int i = 0; i < S::BI; ++i) {
      const int idx = 64 * (w + S::NW * i) + lane, r = idx / CPR, pos = idx % CPR;
      int c = 2 * ((pos >> 1) ^ (r & 3)) + (pos & 1);
      if (n0 + 8 * c >= g.N) c = (int)((g.N - n0) / 8) - 1;
      bvo[i] = (uint32_t)(2 * (int64_t)r * g.ldb) + 16u * c;
    }
  } else {
    bcur += 2 * n0 * g.ldb;
#pragma unroll
    for (int i = 0; i < S::BI; ++i) {
      const int r = 8 * (w + S::NW * i) + (lane >> 3);
      const int64_t row = n0 + r < g.N ? r : g.N - 1 - n0;
      bvo[i] = (uint32_t)(2 * row * g.ldb) + 16u * ((lane & 7) ^ ((r >> 1) & 7));
    }
  }
  // DMA instruction i of the next 64-deep tile (A's, then B's)
  auto issue1 = [&](int buf, int i) {
    char* d = sm + buf * BUF;
    if (i < S::AI)
      lds_dma(acur, avo[i], d + 1024 * (w + S::NW * i));
    else
      lds_dma(bcur, bvo[i - S::AI], d + S::ABYTES + 1024 * (w + S::NW * (i - S::AI)));
  };
  auto advance = [&] {
    acur += 2 * kBK;
    bcur += bstep;
  };
  auto issue = [&](int buf) {
#pragma unroll
    for (int i = 0; i < S::AI + S::BI; ++i) issue1(buf, i);
    advance();
  };

  // operand addresses of contraction step s (16 deep) of the tile: row operands at ro ^ 32 s
  // (+ 4096 per 32 rows); transposing ones at to[..] + 32 BN s
  const uint32_t sw = 16u * (hi ^ ((lq >> 1) & 7));
  const uint32_t aro = (uint32_t)((32 * TM * wm + lq) * 128) + sw;
  uint32_t bro = 0, bto[2] = {0, 0};
  if constexpr (KN) {
    const int k = (lane >> 2) & 3, m = lane & 3, G1 = (lane >> 4) & 1;
    static_assert(TN % 2 == 0, "two 32-column operands per 64-byte swizzle period");
#pragma unroll
    for (int u = 0; u < 2; ++u)
      bto[u] = (uint32_t)((8 * hi + k) * 2 * S::BN + 64 * TN * wn + 8 * m) + 32u * ((2 * u + G1) ^ k);
  } else {
    bro = (uint32_t)((32 * TN * wn + lq) * 128) + sw;
  }
  typedef __attribute__((address_space(3))) s16x4* lds_ptr;
  auto rd_a = [&](const char* tile, int s, int i) {
    return ld16<V8>(tile + ((aro ^ (32u * s)) + 4096u * i));
  };
  auto rd_b = [&](const char* tile, int s, int j) -> V8 {
    if constexpr (KN) {
      const char* p = tile + (bto[j & 1] + 128u * (j >> 1) + (uint32_t)(32 * S::BN) * s);
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(p));
      const s16x4 up = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(p + 8 * S::BN));
      return __builtin_bit_cast(V8, __builtin_shufflevector(lo, up, 0, 1, 2, 3, 4, 5, 6, 7));
    } else {
      return ld16<V8>(tile + ((bro ^ (32u * s)) + 4096u * j));
    }
  };

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x16{};
  V8 fa[2][TM], fb[2][TN];
  constexpr int NM = TM * TN, NR = TM + TN;  // MFMAs and operand reads of one contraction step
  auto rd1 = [&](int slot, const char* buf, int s, int i) {  // B's operands first
    if (i < TN)
      fb[slot][i] = rd_b(buf + S::ABYTES, s, i);
    else
      fa[slot][i - TN] = rd_a(buf, s, i - TN);
  };
  auto mma1 = [&](int slot, int i) {
    acc[i / TN][i % TN] = Mfma<T>::run(fb[slot][i % TN], fa[slot][i / TN], acc[i / TN][i % TN]);
  };

  issue(0);
  __builtin_amdgcn_s_waitcnt(kWaitVm0);
  __syncthreads();
  if (steps > 1) issue(1);
#pragma unroll
  for (int i = 0; i < NR; ++i) rd1(0, sm, 0, i);
  auto tile = [&](int t, auto bc) {
    constexpr int B = decltype(bc)::value;
    const char* cur = sm + B * BUF;
    const char* nxt = sm + (B ^ 1) * BUF;
    // a contraction step's MFMAs with the next step's operand reads between them
#pragma unroll
    for (int s = 0; s < 3; ++s) {
#pragma unroll
      for (int i = 0; i < (NM > NR ? NM : NR); ++i) {
        if (i < NM) mma1(s & 1, i);
        if (i < NR) rd1((s + 1) & 1, cur, s + 1, i);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // every operand of this tile is in registers and the next tile has landed: publish the one,
    // refill the other, all between the last step's MFMAs
    constexpr int PRE = 1;
    __builtin_amdgcn_s_waitcnt(kWaitVmLgkm0);
#pragma unroll
    for (int i = 0; i < PRE; ++i) mma1(1, i);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    const bool more = t + 2 < steps;
    constexpr int ND = S::AI + S::BI, REST = NM - PRE;
#pragma unroll
    for (int i = 0; i < REST; ++i) {
      mma1(1, PRE + i);
#pragma unroll
      for (int k = i * NR / REST; k < (i + 1) * NR / REST; ++k) rd1(0, nxt, 0, k);
      if (more) {
#pragma unroll
        for (int k = i * ND / REST; k < (i + 1) * ND / REST; ++k) issue1(B, k);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (more) advance();
  };
  int t = 0;
  for (; t + 1 < steps; t += 2) {
    tile(t, std::integral_constant<int, 0>{});
    tile(t + 1, std::integral_constant<int, 1>{});
  }
  if (t < steps) tile(t, std::integral_constant<int, 0>{});

  // Epilogue: acc[i][j] element 4 q + e of lane (lq, hi) is row m0 + 32 (TM wm + i) + lq, column
  // n0 + 32 (TN wn + j) + 8 q + 4 hi + e. Each wavefront turns its rows through LDS, 32 at a time,
  // into whole-line stores. (Every wavefront passed the last barrier after its last LDS read.)
  constexpr int CW = 32 * TN;
  auto flush = [&](auto tag, char* cbase, int64_t ldc) {
    using P = decltype(tag);
    constexpr int PITCH = CW * (int)sizeof(P) + 16;
    char* st = sm + w * (32 * PITCH);
    const int64_t col0 = n0 + CW * wn;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = acc[i][j][4 * q + e];
          if constexpr (sizeof(P) == 2) {
            if (g.bias != nullptr) {
              const int64_t n = col0 + 32 * j + 8 * q + 4 * hi;
              if (n < g.N) {
                const T* bp = static_cast<const T*>(g.bias) + n;
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] += (float)bp[e];
              }
            }
            P o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = (P)v[e];
            *reinterpret_cast<uint2*>(st + lq * PITCH + 2 * (32 * j + 8 * q + 4 * hi)) =
                __builtin_bit_cast(uint2, o);
          } else {
            *reinterpret_cast<f32x4*>(st + lq * PITCH + 4 * (32 * j + 8 * q + 4 * hi)) =
                f32x4{v[0], v[1], v[2], v[3]};
          }
        }
      wave_lds_sync();
      constexpr int LPR = CW * (int)sizeof(P) / 16;  // lanes per row
      constexpr int RPI = 64 / LPR;                  // rows per store instruction
      const int64_t row0 = m0 + 32 * (TM * wm + i);
#pragma unroll
      for (int k = 0; k < 32 / RPI; ++k) {
        const int r = RPI * k + lane / LPR, c = lane % LPR;
        const u32x4 v = *reinterpret_cast<const u32x4*>(st + r * PITCH + 16 * c);
        const int64_t col = col0 + (16 / (int)sizeof(P)) * c;
        if (row0 + r < g.M && col < g.N)
          *reinterpret_cast<u32x4*>(cbase + ((row0 + r) * ldc + col) * (int64_t)sizeof(P)) = v;
      }
      wave_lds_sync();
    }
  };
  if (g.splits > 1)
    flush(float{}, reinterpret_cast<char*>(g.part + (int64_t)split * g.M * g.N), g.N);
  else
    flush(O{}, static_cast<char*>(g.c), g.ldc);
}

// C = the splits' sum in order (+ bias); 8 columns per thread.
template <typename T, typename O>
__global__ __launch_bounds__(256) void k_gemm_reduce(const GemmArgs g) {
  const int64_t per = g.N / 8, e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= g.M * per) return;
  const int64_t m = e / per, n = 8 * (e % per);
  const float* p = g.part + m * g.N + n;
  const int64_t plane = g.M * g.N;
  float v[8];
  Chunk<float>::load(p, v);
  for (int s = 1; s < g.splits; ++s) {
    float u[8];
    Chunk<float>::load(p + s * plane, u);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] += u[i];
  }
  if constexpr (sizeof(O) == 2) {
    if (g.bias != nullptr) {
      float u[8];
      Chunk<T>::load(static_cast<const T*>(g.bias) + n, u);
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] += u[i];
    }
  }
  Chunk<O>::store(static_cast<O*>(g.c) + m * g.ldc + n, v);
}

template <typename T, typename O, bool KN, int WM, int WN, int TM, int TN>
hipError_t run(GemmArgs a, hipStream_t s) {
  using S = Shape<WM, WN, TM, TN>;
  a.tiles_m = (int)((a.M + S::BM - 1) / S::BM);
  a.tiles_n = (int)((a.N + S::BN - 1) / S::BN);
  const int total = (int)(a.K / kBK);
  if (a.splits > total) a.splits = total;
  a.steps = (total + a.splits - 1) / a.splits;
  a.splits = (total + a.steps - 1) / a.steps;
  static_assert(S::NW * 32 * (32 * TN * 4 + 16) <= 2 * (S::ABYTES + S::BBYTES), "epilogue");
  hipLaunchKernelGGL((k_gemm<T, O, KN, WM, WN, TM, TN>),
                     dim3((unsigned)(a.tiles_m * a.tiles_n * a.splits)), dim3(S::NT), 0, s, a);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || a.splits == 1) return e;
  hipLaunchKernelGGL((k_gemm_reduce<T, O>), dim3((unsigned)((a.M * (a.N / 8) + 255) / 256)),
                     dim3(256), 0, s, a);
  return hipGetLastError();
}

template <typename T, typename O, bool KN>
hipError_t by_shape(const GemmArgs& a, int shape, hipStream_t s) {
  if (shape == kGemm256x256) return run<T, O, KN, 2, 4, 4, 2>(a, s);
  if (shape == kGemm128x256) return run<T, O, KN, 2, 4, 2, 2>(a, s);
  if (shape == kGemm256x128) return run<T, O, KN, 4, 2, 2, 2>(a, s);
  if (shape == kGemm128x128) return run<T, O, KN, 2, 2, 2, 2>(a, s);
  return run<T, O, KN, 2, 2, 1, 2>(a, s);
}

}  // namespace

GemmPlan gemm_plan(int64_t M, int64_t N, int64_t K) {
  struct Cost {
    int bm, bn;
    double step, alone;  // us per 64-deep tile of a block: share of a full CU; a lone block's
  };
  // Fitted to fp16 measurements at M = 16 .. 8192 over the decoder's projection shapes. Blocks a
  // CU holds by LDS: 1, 1, 1, 2, 3.
  static constexpr Cost cost[] = {{256, 256, 1.60, 1.48},
                                  {128, 256, 0.95, 0.83},
                                  {256, 128, 0.97, 0.85},
                                  {128, 128, 0.51, 0.47},
                                  {64, 128, 0.29, 0.44}};
  const int total = (int)(K / kBK);
  GemmPlan best{0, 1, 1e30};
  for (int i = 0; i < 5; ++i) {
    const int64_t tiles = ((M + cost[i].bm - 1) / cost[i].bm) * ((N + cost[i].bn - 1) / cost[i].bn);
    for (int want = 1; want <= 24 && want <= total; ++want) {
      const int steps = (total + want - 1) / want, splits = (total + steps - 1) / steps;
      if (splits != want || (want > 1 && (steps < 6 || tiles * want > 768))) continue;
      if (want > 1 && M * N * want > (1 << 26)) continue;  // at most 256 MiB of partial sums
      const double per_cu = (double)((tiles * splits + 255) / 256);
      const double step = per_cu * cost[i].step > cost[i].alone ? per_cu * cost[i].step : cost[i].alone;
      double us = 4 + steps * step;
      // the partial sums written and read (largely in the Infinity Cache), and the second launch
      if (splits > 1) us += 3.5 + (double)M * N * (8.0 * splits + 2) / 1e7;
      if (us < best.us) best = GemmPlan{i, splits, us};
    }
  }
  return best;
}

// A table, placed by hand from 3660 products measured against hipBLASLt (torch.mm), M = 16 .. 8192 over
// the projections of fifteen decoder widths and vocabularies, fp16 and bf16 (alike within a few
// percent), launches back to back on warm operands. Ranges of t, the count of 256 x 256 output tiles,
// with the ratio here / library in them (geometric mean, worst) and, after the bar, outside:
//   B [K, N], where the library rarely splits the contraction: the longer it is, the wider the range
//     K >= 16384    t < 96           0.50, 1.09 (1031 x 1536 x 17920 199 us / 74) | 1.02 at the LM head's full
//                                    chunk (4096 x 1536 x 151936 1721 / 1764), 1.1 .. 1.25 past it
//     12288 ..      t <= 75          0.61, 0.92 | 1.06 .. 1.26
//     8192 ..       t <= 48, 64 .. 80  0.65, 1.11 | 1.06 .. 1.16 between, where the plan's unsplit 128-wide
//                                    tiles lose (2300 x 1536 x 8960 79 us / 91), 1.2 past 88
//     3328 ..       t = 1 .. 36      0.81, 1.12 | 1.1 .. 1.33 past 40
//     2049 ..       none             0.64 .. 1.30 without a pattern
//     1281 ..       t = 52 .. 72     0.89, 1.05 (3001 x 1536 x 1536 29 us / 24) | 1.04 .. 1.37 on either side
//     896 ..        t = 12 .. 64     0.82, 1.07 | up to 1.56 below, 1.26 above
//     up to 2048    t >= 250, M <= 4096, where the plan is whole 256 x 256 tiles: 0.97, 1.00 (3001 x 8960 x 1536 87
//                   us / 83) | the smaller tiles 0.80 .. 1.16 (3750 x 8960 x 1536 109 / 119)
//   B [N, K], which the library serves better
//     K >= 16384    t = 1 .. 95      0.56, 1.06
//     12288 ..      t = 4 .. 40      0.86, 1.05 | 1.1 .. 1.4
//     8192 ..       t = 4 .. 20      0.85, 1.06 | 1.05 .. 1.4
//     896 ..        the LM head's logits up to 32 rows 0.79, 0.98, and at 385 .. 512 (two full 256-row tiles)
//                   0.91, 0.98 | 300 rows 185 us / 240; 4096 x 256 x 1536 9 / 22, 512 x 2048 x 1536 9 / 18
// Of the 1030 measured products that it takes, 11 are more than 5% slower here.
bool gemm_pays(int64_t M, int64_t N, int64_t K, bool b_kn) {
  const double t = (double)M * N / 65536;
  if (b_kn) {
    if (K >= 16384) return t < 96;
    if (K >= 12288) return t <= 75;
    if (K >= 8192) return t <= 48 || (t >= 64 && t <= 80);
    if (K >= 3328) return t >= 1 && t <= 36;
    if (K > 2048 || K < 896) return false;  // below 896 not measured
    if (t >= 250 && M <= 4096) {
      const GemmPlan p = gemm_plan(M, N, K);
      return p.shape == kGemm256x256 && p.splits == 1;
    }
    return K > 1280 ? t >= 52 && t < 72 : t >= 12 && t <= 64;
  }
  if (K >= 16384) return t >= 1 && t < 96;
  if (K >= 12288) return t >= 4 && t <= 40;
  if (K >= 8192) return t >= 4 && t <= 20;
  return K >= 896 && ((M <= 32 && t >= 32) || (M > 384 && M <= 512 && t >= 800));
}

hipError_t launch_gemm(const GemmArgs& a, int shape, int b_kn, int dt, int out_dt, hipStream_t s,
                       bool* sup) {
  *sup = dt == 1 || dt == 2;
  if (!*sup) return hipErrorInvalidValue;
  auto go = [&](auto tag) {
    using T = decltype(tag);
    if (out_dt == 0)
      return b_kn ? by_shape<T, float, true>(a, shape, s) : by_shape<T, float, false>(a, shape, s);
    return b_kn ? by_shape<T, T, true>(a, shape, s) : by_shape<T, T, false>(a, shape, s);
  };
  return dt == 1 ? go(_Float16{}) : go(__bf16{});
}

}  // namespace esep
