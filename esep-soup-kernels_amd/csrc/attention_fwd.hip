// Varlen causal attention forward (see attention.hpp for the layout and the MFMA mapping).
#include <cmath>
#include <type_traits>

#include "attention.hpp"

namespace esep {
namespace {

// 32 keys of the online softmax for a wavefront's 32 queries: keys kh .. kh + 31, held in 32 rows of
// the swizzled LDS tiles at ks / vs (the layout, its DMA and its readers are in attention.hpp).
// Lane (lq, hi) gets the scores of its query qi against keys kh + 8 (i / 4) + 4 hi + i % 4, i < 16,
// from S^T = K Q^T (K rows from LDS as the A operand, the wave's Q^T in registers as B), then
// updates (m, l) and O^T += V^T P^T, the contraction in the permuted key order of pb (element e of
// chunk c2 is key kh + 16 c2 + 8 (e / 4) + 4 hi + e % 4).
//
// Online softmax (base 2) with a lazy reference: the lane's m moves only when the 32 keys' maximum
// exceeds it by more than 8, so p <= 2^8 (exact in bf16 / fp16 relative terms) and O, l are
// rescaled only where some lane's m moved. Operands are read ahead of their MFMAs (K three, V^T two,
// the first V^T ones before the softmax, whose VALU work hides their latency), pinned by
// scheduling barriers: the compiler sinks each read to just before its use (config 5 forward
// 2.03 -> 1.93 ms).
template <typename T, int D>
__device__ __forceinline__ void fwd_tile_swz(const char* ks, const char* vs, int kh, int qw0,
                                             int qi, int lane, float scale_log2,
                                             const typename Mfma<T>::v8 (&qb)[D / 16],
                                             f32x16 (&oacc)[D / 32], float& m, float& l) {
  constexpr int RB = 2 * D;
  using V8 = typename Mfma<T>::v8;
  const int lq = lane & 31, hi = lane >> 5;
  // The MFMA runs go at raised wave priority, the softmax between them at the normal one: with
  // several wavefronts per SIMD the arbiter then feeds the matrix core from a wavefront in its
  // MFMA run ahead of another's vector work (all three kernels; config 5: forward 1.44 -> 1.43
  // ms, backward 5.00 -> 4.91 ms).
  __builtin_amdgcn_s_setprio(1);
  f32x16 acc = f32x16{};
  const uint32_t k0 = swz_row_base<RB>(lane);
  constexpr int KA = 3;
  V8 kbuf[KA];
#pragma unroll
  for (int c = 0; c < KA; ++c) kbuf[c] = ld16<V8>(ks + (k0 ^ (32u * c)));
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int c = 0; c < D / 16; ++c) {
    acc = Mfma<T>::run(kbuf[c % KA], qb[c], acc);
    if (c + KA < D / 16) kbuf[c % KA] = ld16<V8>(ks + (k0 ^ (32u * (c + KA))));
    __builtin_amdgcn_sched_barrier(0);
  }
  // V^T operand j: rows 16 (j & 1) .., columns 32 (j >> 1) .. of the V tile
  const SwzTr<RB> vt(lane);
  auto ldv = [&](int j) { return vt.template read<V8>(vs, 16 * (j & 1), j >> 1); };
  constexpr int VA = 2;
  V8 vbuf[VA];
#pragma unroll
  for (int j = 0; j < VA; ++j) vbuf[j] = ldv(j);
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_setprio(0);
  if (kh + 31 > qw0) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int kj = kh + 8 * (i / 4) + 4 * hi + (i % 4);
      if (kj > qi) acc[i] = -INFINITY;
    }
  }
  float mx = acc[0];
#pragma unroll
  for (int i = 1; i < 16; ++i) mx = fmaxf(mx, acc[i]);
  mx = pair_max(mx) * scale_log2;
  const bool grow = mx > m + 8.f;
  float alpha = 1.f;
  if (grow) {
    alpha = exp2_fast(m - mx);
    m = mx;
  }
  const float nm = m == -INFINITY ? 0.f : -m;
  float ps = 0.f;
  V8 pb[2];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const float p = exp2_fast(fmaf(acc[i], scale_log2, nm));
    ps += p;
    pb[i / 8][i % 8] = (T)p;
  }
  ps = pair_sum(ps);
  l = fmaf(l, alpha, ps);
  if (__any(grow)) {
#pragma unroll
    for (int md = 0; md < D / 32; ++md) oacc[md] *= alpha;
  }
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_setprio(1);
#pragma unroll
  for (int j = 0; j < D / 16; ++j) {
    oacc[j / 2] = Mfma<T>::run(vbuf[j % VA], pb[j % 2], oacc[j / 2]);
    if (j + VA < D / 16) vbuf[j % VA] = ldv(j + VA);
    __builtin_amdgcn_sched_barrier(0);
  }
  __builtin_amdgcn_s_setprio(0);
}

// The forward kernel: blocks of 4 wavefronts own 128 queries of one (sequence, query head) with the
// online softmax in registers; the BN-key K / V tiles go through a ring of NBUF = 2 swizzled LDS
// buffers filled by LDS DMA (tile t + 1 in flight while tile t is consumed, one barrier per tile
// publishing it and freeing the buffer consumed before). At D = 64 (rows of 128 bytes, 64-key tiles:
// half the barriers) 12011 tokens in 9 sequences, 14 / 2 heads, bf16, take 64 us, against 121 with K
// and V staged through registers into padded tiles in the hardware's block order (48 in
// level_order).
template <typename T, int D, int BN, int NBUF>
__global__ __launch_bounds__(kAttnThreads, kFwdPerCU<D>) void k_attn_fwd_swz(const AttnArgs a,
                                                                             int qtiles,
                                                                             int order) {
  constexpr int RB = 2 * D;
  constexpr int TILE = BN * RB;  // bytes of one K or V tile
  using V8 = typename Mfma<T>::v8;
  __shared__ __align__(1024) char kv[NBUF][2][TILE];  // [buffer][K, V][swizzled rows]

  const int lin = block_order(attn_block(), qtiles, a.HQ * a.n_seq, order, a.HQ, a.cu, a.n_seq,
                              a.T);
  const int bx = lin % qtiles, rest = lin / qtiles;
  const int h = rest % a.HQ, seq = rest / a.HQ;
  if (seq >= a.n_seq) return;
  int start, end;
  seq_bounds(a.cu, seq, a.T, &start, &end);
  const int ntiles_q = (end - start + kAttnBM - 1) / kAttnBM;
  if (bx >= ntiles_q) return;
  const int q0 = start + (ntiles_q - 1 - bx) * kAttnBM;  // heaviest tiles first
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lq = lane & 31, hi = lane >> 5;
  const int kvh = h / (a.HQ / a.HK);
  const int qw0 = q0 + 32 * w;
  const int qi = qw0 + lq;
  const bool wave_live = qw0 < end;
  const int wq_last = qw0 + 31 < end ? qw0 + 31 : end - 1;

  V8 qb[D / 16];
  {
    const T* qrow = static_cast<const T*>(a.q) + (int64_t)qi * a.q_rs + (int64_t)h * D + 8 * hi;
#pragma unroll
    for (int c = 0; c < D / 16; ++c)
      qb[c] = qi < end ? ld16<V8>(qrow + 16 * c) : V8{};
  }

  f32x16 oacc[D / 32];
#pragma unroll
  for (int md = 0; md < D / 32; ++md) oacc[md] = f32x16{};
  float m = -INFINITY, l = 0.f;
  const int kend = end < q0 + kAttnBM ? end : q0 + kAttnBM;
  const char* kbase = reinterpret_cast<const char*>(static_cast<const T*>(a.k) + (int64_t)kvh * D);
  const char* vbase = reinterpret_cast<const char*>(static_cast<const T*>(a.v) + (int64_t)kvh * D);
  const int64_t krs = a.k_rs * (int64_t)sizeof(T), vrs = a.v_rs * (int64_t)sizeof(T);  // bytes
  const int ntiles = (kend - start + BN - 1) / BN;

  // Rows of a tile past kend repeat row kend - 1: finite data, always masked. Tiles are issued in
  // order, so whole ones step the fillers' running addresses.
  SwzFill<BN, 4, RB> fk(lane, w, krs), fv(lane, w, vrs);
  fk.seq_begin(kbase, start);
  fv.seq_begin(vbase, start);
  auto issue = [&](int buf, int kt) {
    if (kt + BN <= kend) {
      fk.seq_whole(kv[buf][0]);
      fv.seq_whole(kv[buf][1]);
    } else {
      swz_fill2(fk, kv[buf][0], kbase, fv, kv[buf][1], vbase, kt, kend);
    }
  };

  static_assert(NBUF == 2, "the tile loop is unrolled by the ring's two buffers");
  if (ntiles > 0) issue(0, start);
  // Tile t sits in buffer B = t % 2, and the loop is unrolled by two so that B is a constant:
  // the tiles' LDS addresses then fold into the reads' immediate offsets instead of costing a
  // VALU add per read (config-5-like forward 1.39 -> 1.34 ms, the same bits).
  auto tile = [&](int t, auto bc) {
    constexpr int B = decltype(bc)::value;
    // this wavefront's DMA of tile t has landed; the barrier publishes every wavefront's rows
    // and certifies that tile t - 1 is consumed, freeing its buffer for tile t + 1
    __builtin_amdgcn_s_waitcnt(kWaitVm0);
    __syncthreads();
    if (t + 1 < ntiles) issue(B ^ 1, start + (t + 1) * BN);
    const int kt = start + t * BN;
#pragma unroll
    for (int h = 0; h < BN / 32; ++h) {
      if (!wave_live || kt + 32 * h > wq_last) return;
      fwd_tile_swz<T, D>(kv[B][0] + 32 * RB * h, kv[B][1] + 32 * RB * h, kt + 32 * h, qw0, qi, lane,
                         a.scale_log2, qb, oacc, m, l);
    }
  };
  int t = 0;
  for (; t + 1 < ntiles; t += 2) {
    tile(t, std::integral_constant<int, 0>{});
    tile(t + 1, std::integral_constant<int, 1>{});
  }
  if (t < ntiles) tile(t, std::integral_constant<int, 0>{});

  if (!wave_live || qi >= end) return;
  store_rows_t<T, D>(static_cast<T*>(a.o) + (int64_t)qi * a.o_rs + (int64_t)h * D, oacc, hi,
                     l > 0.f ? 1.f / l : 0.f);
  if (hi == 0 && a.lse != nullptr)
    a.lse[(int64_t)h * a.T + qi] = (m + log2f(l)) * 0.69314718055994531f;
}

template <typename T, int D, int BN>
hipError_t fwd_run(const AttnArgs& a, int max_seqlen, hipStream_t s) {
  const int64_t C = (max_seqlen + kAttnBM - 1) / kAttnBM;
  const int64_t n = xcd_grid(C, (int64_t)a.HQ * a.n_seq);
  if (!attn_grid_ok(n)) return hipErrorInvalidValue;
  hipLaunchKernelGGL((k_attn_fwd_swz<T, D, BN, 2>), attn_grid(n), dim3(kAttnThreads), 0, s, a,
                     (int)C, attn_order(n, kFwdPerCU<D>, kRoundsQ, D, a.T, a.n_seq, max_seqlen));
  return hipGetLastError();
}

template <typename T>
hipError_t fwd_d(const AttnArgs& a, int D, int max_seqlen, hipStream_t s, bool* sup) {
  *sup = true;
  if (D == 128) return fwd_run<T, 128, 32>(a, max_seqlen, s);
  if (D == 64) return fwd_run<T, 64, 64>(a, max_seqlen, s);
  *sup = false;
  return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_attn_fwd(const AttnArgs& a, int dt, int D, int max_seqlen, hipStream_t s,
                           bool* sup) {
  if (dt == 1) return fwd_d<_Float16>(a, D, max_seqlen, s, sup);
  if (dt == 2) return fwd_d<__bf16>(a, D, max_seqlen, s, sup);
  *sup = false;
  return hipErrorInvalidValue;
}

}  // namespace esep
