// gemm_stream.hpp -- the bf16 GEMM of decode-sized calls (at most 64 rows of
// A): C[M,N] = A[M,K] @ B[K,N] with the epilogues of gemm_kernels.hpp.
//
// What bounds it: every weight byte is read once and used for at most 64
// rows, so the time is that of streaming B from HBM.  A 64 x 64 tile per
// workgroup (the tiled kernel's smallest) leaves 64 workgroups for N = 4096,
// each a serial chain over all of K: [16, 4096, 16384] took 205 us for 134 MB
// (0.65 TB/s).  Here the K range of a column slice is spread over the WK
// waves of a workgroup and, where the slices alone do not fill the chip, over
// `splits` workgroups.
//
// A workgroup owns a slice of 16*NT columns, 16*MT rows of A and one K split.
// Its WK waves are independent until the end: wave w takes the 32-row k-steps
// w, w + WK, ... of the split through a private ring of STAGES LDS stages
// filled by buffer_load ... lds (HBM -> LDS without registers, the weights
// non-temporal).
//   W part of a stage: 32 row slots of 16*NT bf16.  Slot s holds weight row
//     gs_row(s): the rows one 32-lane pass of ds_read_b64_tr_b16 reads (0-3
//     and 8-11, or 4-7 and 12-15) sit in 8 consecutive slots, and 32-byte unit
//     u of slot s is stored at u ^ gs_xor(s), so that pass covers all 64 banks
//     once.
//   A part: 16*MT rows of 32 bf16, 16-byte chunk c of row r at c ^ ((r >> 2) & 3).
// The MFMA (16x16x32) takes W as its first operand, so lane l holds 4
// consecutive columns of one output row.  At the end the WK partial tiles are
// added in LDS in wave order; one K split applies the epilogue in place,
// several store fp32 partials that gemm_reduce_body adds in split order.
//
// Measured: [16, 16384, 4096] 56 -> 24.1 us and [16, 4096, 16384] 205 -> 27.1 us
// with its reduction (134 MB of weights each, 5.6 and 5.0 TB/s), [16, 28672,
// 8192] 75.8 us (6.2 TB/s).  Without the MFMAs and without A's loads (timing
// only) the first takes 24.6 and 22.3 us: the rest is the weight stream.
//
// Needs K % 8 == 0, N % 8 == 0 and 16-byte aligned A and B; K % 32 != 0 runs a
// last step whose missing rows are zeroed in registers.
#pragma once

#include <type_traits>

#include "gemm_kernels.hpp"

namespace pk {
namespace gk {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int GS_KSTEP = 32;

struct GemmStreamArgs {
  GemmArgs g;
  float *partial;   // [splits][M][N] fp32, splits > 1
  int splits;
  int split_steps;  // k-steps of GS_KSTEP rows per split
  int slices;       // column slices of the grid
};

// Weight row held by LDS row slot s (0..31), its own inverse.
__device__ __forceinline__ int gs_row(int s) {
  return (s & 0x13) | ((s & 4) << 1) | ((s & 8) >> 1);
}
// 32-byte-unit XOR of slot s: 256 bytes of banks hold 8 / NT slots.
template <int NT>
__device__ __forceinline__ int gs_xor(int s) {
  if constexpr (NT == 1) return 0;
  else if constexpr (NT == 2) return (s >> 2) & 1;
  else if constexpr (NT == 4) return (s >> 1) & 3;
  else return s & 7;
}

// Epilogue of 8 consecutive outputs of row m from their fp32 sums; `tab` is the
// GELU table (global or LDS).
template <int EPI>
__device__ __forceinline__ void gemm_finish8(const f32x4 v0, const f32x4 v1, int m, int n, const GemmArgs &g,
                                             const uint16_t *tab) {
#pragma clang fp contract(off)
  u32x4 t = {pack_bf(v0[0], v0[1]), pack_bf(v0[2], v0[3]), pack_bf(v1[0], v1[1]), pack_bf(v1[2], v1[3])};
  if constexpr (EPI == EPI_BIAS_GELU || EPI == EPI_BIAS_RESID) {
    const u32x4 b = g.bias ? *reinterpret_cast<const u32x4 *>(g.bias + n) : u32x4{0, 0, 0, 0};
#pragma unroll
    for (int e = 0; e < 4; ++e) t[e] = pack_bf(lo_bf(t[e]) + lo_bf(b[e]), hi_bf(t[e]) + hi_bf(b[e]));
  }
  if constexpr (EPI == EPI_BIAS_GELU) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      t[e] = gelu_pair_exact(t[e], tab);
  }
  if constexpr (EPI == EPI_BIAS_RESID || EPI == EPI_RESID) {
    const u32x4 r = *reinterpret_cast<const u32x4 *>(g.R + (size_t)m * g.N + n);
#pragma unroll
    for (int e = 0; e < 4; ++e) t[e] = pack_bf(lo_bf(t[e]) + lo_bf(r[e]), hi_bf(t[e]) + hi_bf(r[e]));
  }
  *reinterpret_cast<u32x4 *>(g.C + (size_t)m * g.N + n) = t;
}

// Sum of the split partials in split order and the epilogue, 8 outputs per
// thread: every split's 16-byte loads are independent and in flight at once.
template <int EPI>
__device__ __forceinline__ void gemm_reduce_body(const GemmArgs &g, const float *__restrict__ partial, int splits) {
  const int64_t total = (int64_t)g.M * g.N;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x * 8;
  for (int64_t e = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 8; e < total; e += stride) {
    const float *p = partial + e;
    f32x4 s0 = *reinterpret_cast<const f32x4 *>(p), s1 = *reinterpret_cast<const f32x4 *>(p + 4);
#pragma unroll 8
    for (int sp = 1; sp < splits; ++sp) {
      const float *q = p + (size_t)sp * total;
      s0 += *reinterpret_cast<const f32x4 *>(q);
      s1 += *reinterpret_cast<const f32x4 *>(q + 4);
    }
    gemm_finish8<EPI>(s0, s1, (int)(e / g.N), (int)(e % g.N), g, g.gelu_tab);
  }
}

template <int NT, int MT, int WK, int STAGES, int EPI>
__device__ __forceinline__ void gemm_stream_body(const GemmStreamArgs &a) {
  static_assert(NT == 1 || NT == 2 || NT == 4 || NT == 8, "column tiles");
  static_assert(STAGES >= 2 && STAGES <= 8, "ring depth");
  constexpr int W_BYTES = 1024 * NT;        // 32 rows x 16*NT bf16
  constexpr int STAGE = W_BYTES + 1024 * MT;
  constexpr int RING = STAGES * STAGE;      // per wave
  constexpr int P = NT + MT;                // DMA instructions per step
  constexpr int WN = 16 * NT;               // columns per wave
  constexpr int LD = WN + 4;                // row stride of a wave's fp32 tile (16 rows on distinct banks)
  static_assert(16 * MT * LD * 4 <= RING, "the wave's partial tile reuses its ring");
  __shared__ __attribute__((aligned(1024))) uint8_t ring[WK * RING];
  const GemmArgs &g = a.g;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wk = __builtin_amdgcn_readfirstlane(tid >> 6);
  // consecutive slices share the lines of narrow runs
  const int u = xcd_unit(blockIdx.x, a.slices * a.splits);
  const int slice = u / a.splits, split = u % a.splits;
  const int n0 = slice * WN;
  const int m0 = blockIdx.y * 16 * MT;
  const int ksteps = (g.K + GS_KSTEP - 1) / GS_KSTEP;
  const int w0 = split * a.split_steps;
  const int wsteps = min(ksteps, w0 + a.split_steps) - w0;  // k-steps of the split
  const int T = wsteps > wk ? (wsteps - wk + WK - 1) / WK : 0;  // of this wave

  // ---- DMA sources: one resource per operand, a loop-invariant per-lane
  // offset and the step's first row in the scalar offset.  Columns past N and
  // rows past M are clamped onto valid data whose results are not stored.
  const pk_u32x4 w_rsrc = rsrc_words(g.B + n0, (uint32_t)(((size_t)g.K * g.N - n0) * 2));
  const pk_u32x4 a_rsrc = rsrc_words(g.A + (size_t)m0 * g.K, (uint32_t)((size_t)min(g.M - m0, 16 * MT) * g.K * 2));
  uint32_t w_off[NT], a_off[MT];
  int w_row[NT];
#pragma unroll
  for (int q = 0; q < NT; ++q) {
    const int c = 64 * q + lane;
    const int s = c / (2 * NT), p = c % (2 * NT);
    const int col = min(16 * ((p >> 1) ^ gs_xor<NT>(s)) + 8 * (p & 1), g.N - 8 - n0);
    w_row[q] = gs_row(s);
    w_off[q] = (uint32_t)(w_row[q] * g.N + col) * 2u;
  }
  const int a_k = 8 * ((lane & 3) ^ ((lane >> 4) & 3));  // k of the lane's A chunk (row = 16 q + lane / 4)
#pragma unroll
  for (int q = 0; q < MT; ++q) a_off[q] = (uint32_t)(min(16 * q + (lane >> 2), g.M - 1 - m0) * g.K + a_k) * 2u;

  uint8_t *my = ring + wk * RING;
  auto issue = [&](int st, int t) __attribute__((always_inline)) {
    const int k0 = (w0 + wk + WK * t) * GS_KSTEP;
    uint8_t *base = my + st * STAGE;
    if (k0 + GS_KSTEP <= g.K) {
#pragma unroll
      for (int q = 0; q < NT; ++q) dma_lds16<true>(w_rsrc, base + 1024 * q, w_off[q], (uint32_t)k0 * g.N * 2u);
#pragma unroll
      for (int q = 0; q < MT; ++q) dma_lds16(a_rsrc, base + W_BYTES + 1024 * q, a_off[q], k0 * 2);
    } else {  // the last step of a K that is not a multiple of 32: rows past K repeat the last valid ones
      const int last = g.K - 1 - k0;
#pragma unroll
      for (int q = 0; q < NT; ++q)
        dma_lds16<true>(w_rsrc, base + 1024 * q, w_off[q] - (uint32_t)(max(0, w_row[q] - last) * g.N) * 2u,
                        (uint32_t)k0 * g.N * 2u);
#pragma unroll
      for (int q = 0; q < MT; ++q)
        dma_lds16(a_rsrc, base + W_BYTES + 1024 * q, a_off[q] - (uint32_t)(max(0, a_k - (last & ~7))) * 2u, k0 * 2);
    }
  };

  // ---- per-lane LDS read offsets within a stage
  const int grp = lane >> 4, gi = lane & 15;
  int w_rd[NT][2], a_rd[MT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int s = gs_row(8 * grp + 4 * r + (gi >> 2));
      w_rd[j][r] = s * (2 * WN) + 32 * (j ^ gs_xor<NT>(s)) + 8 * (gi & 3);
    }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) a_rd[mt] = W_BYTES + (16 * mt + gi) * 64 + 16 * (grp ^ ((gi >> 2) & 3));

  f32x4 acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[mt][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // `k_left` < 32 on the last step of a ragged K: this lane's 8 rows are zeroed in
  // both operands when they lie past K (K % 8 == 0)
  auto compute = [&](int st, int k_left) __attribute__((always_inline)) {
    const uint8_t *base = my + st * STAGE;
    const bool none = 8 * grp >= k_left;
    bf16x8 af[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      u32x4 v = *reinterpret_cast<const u32x4 *>(base + a_rd[mt]);
      if (none) v = u32x4{0, 0, 0, 0};
      af[mt] = __builtin_bit_cast(bf16x8, v);
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const i16x4 h0 = lds_read_tr(reinterpret_cast<const uint16_t *>(base + w_rd[j][0]));
      const i16x4 h1 = lds_read_tr(reinterpret_cast<const uint16_t *>(base + w_rd[j][1]));
      u32x4 v = __builtin_bit_cast(u32x4, __builtin_shufflevector(h0, h1, 0, 1, 2, 3, 4, 5, 6, 7));
      if (none) v = u32x4{0, 0, 0, 0};
      const bf16x8 b = __builtin_bit_cast(bf16x8, v);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        acc[mt][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, af[mt], acc[mt][j], 0, 0, 0);
    }
  };

  // ---- steps 0 .. STAGES-2 in flight, then issue step t+STAGES-1 into the
  // stage read at step t-1, wait for step t, compute it
#pragma unroll
  for (int p = 0; p < STAGES - 1; ++p)
    if (p < T) issue(p, p);
  int t = 0, st = 0;
  for (; t + STAGES - 1 < T; ++t) {
    lgkm_wait0();  // reads of the stage being refilled are done
    issue(st == 0 ? STAGES - 1 : st - 1, t + STAGES - 1);
    vm_wait<(STAGES - 1) * P>();
    compute(st, GS_KSTEP);
    st = st == STAGES - 1 ? 0 : st + 1;
  }
  vm_wait<0>();
  for (; t < T; ++t) {
    compute(st, g.K - (w0 + wk + WK * t) * GS_KSTEP);
    st = st == STAGES - 1 ? 0 : st + 1;
  }

  // ---- add the WK tiles of each column group in wave order
  lgkm_wait0();
  float *tile = reinterpret_cast<float *>(my);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int j = 0; j < NT; ++j)
      *reinterpret_cast<f32x4 *>(tile + (16 * mt + gi) * LD + 16 * j + 4 * grp) = acc[mt][j];
  __syncthreads();
  constexpr int C8 = WN / 8;  // 8-column items per row
  for (int it = tid; it < 16 * MT * C8; it += WK * 64) {
    const int r = it / C8, c = 8 * (it % C8);
    const int m = m0 + r, n = n0 + c;
    if (m >= g.M || n >= g.N) continue;
    const float *p = reinterpret_cast<const float *>(ring) + r * LD + c;
    f32x4 v0 = *reinterpret_cast<const f32x4 *>(p), v1 = *reinterpret_cast<const f32x4 *>(p + 4);
#pragma unroll
    for (int k = 1; k < WK; ++k) {
      const float *q = p + k * (RING / 4);
      v0 += *reinterpret_cast<const f32x4 *>(q);
      v1 += *reinterpret_cast<const f32x4 *>(q + 4);
    }
    if (a.splits > 1) {
      float *o = a.partial + ((size_t)split * g.M + m) * g.N + n;
      *reinterpret_cast<f32x4 *>(o) = v0;
      *reinterpret_cast<f32x4 *>(o + 4) = v1;
    } else {
      gemm_finish8<EPI>(v0, v1, m, n, g, g.gelu_tab);
    }
  }
}

}  // namespace gk
}  // namespace pk
