// gemm_odd.hpp -- the bf16 product of at most 64 rows with weights whose rows
// start at any element (N % 8 != 0, or an unaligned B or C): C[M,N] = A[M,K] @
// B[K,N].  A vocabulary head on the last token of each sequence is one.
//
// What bounds it: the weights are read once, as in gemm_stream.hpp, but 16-byte
// LDS DMA cannot fetch rows that start between 16-byte boundaries, and the
// element-wise tile kernel loads 2 bytes per lane.  Here each lane reads its 16
// bytes of a row from the unaligned address into a register ring of DEPTH
// k-steps (global loads need only element alignment) and writes them to the
// streaming kernel's swizzled LDS slots just before the transpose reads; A's
// operand comes straight from L2.  The waves take alternate 32-row k-steps, and
// their tiles are added in LDS in wave order.
//
// Measured: [16, 50257, 5120] 659 -> 111 us (4.6 TB/s), [30, 30001, 2048] 193 ->
// 27.4 (4.5 TB/s), [16, 2049, 4096] 201 -> 15.4 (65 workgroups: a serial chain of
// 16 k-steps per wave).
#pragma once

#include "gemm_stream.hpp"

namespace pk {
namespace gk {

typedef u32x4 u32x4_el __attribute__((aligned(2)));

template <int NT, int MT, int WK, int DEPTH>
__device__ __forceinline__ void gemm_odd_body(const GemmArgs &g) {
  constexpr int WN = 16 * NT, LD = WN + 4;  // columns; row stride of a wave's fp32 tile
  constexpr int STAGE = 1024 * NT, TILE = 16 * MT * LD * 4;
  constexpr int WAVE = STAGE > TILE ? STAGE : TILE;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[WK * WAVE];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wk = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int slice = xcd_unit(blockIdx.x, gridDim.x);  // neighbours share the lines at their edges
  const int n0 = slice * WN;
  const int ksteps = (g.K + GS_KSTEP - 1) / GS_KSTEP;
  const int T = ksteps > wk ? (ksteps - wk + WK - 1) / WK : 0;  // k-steps of this wave
  const uint32_t total = (uint32_t)g.K * (uint32_t)g.N;         // elements of B, under 2^30

  // Row and column of the lane's 16 bytes in each load (gemm_stream_body's
  // slots).  A chunk may run past its row's end, into columns that are not
  // stored; the last row's stop at the end of B (mend()).
  int w_row[NT], w_col[NT];
#pragma unroll
  for (int q = 0; q < NT; ++q) {
    const int c = 64 * q + lane;
    const int s = c / (2 * NT), p = c % (2 * NT);
    w_row[q] = gs_row(s);
    w_col[q] = n0 + 16 * ((p >> 1) ^ gs_xor<NT>(s)) + 8 * (p & 1);
  }
  const int grp = lane >> 4, gi = lane & 15;
  u32x4 w[DEPTH][NT], av[DEPTH][MT];
  auto step_k0 = [&](int t) __attribute__((always_inline)) { return (wk + WK * min(t, T - 1)) * GS_KSTEP; };
  auto load = [&](u32x4 (&wr)[NT], u32x4 (&ar)[MT], int t) __attribute__((always_inline)) {
    const int k0 = step_k0(t);
#pragma unroll
    for (int q = 0; q < NT; ++q) {
      const uint32_t at = (uint32_t)min(k0 + w_row[q], g.K - 1) * (uint32_t)g.N + (uint32_t)w_col[q];
      wr[q] = *reinterpret_cast<const u32x4_el *>(g.B + min(at, total - 8));
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      ar[mt] = *reinterpret_cast<const u32x4 *>(g.A + (size_t)min(16 * mt + gi, g.M - 1) * g.K + min(k0 + 8 * grp, g.K - 8));
  };

  uint8_t *my = smem + wk * WAVE;
  int w_rd[NT][2];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int s = gs_row(8 * grp + 4 * r + (gi >> 2));
      w_rd[j][r] = s * (2 * WN) + 32 * (j ^ gs_xor<NT>(s)) + 8 * (gi & 3);
    }
  f32x4 acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[mt][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // the chunks of the last rows that would run past the end of B, by element
  auto mend = [&](int k0) __attribute__((always_inline)) {
    for (int q = 0; q < NT; ++q) {
      const uint32_t at = (uint32_t)min(k0 + w_row[q], g.K - 1) * (uint32_t)g.N + (uint32_t)w_col[q];
      if (at > total - 8)
        for (uint32_t e = 0; e < 8; ++e)
          reinterpret_cast<uint16_t *>(my + 1024 * q + 16 * lane)[e] = at + e < total ? g.B[at + e] : 0;
    }
  };
  auto compute = [&](const u32x4 (&wr)[NT], const u32x4 (&ar)[MT], int t) __attribute__((always_inline)) {
    const int k0 = step_k0(t);
#pragma unroll
    for (int q = 0; q < NT; ++q) *reinterpret_cast<u32x4 *>(my + 1024 * q + 16 * lane) = wr[q];
    if (k0 + GS_KSTEP >= g.K) mend(k0);
    const bool none = 8 * grp >= g.K - k0;  // the lane's 8 rows lie past K
    bf16x8 af[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) af[mt] = __builtin_bit_cast(bf16x8, none ? u32x4{0, 0, 0, 0} : ar[mt]);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const i16x4 h0 = lds_read_tr(reinterpret_cast<const uint16_t *>(my + w_rd[j][0]));
      const i16x4 h1 = lds_read_tr(reinterpret_cast<const uint16_t *>(my + w_rd[j][1]));
      u32x4 v = __builtin_bit_cast(u32x4, __builtin_shufflevector(h0, h1, 0, 1, 2, 3, 4, 5, 6, 7));
      if (none) v = u32x4{0, 0, 0, 0};
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        acc[mt][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, v), af[mt], acc[mt][j], 0, 0, 0);
    }
  };

  if (T > 0) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) load(w[d], av[d], d);
    for (int t = 0; t < T; t += DEPTH) {
#pragma unroll
      for (int d = 0; d < DEPTH; ++d) {
        if (t + d < T) compute(w[d], av[d], t + d);
        load(w[d], av[d], t + d + DEPTH);  // past the end: the last step again
      }
    }
  }

  // ---- add the WK tiles in wave order
  float *tile = reinterpret_cast<float *>(my);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int j = 0; j < NT; ++j)
      *reinterpret_cast<f32x4 *>(tile + (16 * mt + gi) * LD + 16 * j + 4 * grp) = acc[mt][j];
  __syncthreads();
  for (int it = tid; it < 16 * MT * WN; it += WK * 64) {
    const int m = it / WN, c = it % WN;
    if (m >= g.M || n0 + c >= g.N) continue;
    const float *p = reinterpret_cast<const float *>(smem) + m * LD + c;
    float v = *p;
#pragma unroll
    for (int k = 1; k < WK; ++k) v += p[k * (WAVE / 4)];
    g.C[(size_t)m * g.N + n0 + c] = (uint16_t)f2bf(v);
  }
}

}  // namespace gk
}  // namespace pk
