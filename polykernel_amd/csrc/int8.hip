// int8.hip -- int8 weight-only matmul for decode shapes (small M) on gfx950.
//
// C[M,N] = bf16(scale[n] * sum_k A[m,k] * Wq[k,n]), A bf16 [M,K], Wq int8 [K,N]
// (N contiguous, the reference layout of kernels/generated/matmul_int8.cu:47-88).
// The per-channel scale is applied once to the fp32 dot product instead of to
// every weight (kernels/cpu/matmul_quant.cpp:189-199 dequantises per element);
// int8 values and their products with bf16 activations are exact in fp32, so
// only the summation order and that one rounding differ.
//
// Streaming design (HBM-bound: every weight byte is read once):
//   - a workgroup owns a 64-column slice of N and a K range (split-K);
//   - each of its 4 waves streams a quarter of that K range in 32-row steps:
//     two 16-byte loads per lane fetch a 32x64 int8 block, which is widened to
//     bf16 in registers (exact) and written to the wave's private LDS block in
//     the swizzled N-contiguous layout of the bf16 GEMM;
//   - ds_read_b64_tr_b16 assembles the MFMA B operand (8 consecutive k of one
//     column); A (16 rows of activations) is read straight from global/L2;
//   - v_mfma_f32_16x16x32_bf16, 4 column blocks per step;
//   - the 4 waves' accumulators are summed in LDS in a fixed order; with one
//     K split the epilogue runs in place, otherwise fp32 partials go to a
//     workspace and int8_reduce_kernel sums the splits in split order.
// Epilogues: plain, GELU (exact table) and residual add, each with the
// golden's per-stage bf16 rounding.
#include <mutex>

#include "gemm_plan.hpp"
#include "gemm_ring.hpp"
#include "int8_stream.hpp"

namespace pk {

namespace {

using namespace i8s;

constexpr int I8_BN = 64;      // columns per workgroup
constexpr int I8_STEP = 32;    // k rows per wave step
constexpr int I8_WAVES = 4;
constexpr int I8_THREADS = I8_WAVES * 64;

struct Int8Args {
  const uint16_t *A;
  const int8_t *W;
  const float *scale;
  float *partial;  // [splits][M][N] when splits > 1
  uint16_t *C;
  const uint16_t *R;
  const uint16_t *gelu_tab;
  int M, N, K;
  int splits;
  int kper;  // rows of K per split (multiple of I8_STEP * I8_WAVES)
};

__device__ __forceinline__ int swz64(int k) { return (k & 3) * 2; }

// Widen 4 int8 (one dword) to 4 bf16 in two dwords.  int8 -> fp32 is exact and
// the fp32 value has at most 8 significant bits, so its top half is the bf16.
__device__ __forceinline__ void widen4(uint32_t w, uint32_t &lo, uint32_t &hi) {
  const float f0 = (float)(int8_t)(w & 0xFF), f1 = (float)(int8_t)((w >> 8) & 0xFF);
  const float f2 = (float)(int8_t)((w >> 16) & 0xFF), f3 = (float)(int8_t)(w >> 24);
  lo = (__float_as_uint(f0) >> 16) | (__float_as_uint(f1) & 0xFFFF0000u);
  hi = (__float_as_uint(f2) >> 16) | (__float_as_uint(f3) & 0xFFFF0000u);
}

template <int EPI>
__device__ __forceinline__ uint16_t int8_epilogue(float dot, int m, int n, const Int8Args &g) {
#pragma clang fp contract(off)
  const uint32_t t = f2bf(dot * g.scale[n]);
  if constexpr (EPI == I8_NONE) {
    return (uint16_t)t;
  } else if constexpr (EPI == I8_GELU) {
    return (uint16_t)gelu_bits(t, g.gelu_tab);
  } else {
    return (uint16_t)f2bf(bf2f(t) + bf2f(g.R[(size_t)m * g.N + n]));
  }
}

template <bool ALIGNED, int EPI>
__global__ __launch_bounds__(I8_THREADS) void int8_gemm_kernel(Int8Args g) {
  __shared__ __attribute__((aligned(16))) uint16_t wlds[I8_WAVES][I8_STEP * I8_BN];
  __shared__ float red[I8_WAVES][16 * I8_BN];

  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int n0 = blockIdx.x * I8_BN;
  const int split = blockIdx.y;
  const int m0 = blockIdx.z * 16;
  const int kb0 = split * g.kper;
  const int kb1 = min(g.K, kb0 + g.kper);
  const int wk = g.kper / I8_WAVES;  // rows per wave
  const int kw0 = kb0 + wid * wk;
  const int kw1 = min(kb1, kw0 + wk);

  uint16_t *my = wlds[wid];
  f32x4 acc[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // A operand (16x16x32): row m = lane % 16, k = 8 * (lane / 16) + 0..7.
  const int am = m0 + (lane & 15);
  const int ak = 8 * (lane >> 4);
  // W block loads: part p covers rows p*16 + lane/4, columns (lane%4)*16 .. +15.
  const int wr = lane >> 2, wc = (lane & 3) * 16;
  // tr-read coordinates (per 16-lane group g: k base 8g; lane i -> row i/4, col 4*(i%4)).
  const int grp = lane >> 4, gi = lane & 15;

  for (int k0 = kw0; k0 < kw1; k0 += I8_STEP) {
    // ---- loads
    u32x4 wv[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int k = k0 + p * 16 + wr;
      const int n = n0 + wc;
      if constexpr (ALIGNED) {
        wv[p] = (k < kw1 && n < g.N) ? *reinterpret_cast<const u32x4 *>(g.W + (size_t)k * g.N + n)
                                     : u32x4{0, 0, 0, 0};
      } else {
        uint32_t w4[4] = {0, 0, 0, 0};
        if (k < kw1) {
#pragma unroll
          for (int e = 0; e < 16; ++e)
            if (n + e < g.N)
              w4[e >> 2] |= ((uint32_t)(uint8_t)g.W[(size_t)k * g.N + n + e]) << (8 * (e & 3));
        }
        wv[p] = u32x4{w4[0], w4[1], w4[2], w4[3]};
      }
    }
    u32x4 av;
    {
      const int k = k0 + ak;
      if constexpr (ALIGNED) {
        av = (am < g.M && k < kw1) ? *reinterpret_cast<const u32x4 *>(g.A + (size_t)am * g.K + k)
                                   : u32x4{0, 0, 0, 0};
      } else {
        uint32_t a4[4] = {0, 0, 0, 0};
        if (am < g.M) {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (k + e < kw1) a4[e >> 1] |= (uint32_t)g.A[(size_t)am * g.K + k + e] << (16 * (e & 1));
        }
        av = u32x4{a4[0], a4[1], a4[2], a4[3]};
      }
    }
    // ---- widen to bf16 and stage in this wave's LDS block
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int row = p * 16 + wr;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        uint32_t o0, o1, o2, o3;
        widen4(wv[p][2 * h], o0, o1);
        widen4(wv[p][2 * h + 1], o2, o3);
        const u32x4 o = {o0, o1, o2, o3};
        const int c = (wc >> 3) + h;  // 16-byte chunk of the 128-byte row
        *reinterpret_cast<u32x4 *>(my + row * I8_BN + ((c ^ swz64(row)) << 3)) = o;
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const bf16x8 a = __builtin_bit_cast(bf16x8, av);
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
      i16x4 h[2];
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const int row = 8 * grp + 4 * r + (gi >> 2);
        const int col = nb * 16 + 4 * (gi & 3);
        const int c = col >> 3;
        h[r] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_i16x4 *)(my + row * I8_BN + ((c ^ swz64(row)) << 3) + (col & 7)));
      }
      short tmp[8] = {h[0][0], h[0][1], h[0][2], h[0][3], h[1][0], h[1][1], h[1][2], h[1][3]};
      acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(bf16x8, tmp), acc[nb],
                                                        0, 0, 0);
    }
    // The next step overwrites this wave's block: keep its reads ahead of those writes.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }

  // ---- cross-wave reduction (fixed order) -> epilogue or partial
  // D layout (16x16): acc[nb][i] -> row (lane/16)*4 + i, col nb*16 + lane%16.
#pragma unroll
  for (int nb = 0; nb < 4; ++nb)
#pragma unroll
    for (int i = 0; i < 4; ++i) red[wid][((lane >> 4) * 4 + i) * I8_BN + nb * 16 + (lane & 15)] = acc[nb][i];
  __syncthreads();
  for (int e = tid; e < 16 * I8_BN; e += I8_THREADS) {
    const int r = e / I8_BN, c = e % I8_BN;
    const int m = m0 + r, n = n0 + c;
    if (m >= g.M || n >= g.N) continue;
    float s = red[0][e];
#pragma unroll
    for (int w = 1; w < I8_WAVES; ++w) s += red[w][e];
    if (g.splits > 1)
      g.partial[((size_t)split * g.M + m) * g.N + n] = s;
    else
      g.C[(size_t)m * g.N + n] = int8_epilogue<EPI>(s, m, n, g);
  }
}

// Split reduction, 8 outputs per thread: the partials of all splits are
// loaded with 16-byte loads (independent, so they are all in flight at once)
// and added in split order.  Needs N % 8 == 0 and 16-byte aligned buffers.
template <int EPI>
__global__ __launch_bounds__(PK_I8_REDUCE_THREADS) void int8_reduce8_kernel(Int8Args g) {
  reduce8_body<EPI>(g.partial, g.splits, g.M, g.N, g.scale, g.R, g.gelu_tab, g.C);
}

template <int EPI>
__global__ __launch_bounds__(256) void int8_reduce_kernel(Int8Args g) {
  const int64_t total = (int64_t)g.M * g.N;
  for (int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x; t < total; t += (int64_t)gridDim.x * 256) {
    float s = g.partial[t];
    for (int sp = 1; sp < g.splits; ++sp) s += g.partial[(size_t)sp * total + t];
    const int m = (int)(t / g.N), n = (int)(t % g.N);
    g.C[t] = int8_epilogue<EPI>(s, m, n, g);
  }
}

// The streaming kernel (body in int8_stream.hpp, shared with emitted code
// objects).
template <int NT, int MT, int WAVES, int STAGES, int EPI>
__global__ __launch_bounds__(WAVES * 64, 1) void int8_stream_kernel(I8sArgs g) {
  stream_body<NT, MT, WAVES, STAGES, EPI>(g);
}

// Four or more K splits whose starts lie a multiple of 16 MB apart meet in the
// same memory channels; such a split is made one step longer ([16, 8192, 28672]
// in 14: 45.0 us at 32 steps of 64 rows, 43.2 at 33).
bool aliased_split(int splits, int steps, int N) {
  return splits >= 4 && (size_t)steps * I8S_KSTEP * N % (size_t(16) << 20) == 0;
}

// ---- decode calls on smaller weights (kstream_body) ----------------------------
template <int NT, int MT, int WK, int STAGES, int EPI>
__global__ __launch_bounds__(WK * 64) void int8_kstream_kernel(I8sArgs a) {
  kstream_body<NT, MT, WK, STAGES, EPI>(a);
}
// By slice width (16 * nt columns) and rows (16 * mt); `rate`: weight bytes per
// ns of one workgroup, fitted to [1-32, N, K] for N 1040-16384, K 520-28672.
struct KsVariant {
  int nt, mt;
  double rate;
  void (*fn[3])(dim3, hipStream_t, const I8sArgs &);
};
template <int NT, int MT, int WK, int STAGES, int EPI>
void kstream_launch(dim3 grid, hipStream_t st, const I8sArgs &a) {
  int8_kstream_kernel<NT, MT, WK, STAGES, EPI><<<grid, WK * 64, 0, st>>>(a);
}
#define I8K_V(NT, MT, WK, S, RATE)                                                                    \
  {                                                                                                   \
    NT, MT, RATE, {                                                                                   \
      kstream_launch<NT, MT, WK, S, I8_NONE>, kstream_launch<NT, MT, WK, S, I8_GELU>,                 \
          kstream_launch<NT, MT, WK, S, I8_RESID>                                                     \
    }                                                                                                 \
  }
const KsVariant kI8k[] = {
    I8K_V(8, 1, 4, 2, 33.0), I8K_V(4, 1, 4, 2, 18.0), I8K_V(2, 1, 4, 3, 11.0), I8K_V(1, 1, 4, 4, 7.3),
    I8K_V(8, 2, 4, 2, 29.0), I8K_V(4, 2, 4, 2, 17.0), I8K_V(2, 2, 4, 3, 9.5),  I8K_V(1, 2, 4, 4, 6.5),
};
#undef I8K_V
struct KsPlan {
  const KsVariant *v = nullptr;
  int splits = 1, split_steps = 0, slices = 0;
};
// Up to 32 rows and weights of at most 100 MB, where the reduction of the
// column-split stream's partials is a large part of the call ([16, 16384, 4096]
// 20.5 -> 17.8 us, [16, 11008, 4096] 16.9 -> 14.0, [32, 4096, 14336] 23.4 ->
// 19.5); above, its 512-byte runs win ([16, 28672, 8192] 43.5 against 46.4).
// The time model is that of the bf16 streaming kernel with this kernel's
// rates, and 5.8 TB/s of memory.  Rows of a multiple of 1024 bytes put a slice's
// rows into the same few channels: on such weights above 32 MB a workgroup of 16
// rows draws 28 bytes per ns, and 464-512 workgroups, two to a CU, stream as fast
// as one full round, faster than a round that cannot be filled ([1, 5120, 16384] in
// 12 21.9 us, in 5 26.5, column-split 21.7; [1, 3072, 22784] in 10 18.2, in 8 20.9,
// 21.5; [1, 12288, 7296] in 5 21.4, in 2 23.5, 22.3).
// Not taken, us column-split or generic / here: rows of a k-step or two over many
// columns ([3, 24640, 32] 2.8 / 3.5, [29, 36064, 64] 5.8 / 7.2; whole 64-k steps only
// past 256 slices), and few columns over a long K that is no multiple of 64, which
// the generic kernel splits more finely ([26, 144, 28280] 14.6 / 17.4).
bool kstream_pays(int N, int K) {
  if (K % I8S_KSTEP == 0) return K > I8S_KSTEP || N <= 32768;
  return (K > 104 || N < 4096) && !(N > 64 && N <= 192 && K > 8192);
}
bool kstream_plan(int M, int N, int K, size_t scratch, KsPlan &best) {
  if (M > 32 || N % 16 != 0 || K % 8 != 0 || (size_t)K * N > (size_t)100000000 || !kstream_pays(N, K)) return false;
  const int mt = M <= 16 ? 1 : 2;
  const bool lines = mt == 1 && N % 1024 == 0 && (size_t)K * N > (size_t)32000000;
  const int ksteps = (K + I8S_KSTEP - 1) / I8S_KSTEP;
  double best_us = 0;
  for (const KsVariant &v : kI8k) {
    if (v.mt != mt) continue;
    const int nb = 16 * v.nt, slices = (N + nb - 1) / nb;
    for (int s : {1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16}) {
      int steps = (ksteps + s - 1) / s;
      if (s > 1 && steps < 6) break;
      if (aliased_split(s, steps, N)) ++steps;
      const int splits = (ksteps + steps - 1) / steps;
      const size_t part = splits > 1 ? (size_t)splits * M * N * sizeof(float) : 0;
      if (part > scratch) break;
      const int64_t units = (int64_t)slices * splits;
      const double rounds = std::ceil(units / 256.0);
      const bool full = lines && units >= 464 && units <= 512;
      const int round = slices <= 256 ? 256 / slices * slices : 0;  // the fullest single one
      const double fill = units <= 256 ? 1.0 : !full ? 1.1 : round < (N <= 8192 ? 245 : 210) ? 0.96 : 1.0;
      const double rate = lines && v.nt == 8 ? 28.0 : v.rate;
      const double hbm = (double)N * K * fill * (mt == 2 ? 1.1 : 1.0) / 5.8e6;
      double us = 3.0 + std::max(hbm, rounds * steps * I8S_KSTEP * nb / (rate * 1e3));
      if (splits > 1) us += 2.5 + 2.0 * part / 5e6;
      if (!best.v || us < best_us * (1 - 1e-9)) {
        best_us = us;
        best = KsPlan{&v, splits, steps, slices};
      }
    }
  }
  return best.v != nullptr;
}

// ---- prompt-sized calls (gemm_ring.hpp, weights widened in registers) ---------
template <int FM, int WN, int STAGES, int EPI>
__global__ __launch_bounds__(gk::GR_THREADS, 1) void int8_ring_kernel(gk::GemmRingArgs a) {
  gk::gemm_ring_body<FM, WN, STAGES, EPI, true>(a);
}
using RingLaunch = void (*)(dim3, hipStream_t, const gk::GemmRingArgs &);
template <int FM, int WN, int STAGES, int EPI>
void ring_launch(dim3 grid, hipStream_t st, const gk::GemmRingArgs &a) {
  int8_ring_kernel<FM, WN, STAGES, EPI><<<grid, gk::GR_THREADS, 0, st>>>(a);
}
#define I8R_V(FM, WN, S) \
  { ring_launch<FM, WN, S, I8_NONE>, ring_launch<FM, WN, S, I8_GELU>, ring_launch<FM, WN, S, I8_RESID> }
const RingTile kI8Ring[] = {{2, 2, 0.33}, {4, 2, 0.456}, {5, 2, 0.558}, {4, 4, 0.728}, {5, 4, 0.9}};
const RingLaunch kI8RingFn[][3] = {I8R_V(2, 2, 6), I8R_V(4, 2, 5), I8R_V(5, 2, 5), I8R_V(4, 4, 4), I8R_V(5, 4, 4)};
#undef I8R_V

// Above 32 rows the streaming kernel's workgroups re-read the weights for each
// block of rows ([300, 12288, 4096] 87 us with five blocks of 64, 43.8 here) or
// widen a weight for few MFMAs (M 64: [64, 12288, 4096] 29.0 and 22.0 us, M 33:
// [33, 12288, 4096] 25.9 and 21); at M 32 it still wins or ties.  The model is
// fitted to 32 shapes of 33-1000 rows: within 0.6 % of the best variant.
constexpr int kI8RingRows = 32;
constexpr RingModel kI8RingModel{5.4, 1.1, 0.12, 6.4e6, 2.0, 4.4e6};
constexpr size_t kInt8ScratchBytes = size_t(16) << 20;
// Whether the plan beats the column-split stream (K % 64 == 0) or the generic
// kernel, us of those / here.  Its fixed cost is 4.9 against 2.9 and 2.7, so it
// needs weights to read: `work` bytes, once for each 64 rows, as the stream does
// ([53, 1024, 56] 3.0 / 4.9, [44, 512, 368] 4.1 / 6.8, [39, 8192, 64] 3.5 / 5.0;
// [224, 2800, 184] generic 5.3 / 6.1), and at one or two k-steps rounds that are
// nearly full at one ([160, 36848, 64] 10.9 / 17.1 in 1.1 rounds, [43, 30000, 64] 7.2 / 5.6 in
// 0.9).  Up to 128 columns the stream has no wide slice ([108, 128, 512] 17.1 / 7.6).
// Few tiles over a long K are split in 8 at most, the others in 16 and more ([35,
// 688, 27968] 23 / 30, [66, 48, 27144] generic 13 / 29, [150, 192, 16384] 17 / 21; more
// than 128 rows of up to 128 columns [556, 128, 8576] 20.3 / 16.0).  17000 products of whole
// steps: 392 take over 4 % longer than in the other kernel, 172 would be shorter in this.
bool i8_ring_pays(int M, int N, int K, const RingChoice &p) {
  const double work = (double)((M + 63) / 64) * N * K;
  if (K % I8S_KSTEP != 0)
    return p.units > 128 ? p.units > 180 || work > 1.4e6 : (double)M * N * K > 2e8 && (int64_t)M * N > 50000;
  const double fill = p.units / (256.0 * ((p.units + 255) / 256));
  if (p.splits >= 8 && p.units <= 72 && K > (p.units <= 40 ? 4096 : 8192)) return N <= 128 && M > 128;
  if (N <= 128 || K > 256) return true;
  if (K <= 128)
    return work > (K <= 64 ? 3.6e6 : 3e6) ? K > 64 || p.units <= 256 || fill >= 0.66 : fill > 0.88 && M <= 128;
  return work > 1.3e6 || fill > 0.66 || (N > 1032 && (int64_t)M * N > 75000);
}
RingChoice i8_ring_plan(int M, int N, int K, size_t scratch) {
  if (M <= kI8RingRows) return RingChoice{};
  const RingChoice p =
      ring_choose(kI8Ring, (int)(sizeof kI8Ring / sizeof kI8Ring[0]), kI8RingModel, M, N, K, 1, scratch);
  return p.tile >= 0 && i8_ring_pays(M, N, K, p) ? p : RingChoice{};
}
// The built-in choice ahead of the column-split and generic kernels; neither
// set: those.
struct Int8Plan {
  KsPlan ks;
  RingChoice ring;
};
Int8Plan int8_plan(int M, int N, int K, size_t scratch) {
  static thread_local PlanMemo<Int8Plan> memo;
  return memo.get(M, N, K, scratch, 0, [&] {
    Int8Plan p;
    if (!kstream_plan(M, N, K, scratch, p.ks)) p.ring = i8_ring_plan(M, N, K, scratch);
    return p;
  });
}

// Number of K splits: enough workgroups to cover the chip ~4x, each wave
// keeping at least 8 steps.
int choose_splits(int M, int N, int K) {
  const int tiles = ((N + I8_BN - 1) / I8_BN) * ((M + 15) / 16);
  const int unit = I8_STEP * I8_WAVES;
  const int kunits = (K + unit - 1) / unit;
  int s = 1;
  while (tiles * s < 1024 && kunits / (2 * s) >= 2) s *= 2;
  return s;
}

// The generic kernel's split partials in bytes; its splits go to *g if given.
size_t generic_workspace(int M, int N, int K, Int8Args *g) {
  const int unit = I8_STEP * I8_WAVES;
  int splits = choose_splits(M, N, K);
  const int kper = ((K + splits - 1) / splits + unit - 1) / unit * unit;
  splits = (K + kper - 1) / kper;
  if (g) {
    g->splits = splits;
    g->kper = kper;
  }
  return splits > 1 ? (size_t)splits * M * N * sizeof(float) : 0;
}

// ---- streaming-kernel variants and their selection -------------------------
template <int NT, int MT, int WAVES, int STAGES, int EPI>
void i8s_launch(dim3 grid, hipStream_t st, const I8sArgs &g) {
  int8_stream_kernel<NT, MT, WAVES, STAGES, EPI><<<grid, WAVES * 64, 0, st>>>(g);
}
using I8sLaunch = void (*)(dim3, hipStream_t, const I8sArgs &);
struct I8sVariant {
  int nt, mt, waves, stages;
  I8sLaunch fn[3];
};
#define I8S_V(NT, MT, W, S)                                                                  \
  {                                                                                         \
    NT, MT, W, S, {                                                                         \
      i8s_launch<NT, MT, W, S, I8_NONE>, i8s_launch<NT, MT, W, S, I8_GELU>,                 \
          i8s_launch<NT, MT, W, S, I8_RESID>                                                \
    }                                                                                       \
  }
// (NT, MT, WAVES, STAGES): a workgroup covers 16*NT*WAVES columns.  LDS per
// workgroup: stages * waves * 1 KiB * (NT + 2 MT) <= 144 KiB.  In order of
// preference among equal-cost choices.
const I8sVariant kI8s[] = {
    I8S_V(8, 1, 4, 3), I8S_V(7, 1, 4, 3), I8S_V(8, 1, 2, 6), I8S_V(4, 1, 4, 6), I8S_V(4, 1, 8, 3),
    I8S_V(16, 1, 2, 4), I8S_V(2, 1, 4, 6), I8S_V(1, 1, 4, 6), I8S_V(7, 1, 4, 4),
    I8S_V(8, 2, 4, 3), I8S_V(4, 2, 4, 4), I8S_V(2, 2, 4, 6),
    I8S_V(8, 4, 4, 2), I8S_V(4, 4, 4, 3), I8S_V(2, 4, 4, 3),
};
#undef I8S_V

int device_cus() {
  static int cached[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (!cached[dev]) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    cached[dev] = n;
  }
  return cached[dev];
}

struct I8sPlan {
  const I8sVariant *v = nullptr;
  int splits = 1, split_steps = 0, slices = 0, mblocks = 0;
};

bool i8s_shape_ok(int M, int N, int K) {
  return M > 0 && N > 0 && K > 0 && N % 16 == 0 && K % I8S_KSTEP == 0 && (size_t)K * N < (size_t(1) << 31) &&
         (size_t)M * K * 2 < (size_t(1) << 31);
}

// Relative streaming rate of a workgroup of `waves` waves that reads `run`
// contiguous bytes per weight row, from measurements on MI355X with rotating
// 256 MiB buffers: 512 B runs of 4 waves ~5.0 TB/s (the contiguous-read
// ceiling is ~5.7), 128 B ~3.4; 256 B runs probed at ~4.4 but the kernel
// itself streams them at 0.77-0.8 of its 512 B rate (M 16: [4096, 11008]
// 20.1 us with 256-column units against 16.7 with 512, equal bytes per unit);
// runs that are not a multiple of the 128 B cache line lose ~15 % (lines
// shared by two CUs); 2 or 8 waves per workgroup lose ~10 %.
double i8s_run_efficiency(int run, int waves) {
  double e = run >= 512 ? 1.0 : run >= 256 ? 0.8 : run >= 128 ? 0.68 : run >= 64 ? 0.55 : 0.4;
  if (run % 128 != 0) e *= 0.85;
  if (waves != 4) e *= 0.9;
  return e;
}

// Pick the variant and K split for a shape: every CU should stream the same
// number of weight bytes once (units = slices * splits * m-blocks, close to a
// multiple of the usable CU count), in runs of >= 256 B per row; splits cost
// their fp32 partials (written and read back) plus a second launch (counted
// as ~24 MB of HBM time).  Rounds are counted against 7/8 of the CUs: with
// one unit per CU the launch behaves like two rounds (measured at M 16, 512
// columns per unit: [8192, 8192] 23.9 us at 256 units, 23.5 at 304, 17.6 at
// 192; [4096, 16384] 22.4 at 256, 19.5 at 208; [16384, 4096] 22.7 at 256,
// 19.9 at 160), while 220-224 units stream at full rate.  Fields of `req`
// that are nonzero are honoured; returns false when nothing matches.
bool i8s_search(int M, int N, int K, const pk_config *req, int cus, I8sPlan &best) {
  const int ksteps = K / I8S_KSTEP;
  // rows per block: 16 up to M 16, 32 up to M 64 (two blocks at M 64: the
  // 64-row variant holds only two ring stages; measured M 64 [8192, 28672]
  // 66.1 against 71.3 us, [4096, 14336] 28.6 against 31.2), 64 above.  At
  // M 32 two 16-row blocks lose once the weights outgrow the MALL (the
  // second block re-reads them from HBM: [28672, 8192] 60.8 against 48.7 us),
  // so they are taken only for weights of at most 128 MiB (half the MALL:
  // [14336, 4096] 22.9 against 25.2 us, [4096, 14336] 23.4 against 26.5)
  int mt = M <= 16 ? 1 : M <= 64 ? 2 : 4;
  if (M <= 32 && (size_t)K * N <= (size_t(128) << 20)) mt = 1;
  if (req && req->block_m) {
    if (req->block_m != 16 && req->block_m != 32 && req->block_m != 64) return false;
    mt = req->block_m / 16;
  }
  if (req && req->block_k && (req->block_k % I8S_KSTEP != 0 || req->block_k <= 0)) return false;
  if (req && req->vector_width && req->vector_width != I8S_VECTOR_WIDTH) return false;
  if (req && req->unroll && req->unroll != I8S_UNROLL) return false;
  double best_cost = 0;
  bool found = false;
  for (const I8sVariant &v : kI8s) {
    const int nb = 16 * v.nt * v.waves;  // columns per workgroup
    if (v.mt != mt) continue;
    if (req && req->block_n && req->block_n != nb) continue;
    if (req && req->num_warps && req->num_warps != v.waves) continue;
    if (req && req->shared_memory_stages && req->shared_memory_stages != v.stages) continue;
    const int slices = (N + nb - 1) / nb;
    const int mblocks = (M + 16 * mt - 1) / (16 * mt);
    static const int kSplits[] = {1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16, 20, 24, 28, 32};
    for (int s_req : kSplits) {
      int split_steps;
      if (req && req->block_k) {
        if (s_req != 1) break;
        split_steps = std::min(ksteps, req->block_k / I8S_KSTEP);
      } else {
        split_steps = (ksteps + s_req - 1) / s_req;
        if (s_req > 1 && split_steps < 4) break;
        if (aliased_split(s_req, split_steps, N)) ++split_steps;
      }
      const int splits = (ksteps + split_steps - 1) / split_steps;
      const double units = (double)slices * splits * mblocks;
      const double rounds = std::ceil(units / std::max(1, cus * 7 / 8));
      const int run = std::min(nb, N);
      double cost = rounds * split_steps * I8S_KSTEP * (double)run * cus / i8s_run_efficiency(run, v.waves);
      if (splits > 1) cost += 2.0 * splits * M * (double)N * 4 + 24e6;
      if (!found || cost < best_cost * (1 - 1e-9)) {
        found = true;
        best_cost = cost;
        best.v = &v;
        best.splits = splits;
        best.split_steps = split_steps;
        best.slices = slices;
        best.mblocks = mblocks;
      }
    }
  }
  return found;
}

bool i8s_plan(int M, int N, int K, const pk_config *req, int cus, I8sPlan &best) {
  if (!i8s_shape_ok(M, N, K)) return false;
  if (req) return i8s_search(M, N, K, req, cus, best);
  static thread_local PlanMemo<I8sPlan> memo;  // v null: no variant takes the shape
  best = memo.get(M, N, K, 0, cus, [&] {
    I8sPlan p;
    if (!i8s_search(M, N, K, nullptr, cus, p)) p = I8sPlan{};
    return p;
  });
  return best.v != nullptr;
}

size_t i8s_workspace(const I8sPlan &p, int M, int N) {
  return p.splits > 1 ? (size_t)p.splits * M * N * sizeof(float) : 0;
}

pk_config i8s_config(const I8sVariant &v, int split_steps) {
  return pk_config{16 * v.mt, 16 * v.nt * v.waves, split_steps * I8S_KSTEP, v.waves,
                   I8S_VECTOR_WIDTH, I8S_UNROLL, v.stages};
}

}  // namespace

// Every (variant, K split) the streaming kernel offers for the shape: row
// blocks of 16, 32 or 64 up to M, each variant at every distinct split of
// >= 4 ring steps per workgroup (as i8s_plan searches them).
int int8_configs(int M, int N, int K, pk_config *out, int cap) {
  if (M <= 0 || N <= 0 || K <= 0 || !i8s_shape_ok(M, N, K)) return 0;
  const int ksteps = K / I8S_KSTEP;
  const int mt_max = M <= 16 ? 1 : M <= 32 ? 2 : 4;
  int n = 0;
  for (const I8sVariant &v : kI8s) {
    if (v.mt > mt_max) continue;
    int last = -1;
    static const int kSplits[] = {1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16, 20, 24, 28, 32};
    for (int s : kSplits) {
      const int split_steps = (ksteps + s - 1) / s;
      if (s > 1 && split_steps < 4) break;
      if (split_steps == last) continue;
      last = split_steps;
      if (n < cap && out) out[n] = i8s_config(v, split_steps);
      ++n;
      if (aliased_split(s, split_steps, N)) {  // what i8s_plan takes instead
        if (n < cap && out) out[n] = i8s_config(v, split_steps + 1);
        ++n;
      }
    }
  }
  return n;
}

bool int8_default(int M, int N, int K, pk_config *out) {
  I8sPlan p;
  if (!i8s_plan(M, N, K, nullptr, device_cus(), p)) return false;
  *out = i8s_config(*p.v, p.split_steps);
  return true;
}

// Workspace for the built-in choice, whichever kernel the pointers' alignment
// leads to.
size_t int8_workspace_bytes(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  size_t need = 0;
  I8sPlan p;
  if (i8s_plan(M, N, K, nullptr, device_cus(), p)) need = i8s_workspace(p, M, N);
  const int s = choose_splits(M, N, K);
  return std::max(need, s > 1 ? (size_t)s * M * N * sizeof(float) : 0);
}

static int check_workspace(size_t need, size_t ws_bytes) {
  if (ws_bytes >= need) return PK_OK;
  set_error("int8 matmul: workspace of %zu bytes required, got %zu", need, ws_bytes);
  return PK_ERR_WORKSPACE;
}

static int check_workspace_alignment(const I8sPlan &plan, const void *ws) {
  if (!plan.v || plan.splits <= 1 || aligned16(ws)) return PK_OK;
  set_error("int8 matmul: workspace must be 16-byte aligned");
  return PK_ERR_WORKSPACE;
}

static int use_workspace(size_t need, void *&ws, size_t ws_bytes, hipStream_t st, WorkspaceLease &lease) {
  if (need == 0) return PK_OK;
  if (ws == nullptr) {
    int rc = library_workspace(need, st, lease);
    ws = lease.ptr;
    return rc;
  }
  return check_workspace(need, ws_bytes);
}

// Sum of g.splits partials and the epilogue.
static int reduce_run(int epi, const Int8Args &g, hipStream_t st) {
  const int64_t total = (int64_t)g.M * g.N;
  const bool vec = g.N % 8 == 0 && aligned16(g.partial) && aligned16(g.scale) && aligned16(g.C) &&
                   (epi != I8_RESID || aligned16(g.R));
  if (vec) {
    constexpr int T = PK_I8_REDUCE_THREADS;
    const int blocks = (int)std::min<int64_t>((total / 8 + T - 1) / T, 4096);
    if (epi == I8_NONE) int8_reduce8_kernel<I8_NONE><<<blocks, T, 0, st>>>(g);
    else if (epi == I8_GELU) int8_reduce8_kernel<I8_GELU><<<blocks, T, 0, st>>>(g);
    else int8_reduce8_kernel<I8_RESID><<<blocks, T, 0, st>>>(g);
  } else {
    const int blocks = (int)std::min<int64_t>((total + 255) / 256, 4096);
    if (epi == I8_NONE) int8_reduce_kernel<I8_NONE><<<blocks, 256, 0, st>>>(g);
    else if (epi == I8_GELU) int8_reduce_kernel<I8_GELU><<<blocks, 256, 0, st>>>(g);
    else int8_reduce_kernel<I8_RESID><<<blocks, 256, 0, st>>>(g);
  }
  PK_LAUNCH_CHECK("int8_reduce_kernel");
  return PK_OK;
}

// One product by a K-split stream or ring plan (16-byte aligned operands).
static int int8_plan_run(int epi, const uint16_t *A, const int8_t *W, const float *scale, uint16_t *C, const uint16_t *R,
                         const uint16_t *tab, int M, int N, int K, const Int8Plan &p, float *partial, hipStream_t st) {
  const KsPlan &ks = p.ks;
  const RingChoice &ring = p.ring;
  const int splits = ks.v ? ks.splits : ring.splits;
  if (ks.v) {
    const int units = ks.slices * ks.splits;
    const I8sArgs a{A, W, scale, partial, C, R, tab, M, N, K, ks.splits, ks.split_steps, units};
    ks.v->fn[epi](dim3(units, (M + 16 * ks.v->mt - 1) / (16 * ks.v->mt)), st, a);
    PK_LAUNCH_CHECK("int8_kstream_kernel");
  } else {
    const gk::GemmRingArgs a{{A, nullptr, C, nullptr, R, tab, M, N, K}, partial, ring.splits, ring.split_tiles, W, scale};
    kI8RingFn[ring.tile][epi](dim3(ring.units), st, a);
    PK_LAUNCH_CHECK("int8_ring_kernel");
  }
  return splits > 1 ? reduce_run(epi, Int8Args{A, W, scale, partial, C, R, tab, M, N, K, splits, 0}, st) : PK_OK;
}

int int8_run(int epi, const uint16_t *A, const int8_t *W, const float *scale, uint16_t *C,
             const uint16_t *R, int M, int N, int K, const pk_config *cfg, void *ws,
             size_t ws_bytes, hipStream_t st) {
  const uint16_t *tab = nullptr;
  if (epi == I8_GELU) {
    int rc = gelu_table(&tab);
    if (rc) return rc;
  }
  I8sPlan plan;
  if (!cfg && aligned16(A) && aligned16(W) && aligned16(scale) && aligned16(C) && (epi != I8_RESID || aligned16(R))) {
    // scratch is refused where the column-split or generic kernel's splits would not fit it
    auto base = [&] {
      return i8s_plan(M, N, K, nullptr, device_cus(), plan) ? i8s_workspace(plan, M, N) : generic_workspace(M, N, K, nullptr);
    };
    if (ws) {
      if (int rc = check_workspace(base(), ws_bytes)) return rc;
      if (int rc = check_workspace_alignment(plan, ws)) return rc;
    }
    // a caller's scratch as it is (launch_matmul_int8_noalloc's static buffer
    // is the cap for all, so that calls with and without it split alike),
    // library scratch as far as it can be had
    Int8Plan p;
    auto choose = [&](size_t scratch) {
      p = int8_plan(M, N, K, std::min(scratch, kInt8ScratchBytes));
      const int splits = p.ks.v ? p.ks.splits : p.ring.tile >= 0 ? p.ring.splits : 1;
      return splits > 1 ? (size_t)splits * M * N * sizeof(float) : 0;
    };
    WorkspaceLease lease;
    // unaligned scratch that was taken (the column-split kernel uses none) holds no partials
    const size_t part = choose(ws ? (aligned16(ws) ? ws_bytes : 0) : kInt8ScratchBytes);
    float *partial = static_cast<float *>(ws);
    if (part && !ws) {
      int rc = library_workspace(std::min(base(), part), part, st, lease);
      if (rc) return rc;
      partial = static_cast<float *>(lease.ptr);
      if (lease.bytes < part) choose(lease.bytes);
    }
    if (p.ks.v || p.ring.tile >= 0) return int8_plan_run(epi, A, W, scale, C, R, tab, M, N, K, p, partial, st);
  }
  const bool fast = aligned16(A) && aligned16(W) && aligned16(scale) && aligned16(C) &&
                    (epi != I8_RESID || aligned16(R)) && i8s_plan(M, N, K, cfg, device_cus(), plan);
  if (cfg && !fast) {
    set_error("int8 matmul: configuration {block_m %d, block_n %d, block_k %d, num_warps %d, "
              "vector_width %d, unroll %d, stages %d} not available for M=%d N=%d K=%d%s",
              cfg->block_m, cfg->block_n, cfg->block_k, cfg->num_warps, cfg->vector_width, cfg->unroll,
              cfg->shared_memory_stages, M, N, K,
              i8s_shape_ok(M, N, K) ? "" : " (the shape or operand alignment needs the generic kernel)");
    return PK_ERR_UNSUPPORTED;
  }
  Int8Args g{A, W, scale, nullptr, C, R, tab, M, N, K, 1, 0};
  WorkspaceLease lease;  // library scratch, held until the reduction is queued
  if (fast) {
    int rc = use_workspace(i8s_workspace(plan, M, N), ws, ws_bytes, st, lease);
    if (rc) return rc;
    if (int rc = check_workspace_alignment(plan, ws)) return rc;
    I8sArgs a{A, W, scale, static_cast<float *>(ws), C, R, tab, M, N, K,
              plan.splits, plan.split_steps, plan.slices * plan.splits};
    plan.v->fn[epi](dim3(plan.slices * plan.splits, plan.mblocks), st, a);
    PK_LAUNCH_CHECK("int8_stream_kernel");
    g.splits = plan.splits;
    g.partial = a.partial;
  } else {
    const size_t need = generic_workspace(M, N, K, &g);
    int rc = use_workspace(need, ws, ws_bytes, st, lease);
    if (rc) return rc;
    g.partial = static_cast<float *>(ws);
    const bool aligned = (N % 16 == 0) && (K % 8 == 0) && aligned16(A) && aligned16(W);
    dim3 grid((N + I8_BN - 1) / I8_BN, g.splits, (M + 15) / 16);
#define PK_I8(E)                                                                          \
  do {                                                                                    \
    if (aligned) int8_gemm_kernel<true, E><<<grid, I8_THREADS, 0, st>>>(g);               \
    else int8_gemm_kernel<false, E><<<grid, I8_THREADS, 0, st>>>(g);                      \
  } while (0)
    if (epi == I8_NONE) PK_I8(I8_NONE);
    else if (epi == I8_GELU) PK_I8(I8_GELU);
    else PK_I8(I8_RESID);
#undef PK_I8
    PK_LAUNCH_CHECK("int8_gemm_kernel");
  }
  return g.splits > 1 ? reduce_run(epi, g, st) : PK_OK;
}

// ---- the no-allocation variant of launch_matmul_int8 -------------------------
// Split-K partials go to this file-scope device array instead of library or
// caller memory.  Every GPU the library runs on holds its own copy (16 MiB)
// until the process ends.  In host code `scratch` names a host-side stand-in,
// not device memory: its device address is looked up per device with
// hipGetSymbolAddress once (int8_scratch_setup) and only that address is
// passed to kernels.
static __device__ __align__(256) float scratch[kInt8ScratchBytes / sizeof(float)];

namespace {
constexpr int kScratchDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kScratchDevices] = {};
}  // namespace

// Device address of the current device's `scratch` (looked up on the first
// call per device; later calls only read the table).
int int8_scratch_setup(void **out) {
  int dev = 0;
  PK_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kScratchDevices) {
    set_error("device ordinal %d out of range", dev);
    return PK_ERR_UNSUPPORTED;
  }
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) return hip_fail(e != hipSuccess ? e : hipErrorInvalidSymbol, "hipGetSymbolAddress(scratch)");
    g_scratch_ptr[dev] = p;
  }
  if (out) *out = g_scratch_ptr[dev];
  return PK_OK;
}

}  // namespace pk

using namespace pk;

extern "C" {

int launch_matmul_int8_noalloc(const uint16_t *A, const int8_t *Wq, const float *scale, uint16_t *C, int M, int N,
                               int K, void *stream) {
  PK_CHECK_ARG(A && Wq && scale && C, "launch_matmul_int8_noalloc: null tensor pointer");
  PK_CHECK_ARG(M >= 0 && N >= 0 && K > 0, "launch_matmul_int8_noalloc: invalid shape M=%d N=%d K=%d", M, N, K);
  if (M == 0 || N == 0) return PK_OK;
  const size_t need = int8_workspace_bytes(M, N, K);
  if (need > kInt8ScratchBytes) {
    set_error("launch_matmul_int8_noalloc: M=%d N=%d K=%d needs %zu bytes of split-K scratch, more than the %zu "
              "of the static buffer; use launch_matmul_int8 or pk_matmul_int8_ex with a workspace",
              M, N, K, need, kInt8ScratchBytes);
    return PK_ERR_WORKSPACE;
  }
  void *ws = nullptr;
  int rc = int8_scratch_setup(&ws);
  if (rc) return rc;
  // A caller workspace (the scratch) is never grown or replaced: int8_run
  // allocates nothing when it is given one.
  return int8_run(I8_NONE, A, Wq, scale, C, nullptr, M, N, K, nullptr, ws, kInt8ScratchBytes,
                  (hipStream_t)stream);
}

int launch_matmul_int8(const uint16_t *A, const int8_t *Wq, const float *scale, uint16_t *C,
                       int M, int N, int K, void *stream) {
  PK_CHECK_ARG(A && Wq && scale && C, "launch_matmul_int8: null tensor pointer");
  PK_CHECK_ARG(M >= 0 && N >= 0 && K > 0, "launch_matmul_int8: invalid shape M=%d N=%d K=%d", M, N, K);
  if (M == 0 || N == 0) return PK_OK;
  return int8_run(I8_NONE, A, Wq, scale, C, nullptr, M, N, K, nullptr, nullptr, 0, (hipStream_t)stream);
}

int pk_int8_default_config(int M, int N, int K, pk_config *out) {
  PK_CHECK_ARG(out && M > 0 && N > 0 && K > 0, "pk_int8_default_config: invalid argument");
  if (!int8_default(M, N, K, out)) {
    set_error("pk_int8_default_config: M=%d N=%d K=%d takes the generic kernel", M, N, K);
    return PK_ERR_UNSUPPORTED;
  }
  return PK_OK;
}

int pk_matmul_int8_ex(int epi, const uint16_t *A, const int8_t *Wq, const float *scale, uint16_t *C,
                      const uint16_t *R, int M, int N, int K, const pk_config *cfg,
                      void *workspace, size_t workspace_bytes, void *stream) {
  PK_CHECK_ARG(epi >= I8_NONE && epi <= I8_RESID, "pk_matmul_int8_ex: epilogue %d not in 0..2", epi);
  PK_CHECK_ARG(A && Wq && scale && C && (epi != I8_RESID || R), "pk_matmul_int8_ex: null tensor pointer");
  PK_CHECK_ARG(M >= 0 && N >= 0 && K > 0, "pk_matmul_int8_ex: invalid shape M=%d N=%d K=%d", M, N, K);
  if (M == 0 || N == 0) return PK_OK;
  return int8_run(epi, A, Wq, scale, C, R, M, N, K, cfg, workspace, workspace_bytes, (hipStream_t)stream);
}

int pk_int8_plan(int M, int N, int K, size_t scratch_bytes, pk_plan *out) {
  PK_CHECK_ARG(out && M > 0 && N > 0 && K > 0, "pk_int8_plan: invalid argument");
  const Int8Plan p = int8_plan(M, N, K, std::min(scratch_bytes, kInt8ScratchBytes));
  *out = pk_plan{PK_PLAN_TILE, 0, 0, 1, 0};
  if (p.ks.v) *out = pk_plan{PK_PLAN_STREAM, 16 * p.ks.v->mt, 16 * p.ks.v->nt, p.ks.splits, p.ks.split_steps};
  else if (p.ring.tile >= 0)
    *out = pk_plan{PK_PLAN_RING, 32 * kI8Ring[p.ring.tile].fm, 64 * kI8Ring[p.ring.tile].wn, p.ring.splits, p.ring.split_tiles};
  return PK_OK;
}

int pk_int8_plan_ex(int epi, const uint16_t *A, const int8_t *Wq, const float *scale, uint16_t *C, const uint16_t *R,
                    int M, int N, int K, const pk_plan *plan, void *workspace, size_t workspace_bytes, void *stream) {
  PK_CHECK_ARG(epi >= I8_NONE && epi <= I8_RESID, "pk_int8_plan_ex: epilogue %d not in 0..2", epi);
  PK_CHECK_ARG(A && Wq && scale && C && plan && (epi != I8_RESID || R), "pk_int8_plan_ex: null pointer");
  PK_CHECK_ARG(M > 0 && N > 0 && K > 0 && plan->splits >= 1, "pk_int8_plan_ex: invalid shape or plan");
  const uint16_t *tab = nullptr;
  if (epi == I8_GELU)
    if (int rc = gelu_table(&tab)) return rc;
  const int ksteps = (K + 63) / 64;  // of both kernels
  const int steps = (ksteps + plan->splits - 1) / plan->splits, splits = (ksteps + steps - 1) / steps;
  const size_t part = splits > 1 ? (size_t)splits * M * N * sizeof(float) : 0;
  if (part && (workspace_bytes < part || !aligned16(workspace))) {
    set_error("pk_int8_plan_ex: %zu aligned bytes of workspace required, got %zu", part, workspace_bytes);
    return PK_ERR_WORKSPACE;
  }
  Int8Plan p;
  if (aligned16(A) && aligned16(Wq) && aligned16(scale) && aligned16(C) && (epi != I8_RESID || aligned16(R)) &&
      ring_shape_ok(N, K, 1)) {
    if (plan->kernel == PK_PLAN_STREAM) {
      for (const KsVariant &v : kI8k)
        if (16 * v.mt == plan->block_m && 16 * v.nt == plan->block_n)
          p.ks = KsPlan{&v, splits, steps, (N + 16 * v.nt - 1) / (16 * v.nt)};
    } else if (plan->kernel == PK_PLAN_RING) {
      for (int i = 0; i < (int)(sizeof kI8Ring / sizeof kI8Ring[0]); ++i) {
        const int64_t units = (((int64_t)M + 32 * kI8Ring[i].fm - 1) / (32 * kI8Ring[i].fm)) *
                              (((int64_t)N + 64 * kI8Ring[i].wn - 1) / (64 * kI8Ring[i].wn)) * splits;
        if (32 * kI8Ring[i].fm == plan->block_m && 64 * kI8Ring[i].wn == plan->block_n && units <= INT32_MAX / 2)
          p.ring = RingChoice{i, splits, steps, (int)units, 0};
      }
    }
  }
  if (p.ks.v || p.ring.tile >= 0)
    return int8_plan_run(epi, A, Wq, scale, C, R, tab, M, N, K, p, static_cast<float *>(workspace), (hipStream_t)stream);
  set_error("pk_int8_plan_ex: kernel %d with %d x %d blocks does not take M=%d N=%d K=%d with these operands",
            plan->kernel, plan->block_m, plan->block_n, M, N, K);
  return PK_ERR_UNSUPPORTED;
}

size_t pk_decode_mlp_int8_workspace_size(int M, int d, int F) {
  if (M <= 0 || d <= 0 || F <= 0) return 0;  // no launch takes a workspace
  auto up = [](size_t v) { return (v + 255) & ~size_t(255); };
  const size_t p = std::max(int8_workspace_bytes(M, F, d), int8_workspace_bytes(M, d, F));
  return up((size_t)M * F * 2) + up(p);
}

int launch_decode_mlp_int8(const uint16_t *x, const int8_t *W1q, const float *s1,
                           const int8_t *W2q, const float *s2, uint16_t *out, int M, int d, int F,
                           void *workspace, size_t workspace_bytes, void *stream) {
  PK_CHECK_ARG(x && W1q && s1 && W2q && s2 && out, "launch_decode_mlp_int8: null tensor pointer");
  PK_CHECK_ARG(M >= 0 && d > 0 && F > 0, "launch_decode_mlp_int8: invalid shape");
  if (M == 0) return PK_OK;
  const size_t need = pk_decode_mlp_int8_workspace_size(M, d, F);
  if (!workspace || workspace_bytes < need) {
    set_error("launch_decode_mlp_int8: workspace of %zu bytes required, got %zu", need,
              workspace_bytes);
    return PK_ERR_WORKSPACE;
  }
  hipStream_t st = (hipStream_t)stream;
  const size_t hbytes = ((size_t)M * F * 2 + 255) & ~size_t(255);
  uint16_t *h = static_cast<uint16_t *>(workspace);
  void *part = static_cast<char *>(workspace) + hbytes;
  const size_t part_bytes = workspace_bytes - hbytes;
  int rc = int8_run(I8_GELU, x, W1q, s1, h, nullptr, M, F, d, nullptr, part, part_bytes, st);
  if (rc) return rc;
  return int8_run(I8_RESID, h, W2q, s2, out, x, M, d, F, nullptr, part, part_bytes, st);
}

}  // extern "C"
