// gemm.hip -- bf16 MFMA GEMM for gfx950 with fused epilogues.
//
// C[M,N] = A[M,K] @ B[K,N] with A K-contiguous and B N-contiguous (the
// reference layouts, kernels/cpu/cpu_reference.cpp:64-78), fp32 accumulation on
// v_mfma_f32_32x32x16_bf16.  Per workgroup a BM x BN tile; WM x WN waves, each
// owning a (BM/WM) x (BN/WN) sub-tile of 32x32 MFMA blocks.  A and B k-tiles of
// 64 are staged through LDS, double-buffered with one barrier per k-tile:
//   - A rows (128 B) are stored with 16-byte chunks XOR-swizzled by
//     (row >> 1) & 7, read as one ds_read_b128 per MFMA A-operand;
//   - B rows keep the global N-contiguous order (16-byte chunks swizzled by
//     k), and the MFMA B-operand (8 consecutive k of one column) is assembled
//     by two ds_read_b64_tr_b16 transpose reads, so no pre-packed weights and
//     no register transposes are needed.
// Workgroups are remapped so each XCD gets a contiguous band of tiles, rastered
// in groups of tile-rows for L2 reuse.
//
// Epilogues reproduce the golden per-stage bf16 rounding
// (tests/golden/golden.py:48-66, kernels/cpu/cpu_reference.cpp:92-105):
//   EPI_NONE        c = bf16(acc)
//   EPI_BIAS_GELU   c = gelu(bf16(bf16(acc) + bias[n]))      (exact GELU, gelu_bits)
//   EPI_BIAS_RESID  c = bf16(bf16(bf16(acc) + bias[n]) + R[m,n])
//   EPI_RESID       c = bf16(bf16(acc) + R[m,n])
#include <type_traits>

#include "gemm_kernels.hpp"
#include "gemm_plan.hpp"
#include "gemm_odd.hpp"
#include "gemm_ring.hpp"

namespace pk {


namespace {

using namespace gk;

// The kernels, as the library launches them (bodies in gemm_kernels.hpp).
template <int BM, int BN, int WM, int WN, int EPI, bool ALIGNED>
__global__ __launch_bounds__(WM *WN * 64) void gemm_kernel(GemmArgs g) {
  gemm_reg_body<BM, BN, WM, WN, EPI, ALIGNED>(g);
}

template <int EPI, int STAGES, int W = G2_WAVES, int WNN = G2_WAVES_N>
__global__ __launch_bounds__(W * 64, 1) void gemm_dma_kernel(GemmArgs g) {
  gemm_dma_body<EPI, STAGES, W, WNN>(g);
}

template <int NT, int MT, int WK, int STAGES, int EPI>
__global__ __launch_bounds__(WK * 64) void gemm_stream_kernel(GemmStreamArgs a) {
  gemm_stream_body<NT, MT, WK, STAGES, EPI>(a);
}

template <int NT, int MT, int WK, int DEPTH>
__global__ __launch_bounds__(WK * 64, 1) void gemm_odd_kernel(GemmArgs g) {
  gemm_odd_body<NT, MT, WK, DEPTH>(g);
}
template <int FM, int WN, int STAGES, int EPI>
__global__ __launch_bounds__(GR_THREADS, 1) void gemm_ring_kernel(GemmRingArgs a) {
  gemm_ring_body<FM, WN, STAGES, EPI>(a);
}

constexpr int GS_REDUCE_THREADS = 128;
template <int EPI>
__global__ __launch_bounds__(GS_REDUCE_THREADS) void gemm_reduce_kernel(GemmArgs g, const float *partial, int splits) {
  gemm_reduce_body<EPI>(g, partial, splits);
}

template <int BM, int BN, int WM, int WN, int EPI>
int launch_tile(const GemmArgs &g, bool aligned, hipStream_t st) {
  const int tiles = ((g.M + BM - 1) / BM) * ((g.N + BN - 1) / BN);
  if (aligned)
    gemm_kernel<BM, BN, WM, WN, EPI, true><<<tiles, WM * WN * 64, 0, st>>>(g);
  else
    gemm_kernel<BM, BN, WM, WN, EPI, false><<<tiles, WM * WN * 64, 0, st>>>(g);
  PK_LAUNCH_CHECK("gemm_kernel");
  return PK_OK;
}

// The kernels map blockIdx.x to (tile row, tile column) and round M, N and K
// up to whole tiles in 32-bit arithmetic: each stays 1023 below INT32_MAX,
// and a grid of the smallest tile (bm x bn) within INT32_MAX workgroups.
int tile_grid_ok(int M, int N, int K, int bm, int bn, const char *name) {
  if (M > INT32_MAX - 1023 || N > INT32_MAX - 1023 || K > INT32_MAX - 1023) {
    set_error("%s: M=%d, N=%d or K=%d is within 1023 of INT32_MAX", name, M, N, K);
    return PK_ERR_UNSUPPORTED;
  }
  if ((((int64_t)M + bm - 1) / bm) * (((int64_t)N + bn - 1) / bn) <= INT32_MAX) return PK_OK;
  set_error("%s: M=%d x N=%d needs more than %d workgroups", name, M, N, INT32_MAX);
  return PK_ERR_UNSUPPORTED;
}

// Whether every operand and every row of it can be read and written in 16-byte
// vectors.
bool gemm_vec_ok(const GemmArgs &g) {
  return (g.K % 8 == 0) && (g.N % 8 == 0) && aligned16(g.A) && aligned16(g.B) && aligned16(g.C) &&
         (!g.R || aligned16(g.R)) && (!g.bias || aligned16(g.bias));
}

// Whether tile 0 runs the direct-to-LDS 256x256 kernel for these operands
// (otherwise the register-staged one).
bool gemm_dma_fits(const GemmArgs &g) {
  const bool offsets32 = (size_t)g.K * g.N * 2 < (size_t(1) << 31) &&
                         (size_t)G2_BM * g.K * 2 < (size_t(1) << 31);
  return gemm_vec_ok(g) && offsets32 && g.K % G2_BK == 0 && g.N >= 8;
}

template <int EPI>
int gemm_dispatch(const GemmArgs &g, int tile, hipStream_t st) {
  const bool aligned = (g.K % 8 == 0) && (g.N % 8 == 0) && aligned16(g.A) && aligned16(g.B);
  if (tile == 0 && gemm_dma_fits(g)) {
    const int tiles = ((g.M + G2_BM - 1) / G2_BM) * ((g.N + G2_BN - 1) / G2_BN);
    gemm_dma_kernel<EPI, 5><<<tiles, G2_THREADS, 0, st>>>(g);
    PK_LAUNCH_CHECK("gemm_dma_kernel");
    return PK_OK;
  }
  if (tile == 3) tile = 0;  // the 8-wave register-staged 256x256 kernel
  switch (tile) {
    case 0: return launch_tile<256, 256, 2, 4, EPI>(g, aligned, st);
    case 1: return launch_tile<128, 128, 2, 2, EPI>(g, aligned, st);
    default: return launch_tile<64, 64, 2, 2, EPI>(g, aligned, st);
  }
}

// ---- configurations in the tuning-cache vocabulary ------------------------
// Variants, in order of preference: the DMA ring at 5 and 4 stages, then the
// register-staged kernels.  vector_width 8 needs K % 8 == 0, N % 8 == 0 and
// 16-byte aligned operands; 1 is the element-wise load path.
enum GemmVariant { GV_DMA5, GV_DMA4, GV_REG256, GV_REG128, GV_REG64, GV_COUNT };

pk_config gemm_variant_config(int v, int vw) {
  switch (v) {
    case GV_DMA5: return pk_config{G2_BM, G2_BN, G2_BK, G2_THREADS / 64, 8, G2_BK / 16, 5};
    case GV_DMA4: return pk_config{G2_BM, G2_BN, G2_BK, G2_THREADS / 64, 8, G2_BK / 16, 4};
    case GV_REG256: return pk_config{256, 256, BK, 8, vw, BK / 16, 2};
    case GV_REG128: return pk_config{128, 128, BK, 4, vw, BK / 16, 2};
    default: return pk_config{64, 64, BK, 4, vw, BK / 16, 2};
  }
}

bool gemm_dma_shape_ok(int N, int K) {
  return K % G2_BK == 0 && N % 8 == 0 && N >= 8 && (size_t)K * N * 2 < (size_t(1) << 31) &&
         (size_t)G2_BM * K * 2 < (size_t(1) << 31);
}

bool cfg_matches(const pk_config &req, const pk_config &c) {
  return (!req.block_m || req.block_m == c.block_m) && (!req.block_n || req.block_n == c.block_n) &&
         (!req.block_k || req.block_k == c.block_k) && (!req.num_warps || req.num_warps == c.num_warps) &&
         (!req.vector_width || req.vector_width == c.vector_width) && (!req.unroll || req.unroll == c.unroll) &&
         (!req.shared_memory_stages || req.shared_memory_stages == c.shared_memory_stages);
}

template <int EPI>
int gemm_launch_variant(const GemmArgs &g, int v, bool vec, hipStream_t st) {
  switch (v) {
    case GV_DMA5:
      gemm_dma_kernel<EPI, 5><<<((g.M + G2_BM - 1) / G2_BM) * ((g.N + G2_BN - 1) / G2_BN), G2_THREADS, 0, st>>>(g);
      PK_LAUNCH_CHECK("gemm_dma_kernel");
      return PK_OK;
    case GV_DMA4:
      gemm_dma_kernel<EPI, 4><<<((g.M + G2_BM - 1) / G2_BM) * ((g.N + G2_BN - 1) / G2_BN), G2_THREADS, 0, st>>>(g);
      PK_LAUNCH_CHECK("gemm_dma_kernel");
      return PK_OK;
    case GV_REG256: return launch_tile<256, 256, 2, 4, EPI>(g, vec, st);
    case GV_REG128: return launch_tile<128, 128, 2, 2, EPI>(g, vec, st);
    default: return launch_tile<64, 64, 2, 2, EPI>(g, vec, st);
  }
}

// ---- decode-sized calls (gemm_stream.hpp) -----------------------------------
// The streaming kernel's variants, by slice width (16 * nt columns) and rows
// (16 * mt), with the fewest waves and ring stages that keep the rate: two
// waves stream faster than four or eight, since the rows in flight then span
// fewer DRAM pages ([16, 16384, 4096] 24.1 us with 2 waves of 3 stages, 26.7
// with 4, 26.8 with 8; 4 waves of 6 stages 27.4).  `rate` is the weight bytes
// per ns one workgroup draws, fitted to [16-64, N, K] for N 512-28672, K
// 512-16384 (narrow slices read short runs: 32 bytes per weight row at nt 1).
struct StreamVariant {
  int nt, mt;
  double rate;
  void (*fn[4])(dim3, hipStream_t, const GemmStreamArgs &);
};
template <int NT, int MT, int WK, int STAGES, int EPI>
void stream_launch(dim3 grid, hipStream_t st, const GemmStreamArgs &a) {
  gemm_stream_kernel<NT, MT, WK, STAGES, EPI><<<grid, WK * 64, 0, st>>>(a);
}
#define PK_GS(NT, MT, WK, S, RATE)                                                                    \
  {                                                                                                   \
    NT, MT, RATE, {                                                                                   \
      stream_launch<NT, MT, WK, S, EPI_NONE>, stream_launch<NT, MT, WK, S, EPI_BIAS_GELU>,            \
          stream_launch<NT, MT, WK, S, EPI_BIAS_RESID>, stream_launch<NT, MT, WK, S, EPI_RESID>       \
    }                                                                                                 \
  }
const StreamVariant kStream[] = {
    PK_GS(4, 1, 2, 3, 30.0), PK_GS(8, 1, 2, 2, 45.0), PK_GS(2, 1, 2, 4, 16.0), PK_GS(1, 1, 4, 4, 10.0),
    PK_GS(4, 2, 2, 3, 27.0), PK_GS(8, 2, 2, 2, 40.0), PK_GS(2, 2, 2, 4, 14.5), PK_GS(1, 2, 4, 4, 9.0),
    PK_GS(4, 4, 2, 3, 22.0), PK_GS(8, 4, 2, 3, 33.0), PK_GS(2, 4, 4, 3, 11.0), PK_GS(1, 4, 4, 4, 7.5),
};
#undef PK_GS
constexpr int kStreamRows = 64;

struct StreamPlan {
  const StreamVariant *v = nullptr;
  int splits = 1, split_steps = 0, slices = 0;
};

// Whether the streaming kernel takes the shape (operands 16-byte aligned): its
// buffer descriptors and lane offsets hold both operands in 32 bits.
bool stream_shape_ok(int M, int N, int K) {
  return M <= kStreamRows && N % 8 == 0 && K % 8 == 0 && (size_t)K * N * 2 < (size_t(1) << 31) &&
         (size_t)M * K * 2 < (size_t(1) << 31);
}

// Slice width and K splits by a time model (us) fitted to the same sweep: 3
// for the launch, the larger of the memory time of all weights (6.4 TB/s; A's
// own loads cost a part of the weights' per byte) and of the busiest CU's
// units, and for a split 2.5 for the reduction's launch plus its partials at 5
// TB/s.  Grids between one and two and a half workgroups per CU stream slower
// ([16, 28672, 8192] 75.8 us with 224 units, 82.5 with 448, 80.5 with 672), and
// so do split slices of 128-byte runs.  Rows of N * 2 bytes that do not start
// on 128-byte lines share lines between slices: the wide slice then streams at
// 0.9, the others at 0.72 ([8, 50256, 2048]: 44 us with 128 columns, 59 with
// 64).  Four or more splits whose starts lie a multiple of 16 MB apart meet in
// the same memory channels, so such a split is one step longer ([16, 4096,
// 16384] in 8: 29.0 -> 27.1 us).  Splits use at most `scratch` bytes.
bool stream_plan(int M, int N, int K, size_t scratch, StreamPlan &best) {
  if (!stream_shape_ok(M, N, K)) return false;
  const int mt = M <= 16 ? 1 : M <= 32 ? 2 : 4;
  const int ksteps = (K + GS_KSTEP - 1) / GS_KSTEP;
  double best_us = 0;
  for (const StreamVariant &v : kStream) {
    if (v.mt != mt) continue;
    const int nb = 16 * v.nt, slices = (N + nb - 1) / nb;
    const double a_share = 1.0 + (v.mt == 4 ? 0.45 : 0.35) * (v.mt - 1) / v.nt;
    const double line = N % 64 == 0 ? 1.0 : v.nt == 8 ? 0.9 : 0.72;
    for (int s : {1, 2, 3, 4, 5, 6, 8, 10, 12, 14, 16}) {
      int steps = (ksteps + s - 1) / s;
      if (s > 1 && steps < 8) break;
      if (s >= 4 && (size_t)steps * GS_KSTEP * N * 2 % (size_t(16) << 20) == 0) ++steps;
      const int splits = (ksteps + steps - 1) / steps;
      const size_t part = splits > 1 ? (size_t)splits * M * N * sizeof(float) : 0;
      if (part > scratch) break;
      const int64_t units = (int64_t)slices * splits;
      const double rounds = std::ceil(units / 256.0);
      const double grid = units <= 256 ? 1.0 : units < 640 ? 1.2 : 1.04;
      const double hbm = (double)N * K * 2 * a_share * grid * (v.nt == 4 && splits > 1 ? 1.1 : 1.0) / 6.4e6;
      double us = 3.0 + std::max(hbm, rounds * steps * GS_KSTEP * nb * 2 / (v.rate * 1e3)) / line;
      if (splits > 1) us += 2.5 + 2.0 * part / 5e6;
      if (!best.v || us < best_us * (1 - 1e-9)) {
        best_us = us;
        best = StreamPlan{&v, splits, steps, slices};
      }
    }
  }
  return best.v != nullptr;
}

int reduce_run(int epi, const GemmArgs &g, const float *partial, int splits, hipStream_t st) {
  const int64_t items = (int64_t)g.M * g.N / 8;
  const int blocks = (int)std::min<int64_t>((items + GS_REDUCE_THREADS - 1) / GS_REDUCE_THREADS, 4096);
  switch (epi) {
    case EPI_NONE: gemm_reduce_kernel<EPI_NONE><<<blocks, GS_REDUCE_THREADS, 0, st>>>(g, partial, splits); break;
    case EPI_BIAS_GELU: gemm_reduce_kernel<EPI_BIAS_GELU><<<blocks, GS_REDUCE_THREADS, 0, st>>>(g, partial, splits); break;
    case EPI_BIAS_RESID: gemm_reduce_kernel<EPI_BIAS_RESID><<<blocks, GS_REDUCE_THREADS, 0, st>>>(g, partial, splits); break;
    default: gemm_reduce_kernel<EPI_RESID><<<blocks, GS_REDUCE_THREADS, 0, st>>>(g, partial, splits); break;
  }
  PK_LAUNCH_CHECK("gemm_reduce_kernel");
  return PK_OK;
}

int stream_run(int epi, const GemmArgs &g, const StreamPlan &p, void *scratch, hipStream_t st) {
  const GemmStreamArgs a{g, static_cast<float *>(scratch), p.splits, p.split_steps, p.slices};
  p.v->fn[epi](dim3(p.slices * p.splits, (g.M + 16 * p.v->mt - 1) / (16 * p.v->mt)), st, a);
  PK_LAUNCH_CHECK("gemm_stream_kernel");
  return p.splits > 1 ? reduce_run(epi, g, a.partial, p.splits, st) : PK_OK;
}

// ---- few rows and weights without 16-byte rows (gemm_odd.hpp) ---------------
// At most kStreamRows rows of A in whole 16-byte chunks; B and C at any element.
// Against the 64 x 64 tiles with element loads (us, rotating weights): [1, 50257,
// 2048] 251 / 45.5, [64, 50257, 4096] 580 / 115, [16, 12001, 4096] 261 / 27.6, [8,
// 5003, 2048] 99 / 9.1, [64, 2101, 512] 26.1 / 12.4.  Wide slices share fewer
// lines at their edges and are taken where they still fill the chip and K has
// more than a k-step or two ([22, 20770, 8] 4.9 us on tiles, 6.6 wide, 5 narrow);
// above 32 rows such a K leaves mostly the stores of single outputs, at which the
// tiles are faster ([51, 25172, 8] 5.9 / 9.7, [43, 59653, 16] 11.9 / 16.8).
bool odd_ok(const GemmArgs &g) {
  return g.M <= kStreamRows && g.K % 8 == 0 && g.N >= 8 && aligned16(g.A) && (size_t)g.K * g.N * 2 < (size_t(1) << 31) &&
         (g.M <= 32 || g.N <= 64 * 128 || g.K >= 64);
}
template <int MT>
int odd_run(const GemmArgs &g, hipStream_t st) {
  if (g.N >= 128 * 160 && g.K >= 64) gemm_odd_kernel<8, MT, 4, 3><<<(g.N + 127) / 128, 256, 0, st>>>(g);
  else if (g.N >= 64 * 128 && g.K >= 64) gemm_odd_kernel<4, MT, 8, 4><<<(g.N + 63) / 64, 512, 0, st>>>(g);
  else gemm_odd_kernel<2, MT, 8, 5><<<(g.N + 31) / 32, 512, 0, st>>>(g);
  PK_LAUNCH_CHECK("gemm_odd_kernel");
  return PK_OK;
}
int odd_run(const GemmArgs &g, hipStream_t st) {
  return g.M <= 16 ? odd_run<1>(g, st) : g.M <= 32 ? odd_run<2>(g, st) : odd_run<4>(g, st);
}

// ---- prompt-sized calls (gemm_ring.hpp) -------------------------------------
using RingLaunch = void (*)(dim3, hipStream_t, const GemmRingArgs &);
template <int FM, int WN, int STAGES, int EPI>
void ring_launch(dim3 grid, hipStream_t st, const GemmRingArgs &a) {
  gemm_ring_kernel<FM, WN, STAGES, EPI><<<grid, GR_THREADS, 0, st>>>(a);
}
#define PK_GR(FM, WN, S)                                                            \
  {                                                                                 \
    ring_launch<FM, WN, S, EPI_NONE>, ring_launch<FM, WN, S, EPI_BIAS_GELU>,        \
        ring_launch<FM, WN, S, EPI_BIAS_RESID>, ring_launch<FM, WN, S, EPI_RESID>   \
  }
const RingTile kRing[] = {{2, 2, 0.27}, {3, 2, 0.375}, {4, 2, 0.44}, {3, 4, 0.67}, {4, 4, 0.75}, {5, 4, 0.925}};
const RingLaunch kRingFn[][4] = {PK_GR(2, 2, 4), PK_GR(3, 2, 4), PK_GR(4, 2, 4),
                                 PK_GR(3, 4, 3), PK_GR(4, 4, 3), PK_GR(5, 4, 3)};
#undef PK_GR
constexpr int kRingWide = 3;  // 96 x 256

// Fitted to 60 shapes of 65-3850 rows, N 512-16384 and K 512-16384: its choice
// is within 0.7 % of the best variant in the geometric mean, 10 % at worst.
constexpr RingModel kRingModel{3.6, 1.7, 0.2, 9.5e6, 2.8, 4.6e6};
RingChoice ring_plan(int M, int N, int K, size_t scratch) {
  return ring_choose(kRing, (int)(sizeof kRing / sizeof kRing[0]), kRingModel, M, N, K, 2, scratch);
}

// The same model of the 256 x 256 kernel: 5.8 us, 2 per round and 0.5 per
// 32-deep k-tile, up to half as much again in launches of three rounds or more.
double dma_us(int M, int N, int K) {
  const double rounds = std::ceil((double)(((int64_t)M + 255) / 256) * (((int64_t)N + 255) / 256) / 256);
  return 5.8 + rounds * (2.0 + K / 32.0 * 0.5 * (1.0 + 0.5 * std::min(1.0, (rounds - 1) / 2)));
}

int ring_run(int epi, const GemmArgs &g, const RingChoice &p, void *scratch, hipStream_t st) {
  const GemmRingArgs a{g, static_cast<float *>(scratch), p.splits, p.split_tiles, nullptr, nullptr};
  kRingFn[p.tile][epi](dim3(p.units), st, a);
  PK_LAUNCH_CHECK("gemm_ring_kernel");
  return p.splits > 1 ? reduce_run(epi, g, a.partial, p.splits, st) : PK_OK;
}

// Largest tile that still gives at least ~one workgroup per CU.
// With the direct-to-LDS kernel (`dma`), 256x256 from 72 tiles up: even one
// round that leaves most CUs idle beats the 128x128 kernel's rounds (K 4096:
// [1280, 4096] 80 tiles 69.5 against 73.0 us, [2048, 4096] 128 tiles 72.1
// against 84.6, [3072, 3072] 144 tiles 73.4 against 137.0, [2048, 6144] 192
// tiles 87.4 against 141.4), while at 64 tiles one full round of 128x128
// tiles wins ([1024, 4096] 59.4 against 68.9 us).  The register-staged
// 256x256 kernel keeps the 200-tile threshold; 64x64 below 200 128x128
// tiles ([512, 4096] 41.4 against 57.4 us for 128x128).
int pick_tile(int M, int N, bool dma) {
  const long t256 = (((long)M + 255) / 256) * (((long)N + 255) / 256);
  const long t128 = (((long)M + 127) / 128) * (((long)N + 127) / 128);
  if (t256 >= (dma ? 72 : 200)) return 0;
  if (t128 >= 200) return 1;
  return 2;
}

// Whether the ring plan is faster than the tile of pick_tile (`tile`; `dma`: tile
// 0 is the direct-to-LDS kernel).  All figures without and with K split alike, us
// in a replayed graph, tile / ring.
//
// Against the 256 x 256 direct-to-LDS kernel: the two time models, and for GELU
// what the epilogues take in each round -- 1.5 us per 10 000 outputs of the ring's
// tile, which finishes them 32 rows at a time, 3 us and 1 per further round of the
// other ([4000, 2304, 256] 20.3 / 22.7, [10000, 4096, 512] 76.6 / 98.8 with GELU,
// 16.4 / 14.6 and 65.6 / 71.5 without; with these terms the choice is within
// 0.2 % of the better one over 366 shapes, 4.4 % without).
// Against the register-staged 64 x 64 kernel: it starts at 2.9 us (4.7 with GELU)
// and takes 0.42 per 64-deep k-step, one tile of the ring 4.4 (6.1) and 0.24: a
// deep ring to fill, waves' tiles to add.  So the ring needs some k: [300, 1024,
// K 128] 4.0 / 5.0, 256 4.8 / 5.5, 384 6.5 / 6.3, 512 7.0 / 6.8; with an epilogue
// that reads more, on a filled chip, less ([700, 4096, 128] + bias and residual
// 9.9 / 8.9), and where the columns fill a fraction of its tile, whose lanes then
// finish rows alone, more ([1555, 16, 512] + GELU 7.7 / 9.7).
// Against the register-staged 128 and 256 tiles it wins unless K is tiny and the
// epilogue empty ([4000, 1024, 64] 4.2 / 4.5, [4000, 16384, 8] 45.9 / 55).
bool ring_pays(int epi, int M, int N, int K, int tile, bool dma, const RingChoice &p) {
  if (tile == 0 && dma) {
    double ring = p.us, direct = dma_us(M, N, K);
    if (epi == EPI_BIAS_GELU) {
      const RingTile &t = kRing[p.tile];
      ring += std::ceil(p.units / 256.0) * 1.5e-4 * (32 * t.fm) * (64 * t.wn);
      direct += 2.0 + std::ceil((((int64_t)M + 255) / 256) * (((int64_t)N + 255) / 256) / 256.0);
    }
    return ring < direct;
  }
  if (tile == 2) {
    const int64_t units = (((int64_t)M + 63) / 64) * (((int64_t)N + 63) / 64);
    if (epi == EPI_NONE) return K >= (units <= 32 ? 448 : 352);
    if (epi == EPI_BIAS_GELU)
      return K >= (N <= 32 ? (units <= 32 ? 704 : 448) : units <= 64 ? 352 : units <= 256 ? 256 : 136);
    return K >= (N <= 32 ? (units <= 32 ? 512 : 384) : units <= 32 ? 320 : units <= 256 ? 224 : 136);
  }
  if (epi != EPI_NONE || K > 64) return true;
  return tile == 1 ? (((int64_t)M + 127) / 128) * (((int64_t)N + 127) / 128) > 496 : (int64_t)M * N < 24000000;
}

// Up to kStreamRows rows: whether the streaming kernel is faster than the 64 x 64
// tile, where pick_tile has that one.  It is, but for 33-64 rows on a second round
// of 64-column slices over a short K, whose wide slices leave half the waves
// ([64, 16448, 64] + bias and residual 6.0 / 7.2 us tile / stream, [64, 20000, 16] 3.9 / 4.5).
bool stream_pays(int epi, int M, int N, int K, int tile) {
  return M <= 32 || N <= 16384 || tile != 2 || K > (epi == EPI_NONE ? 256 : 512);
}
// 33-64 rows and more than 256 slices of 128 columns, a vocabulary head say: a
// second round of slices that no CU shares evenly streams at 3.5-4.2 TB/s, one
// round of the ring's 96 x 256 tiles at 4.6-4.9 ([64, 42496, 4544] 117 -> 78.7 us, 97
// on 256 x 256 tiles; [40, 50256, 2560] 56.9 -> 48.0).
bool ring_streams(int M, int N, int K) {
  return M > 32 && N > 32768 && N <= 65536 && K >= 2048 && ring_shape_ok(N, K, 2);
}

// The kernel of the built-in choice for vector-aligned operands and at most
// `scratch` bytes of partials: the streaming kernel up to kStreamRows rows,
// above it the ring kernel where it pays, else `tile` (`dma`: the 256 x 256
// direct-to-LDS kernel takes these operands).
struct GemmPlan {
  StreamPlan stream;
  RingChoice ring;
  int tile = 0;
  size_t part(int M, int N) const {
    const int s = stream.v ? stream.splits : ring.tile >= 0 ? ring.splits : 1;
    return s > 1 ? (size_t)s * M * N * sizeof(float) : 0;
  }
};
GemmPlan gemm_plan(int epi, int M, int N, int K, bool dma, size_t scratch) {
  static thread_local PlanMemo<GemmPlan> memo;
  return memo.get(M, N, K, scratch, epi << 1 | dma, [&] {
    GemmPlan p;
    p.tile = pick_tile(M, N, dma);
    if (M <= kStreamRows && ring_streams(M, N, K)) {
      p.ring = RingChoice{kRingWide, 1, (K + GR_BK - 1) / GR_BK, (N + 255) / 256, 0};
      return p;
    }
    if (M <= kStreamRows && stream_pays(epi, M, N, K, p.tile) && stream_plan(M, N, K, scratch, p.stream)) return p;
    p.ring = ring_plan(M, N, K, scratch);
    if (p.ring.tile >= 0 && !ring_pays(epi, M, N, K, p.tile, dma, p.ring)) p.ring = RingChoice{};
    return p;
  });
}

// Bytes of split partials the built-in choice wants for aligned operands (0:
// none); a caller with less scratch gets the best choice within it.
constexpr size_t kGemmScratchMax = size_t(64) << 20;
size_t gemm_scratch_bytes(int epi, int M, int N, int K) {
  constexpr int most = INT32_MAX - 1023;  // as tile_grid_ok
  if (M <= 0 || N <= 0 || K <= 0 || M > most || N > most || K > most) return 0;
  return gemm_plan(epi, M, N, K, gemm_dma_shape_ok(N, K), kGemmScratchMax).part(M, N);
}

}  // namespace

int gemm_configs(int M, int N, int K, pk_config *out, int cap) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const int vw = (K % 8 == 0 && N % 8 == 0) ? 8 : 1;
  int n = 0;
  for (int v = 0; v < GV_COUNT; ++v) {
    if ((v == GV_DMA5 || v == GV_DMA4) && !gemm_dma_shape_ok(N, K)) continue;
    if (out && n < cap) out[n] = gemm_variant_config(v, vw);
    ++n;
    if (vw == 8 && v >= GV_REG256) {  // the element-wise load path is always there too
      if (out && n < cap) out[n] = gemm_variant_config(v, 1);
      ++n;
    }
  }
  return n;
}

// The configuration of the tuning cache nearest to what gemm_run picks for
// 16-byte aligned operands: the streaming and ring kernels are no
// configurations, so where gemm_plan takes one this is the tile that a cache
// entry without a sweep would serve.
bool gemm_default(int M, int N, int K, pk_config *out) {
  if (M <= 0 || N <= 0 || K <= 0) return false;
  const int vw = (K % 8 == 0 && N % 8 == 0) ? 8 : 1;
  const bool dma = vw == 8 && gemm_dma_shape_ok(N, K);
  const int tile = pick_tile(M, N, dma);
  int v = tile == 0 ? GV_REG256 : tile == 1 ? GV_REG128 : GV_REG64;
  if (tile == 0 && dma) v = GV_DMA5;
  *out = gemm_variant_config(v, vw);
  return true;
}

int gemm_run_config(int epi, const uint16_t *A, const uint16_t *B, uint16_t *C, const uint16_t *bias,
                    const uint16_t *R, int M, int N, int K, const pk_config &req, hipStream_t st) {
  if (int rc = tile_grid_ok(M, N, K, 64, 64, "matmul")) return rc;
  GemmArgs g{A, B, C, bias, R, nullptr, M, N, K};
  const bool shape_vec = (K % 8 == 0) && (N % 8 == 0);
  const bool ptr_vec = aligned16(A) && aligned16(B);
  const bool ep_aligned = aligned16(C) && (!R || aligned16(R)) && (!bias || aligned16(bias));
  int chosen = -1;
  bool vec = false;
  for (int v = 0; v < GV_COUNT && chosen < 0; ++v) {
    if ((v == GV_DMA5 || v == GV_DMA4) && !(gemm_dma_shape_ok(N, K) && ptr_vec && ep_aligned)) continue;
    for (int vw : {8, 1}) {
      if (vw == 8 && !(shape_vec && ptr_vec)) continue;
      if (vw == 1 && (v == GV_DMA5 || v == GV_DMA4)) continue;
      if (cfg_matches(req, gemm_variant_config(v, vw))) {
        chosen = v;
        vec = vw == 8;
        break;
      }
    }
  }
  if (chosen < 0) {
    set_error("gemm: configuration {block_m %d, block_n %d, block_k %d, num_warps %d, vector_width %d, "
              "unroll %d, stages %d} not available for M=%d N=%d K=%d with these operand alignments",
              req.block_m, req.block_n, req.block_k, req.num_warps, req.vector_width, req.unroll,
              req.shared_memory_stages, M, N, K);
    return PK_ERR_UNSUPPORTED;
  }
  if (epi == EPI_BIAS_GELU) {
    int rc = gelu_table(&g.gelu_tab);
    if (rc) return rc;
  }
  switch (epi) {
    case EPI_NONE: return gemm_launch_variant<EPI_NONE>(g, chosen, vec, st);
    case EPI_BIAS_GELU: return gemm_launch_variant<EPI_BIAS_GELU>(g, chosen, vec, st);
    case EPI_BIAS_RESID: return gemm_launch_variant<EPI_BIAS_RESID>(g, chosen, vec, st);
    default: return gemm_launch_variant<EPI_RESID>(g, chosen, vec, st);
  }
}

int gemm_run(int epi, const uint16_t *A, const uint16_t *B, uint16_t *C, const uint16_t *bias,
             const uint16_t *R, int M, int N, int K, hipStream_t st, int tile = -1, void *scratch = nullptr,
             size_t scratch_bytes = 0) {
  if (int rc = tile_grid_ok(M, N, K, 64, 64, "matmul")) return rc;
  GemmArgs g{A, B, C, bias, R, nullptr, M, N, K};
  if (epi == EPI_BIAS_GELU) {
    int rc = gelu_table(&g.gelu_tab);
    if (rc) return rc;
  }
  if (tile < 0 && gemm_vec_ok(g)) {
    const GemmPlan p =
        gemm_plan(epi, M, N, K, gemm_dma_fits(g), aligned16(scratch) ? std::min(scratch_bytes, kGemmScratchMax) : 0);
    if (p.stream.v) return stream_run(epi, g, p.stream, scratch, st);
    if (p.ring.tile >= 0) return ring_run(epi, g, p.ring, scratch, st);
    tile = p.tile;
  }
  if (tile < 0 && epi == EPI_NONE && odd_ok(g)) return odd_run(g, st);
  if (tile < 0) tile = pick_tile(M, N, false);
  switch (epi) {
    case EPI_NONE: return gemm_dispatch<EPI_NONE>(g, tile, st);
    case EPI_BIAS_GELU: return gemm_dispatch<EPI_BIAS_GELU>(g, tile, st);
    case EPI_BIAS_RESID: return gemm_dispatch<EPI_BIAS_RESID>(g, tile, st);
    default: return gemm_dispatch<EPI_RESID>(g, tile, st);
  }
}

// The RMSNorm -> MatMul panel kernel (body in gemm_kernels.hpp).
__global__ __launch_bounds__(RQ_THREADS) void rmsnorm_panel_gemm_fast_kernel(PanelArgs a) {
  rmsnorm_panel_fast_body(a);
}

int rmsnorm_launch(const uint16_t *x, const uint16_t *w, uint16_t *y, int rows, int cols,
                   float eps, hipStream_t st);

// The whole-K panel kernel (x panel and W slice in LDS, 32 x 64 tiles) when K
// <= 832 and its grid is one round of at most 256 tiles: a latency kernel
// that reloads W for every 32 rows, so past one round RMSNorm into workspace
// and the GEMM win (K 768: M 128 8.4 against 13.2 us; M 192 14.9 against 13.3;
// M 1024 56.5 against 21.7; [4096, 4096] 215.8 against 36.5 us).  The
// double-buffered panel kernel (2 waves, 64-deep k-tiles, K <= 1536) lost at
// every measured shape (M 16-128, N 4096, K 1024: 25.9-34.9 against 14.0-15.2
// us; [4096, 4096, 1024] 1152.6 against 43.0 us) and was removed.
bool fast_panel_fits(int M, int N, int K) {
  const long tiles = (((long)M + RQ_BM - 1) / RQ_BM) * (((long)N + RQ_BN - 1) / RQ_BN);
  return K <= RQ_MAX_K && tiles <= 256 && (size_t)K * N * 2 < (size_t(1) << 31);
}

// The kernel fused_rmsnorm_matmul runs for aligned operands, as a config: the
// whole-K panel kernel where fast_panel_fits, otherwise row normalisation into
// workspace followed by the GEMM's own choice.
bool rmsnorm_matmul_config(int M, int N, int K, pk_config *out) {
  if (M <= 0 || N <= 0 || K <= 0) return false;
  const bool panel_ok = (K % BK == 0) && (N % 8 == 0);
  if (panel_ok && fast_panel_fits(M, N, K)) {
    *out = pk_config{RQ_BM, RQ_BN, K, RQ_THREADS / 64, 8, K / 16, 1};
    return true;
  }
  return gemm_default(M, N, K, out);
}

// The library workspace of a row normalisation followed by the GEMM: the rows,
// and behind them the GEMM's split partials where the workspace can hold them
// (*part: their bytes, 0 if not).
int normed_rows_workspace(int M, int N, int K, void *st, WorkspaceLease &lease, void **scratch, size_t *part) {
  const size_t row_bytes = ((size_t)M * K * 2 + 255) & ~size_t(255);
  *part = gemm_scratch_bytes(EPI_NONE, M, N, K);
  int rc = library_workspace((size_t)M * K * 2, *part ? row_bytes + *part : (size_t)M * K * 2, st, lease);
  if (rc) return rc;
  *scratch = static_cast<char *>(lease.ptr) + row_bytes;
  if (lease.bytes < row_bytes + *part) *part = 0;
  return PK_OK;
}

int gemm_planned(const uint16_t *A, const uint16_t *B, uint16_t *C, int M, int N, int K, void *scratch,
                 size_t scratch_bytes, void *st, bool *ran) {
  const GemmArgs g{A, B, C, nullptr, nullptr, nullptr, M, N, K};
  *ran = false;
  if (gemm_vec_ok(g)) {
    const GemmPlan p = gemm_plan(EPI_NONE, M, N, K, gemm_dma_fits(g), std::min(scratch_bytes, kGemmScratchMax));
    if (!p.stream.v && p.ring.tile < 0) return PK_OK;
  } else if (!odd_ok(g)) {
    return PK_OK;
  }
  *ran = true;
  return gemm_run(EPI_NONE, A, B, C, nullptr, nullptr, M, N, K, (hipStream_t)st, -1, scratch, scratch_bytes);
}

int fused_rmsnorm_matmul(const uint16_t *x, const uint16_t *gamma, const uint16_t *W, uint16_t *out,
                         int M, int N, int K, float eps, hipStream_t st, const char *name) {
  PK_CHECK_ARG(x && W && out, "%s: null tensor pointer", name);
  PK_CHECK_ARG(M >= 0 && N >= 0 && K > 0, "%s: invalid shape M=%d N=%d K=%d", name, M, N, K);
  if (M == 0 || N == 0) return PK_OK;
  if (int rc = tile_grid_ok(M, N, K, RQ_BM, RQ_BN, name)) return rc;
  const bool panel_ok = (K % BK == 0) && (N % 8 == 0) && aligned16(x) &&
                        aligned16(W) && (!gamma || aligned16(gamma));
  if (panel_ok && fast_panel_fits(M, N, K) && aligned16(out)) {
    const int tiles = ((M + RQ_BM - 1) / RQ_BM) * ((N + RQ_BN - 1) / RQ_BN);
    const size_t lds = pk_panel_lds_bytes(K);
    rmsnorm_panel_gemm_fast_kernel<<<tiles, RQ_THREADS, lds, st>>>(
        PanelArgs{x, gamma, W, out, M, N, K, 1.0f / (float)K, eps});
    PK_LAUNCH_CHECK(name);
    return PK_OK;
  }
  // Otherwise: normalise once into library workspace, then the plain GEMM.
  WorkspaceLease lease;  // held until the GEMM that reads the panel is queued
  void *scratch = nullptr;
  size_t part = 0;
  int rc = normed_rows_workspace(M, N, K, st, lease, &scratch, &part);
  if (rc) return rc;
  uint16_t *a = static_cast<uint16_t *>(lease.ptr);
  rc = rmsnorm_launch(x, gamma, a, M, K, eps, st);
  if (rc) return rc;
  return gemm_run(EPI_NONE, a, W, out, nullptr, nullptr, M, N, K, st, -1, scratch, part);
}

}  // namespace pk

using namespace pk;

extern "C" {

int launch_matmul(const uint16_t *A, const uint16_t *B, uint16_t *C, int M, int N, int K,
                  void *stream) {
  PK_CHECK_ARG(A && B && C, "launch_matmul: null tensor pointer");
  PK_CHECK_ARG(M >= 0 && N >= 0 && K >= 0, "launch_matmul: invalid shape");
  if (M == 0 || N == 0) return PK_OK;
  PK_CHECK_ARG(K > 0, "launch_matmul: K must be positive");
  return gemm_run(EPI_NONE, A, B, C, nullptr, nullptr, M, N, K, (hipStream_t)stream);
}

int launch_fused_matmul_bias_gelu(const uint16_t *a, const uint16_t *b, const uint16_t *bias,
                                  uint16_t *output, int M, int N, int K, void *stream) {
  PK_CHECK_ARG(a && b && bias && output, "launch_fused_matmul_bias_gelu: null tensor pointer");
  PK_CHECK_ARG(M >= 0 && N >= 0 && K > 0, "launch_fused_matmul_bias_gelu: invalid shape");
  if (M == 0 || N == 0) return PK_OK;
  return gemm_run(EPI_BIAS_GELU, a, b, output, bias, nullptr, M, N, K, (hipStream_t)stream);
}

int launch_fused_matmul_bias_residual(const uint16_t *a, const uint16_t *b, const uint16_t *bias,
                                      const uint16_t *residual, uint16_t *out, int M, int N, int K,
                                      void *stream) {
  PK_CHECK_ARG(a && b && residual && out, "launch_fused_matmul_bias_residual: null tensor pointer");
  PK_CHECK_ARG(M >= 0 && N >= 0 && K > 0, "launch_fused_matmul_bias_residual: invalid shape");
  if (M == 0 || N == 0) return PK_OK;
  return gemm_run(bias ? EPI_BIAS_RESID : EPI_RESID, a, b, out, bias, residual, M, N, K,
                  (hipStream_t)stream);
}

int launch_fused_rmsnorm_matmul(const uint16_t *input, const uint16_t *weight, uint16_t *output,
                                int M, int N, int K, float eps, void *stream) {
  return fused_rmsnorm_matmul(input, nullptr, weight, output, M, N, K, eps, (hipStream_t)stream,
                              "launch_fused_rmsnorm_matmul");
}

int launch_fused_rmsnorm_matmul_gamma(const uint16_t *x, const uint16_t *gamma, const uint16_t *W,
                                      uint16_t *out, int M, int N, int K, float eps, void *stream) {
  return fused_rmsnorm_matmul(x, gamma, W, out, M, N, K, eps, (hipStream_t)stream,
                              "launch_fused_rmsnorm_matmul_gamma");
}

// The normalised rows and the hidden activations: what launch_mlp_block cannot
// do without.  Workspace beyond it holds split partials.
static size_t mlp_rows_bytes(int M, int d, int F) {
  auto up = [](size_t v) { return (v + 255) & ~size_t(255); };
  return up((size_t)M * d * 2) + up((size_t)M * F * 2);
}

size_t pk_mlp_block_workspace_size(int M, int d, int F) {
  if (M <= 0 || d <= 0 || F <= 0) return 0;  // no launch takes a workspace
  return mlp_rows_bytes(M, d, F) + std::max(gemm_scratch_bytes(EPI_BIAS_GELU, M, F, d), gemm_scratch_bytes(EPI_BIAS_RESID, M, d, F));
}

int launch_mlp_block(const uint16_t *x, const uint16_t *gamma, const uint16_t *W1,
                     const uint16_t *b1, const uint16_t *W2, const uint16_t *b2, uint16_t *out,
                     int M, int d, int F, float eps, void *workspace, size_t workspace_bytes,
                     void *stream) {
  PK_CHECK_ARG(x && W1 && b1 && W2 && b2 && out, "launch_mlp_block: null tensor pointer");
  PK_CHECK_ARG(M >= 0 && d > 0 && F > 0, "launch_mlp_block: invalid shape");
  if (M == 0) return PK_OK;
  if (int rc = tile_grid_ok(M, std::max(d, F), std::max(d, F), 64, 64, "launch_mlp_block")) return rc;  // before any launch
  const size_t need = mlp_rows_bytes(M, d, F);
  if (!workspace || workspace_bytes < need) {
    set_error("launch_mlp_block: workspace of %zu bytes required, got %zu", need, workspace_bytes);
    return PK_ERR_WORKSPACE;
  }
  hipStream_t st = (hipStream_t)stream;
  uint16_t *a = static_cast<uint16_t *>(workspace);
  uint16_t *h = a + (((size_t)M * d * 2 + 255) & ~size_t(255)) / 2;
  int rc = rmsnorm_launch(x, gamma, a, M, d, eps, st);
  if (rc) return rc;
  void *scratch = static_cast<char *>(workspace) + need;
  rc = gemm_run(EPI_BIAS_GELU, a, W1, h, b1, nullptr, M, F, d, st, -1, scratch, workspace_bytes - need);
  if (rc) return rc;
  return gemm_run(EPI_BIAS_RESID, h, W2, out, b2, x, M, d, F, st, -1, scratch, workspace_bytes - need);
}

// Test/tuning hook: run one GEMM epilogue variant with an explicit tile choice
// (0: 256x256 -- the DMA-pipelined kernel when K % 32 == 0 and the operands
// are aligned, 1: 128x128, 2: 64x64, 3: the register-staged 256x256 kernel;
// -1: heuristic).
int pk_gemm_config_ex(int epi, const uint16_t *A, const uint16_t *B, uint16_t *C, const uint16_t *bias,
                      const uint16_t *R, int M, int N, int K, const pk_config *cfg, void *stream) {
  PK_CHECK_ARG(A && B && C, "pk_gemm_config_ex: null tensor pointer");
  PK_CHECK_ARG(M > 0 && N > 0 && K > 0, "pk_gemm_config_ex: invalid shape");
  PK_CHECK_ARG(epi >= 0 && epi <= 3, "pk_gemm_config_ex: epilogue %d not in 0..3", epi);
  PK_CHECK_ARG((epi != EPI_BIAS_GELU || bias) && (epi < EPI_BIAS_RESID || R),
               "pk_gemm_config_ex: epilogue %d needs its bias/residual operand", epi);
  if (!cfg) return gemm_run(epi, A, B, C, bias, R, M, N, K, (hipStream_t)stream);
  return gemm_run_config(epi, A, B, C, bias, R, M, N, K, *cfg, (hipStream_t)stream);
}

int pk_gemm_ex(int epi, const uint16_t *A, const uint16_t *B, uint16_t *C, const uint16_t *bias,
               const uint16_t *R, int M, int N, int K, int tile, void *stream) {
  PK_CHECK_ARG(A && B && C, "pk_gemm_ex: null tensor pointer");
  PK_CHECK_ARG(M > 0 && N > 0 && K > 0, "pk_gemm_ex: invalid shape");
  PK_CHECK_ARG(epi >= 0 && epi <= 3 && tile >= -1 && tile <= 3, "pk_gemm_ex: bad epi/tile");
  return gemm_run(epi, A, B, C, bias, R, M, N, K, (hipStream_t)stream, tile);
}

int pk_gemm_plan(int epi, int M, int N, int K, size_t scratch_bytes, pk_plan *out) {
  PK_CHECK_ARG(out && M > 0 && N > 0 && K > 0 && epi >= 0 && epi <= 3, "pk_gemm_plan: invalid argument");
  if (int rc = tile_grid_ok(M, N, K, 64, 64, "pk_gemm_plan")) return rc;
  *out = pk_plan{};
  out->splits = 1;
  if (K % 8 == 0 && N % 8 == 0) {
    const GemmPlan p = gemm_plan(epi, M, N, K, gemm_dma_shape_ok(N, K), std::min(scratch_bytes, kGemmScratchMax));
    out->block_m = out->block_n = p.tile == 0 ? 256 : p.tile == 1 ? 128 : 64;
    if (p.stream.v) {
      *out = pk_plan{PK_PLAN_STREAM, 16 * p.stream.v->mt, 16 * p.stream.v->nt, p.stream.splits, p.stream.split_steps};
      return PK_OK;
    }
    if (p.ring.tile >= 0) {
      const RingTile &t = kRing[p.ring.tile];
      *out = pk_plan{PK_PLAN_RING, 32 * t.fm, 64 * t.wn, p.ring.splits, p.ring.split_tiles};
      return PK_OK;
    }
    return PK_OK;
  }
  const int tile = pick_tile(M, N, false);
  out->block_m = out->block_n = tile == 0 ? 256 : tile == 1 ? 128 : 64;
  if (epi == EPI_NONE && odd_ok(GemmArgs{nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, M, N, K}))
    *out = pk_plan{PK_PLAN_ODD, 0, 0, 1, 0};
  return PK_OK;
}

int pk_gemm_plan_ex(int epi, const uint16_t *A, const uint16_t *B, uint16_t *C, const uint16_t *bias,
                    const uint16_t *R, int M, int N, int K, const pk_plan *plan, void *workspace,
                    size_t workspace_bytes, void *stream) {
  PK_CHECK_ARG(A && B && C && plan, "pk_gemm_plan_ex: null pointer");
  PK_CHECK_ARG(M > 0 && N > 0 && K > 0 && epi >= 0 && epi <= 3, "pk_gemm_plan_ex: invalid shape or epilogue");
  PK_CHECK_ARG(plan->splits >= 1, "pk_gemm_plan_ex: splits %d", plan->splits);
  if (int rc = tile_grid_ok(M, N, K, 64, 64, "pk_gemm_plan_ex")) return rc;
  GemmArgs g{A, B, C, bias, R, nullptr, M, N, K};
  if (epi == EPI_BIAS_GELU)
    if (int rc = gelu_table(&g.gelu_tab)) return rc;
  // the splits of the plan as the planners form them: whole k-steps, none empty
  const bool stream_kernel = plan->kernel == PK_PLAN_STREAM;
  const int ksteps = (K + (stream_kernel ? GS_KSTEP : GR_BK) - 1) / (stream_kernel ? GS_KSTEP : GR_BK);
  const int steps = (ksteps + plan->splits - 1) / plan->splits, splits = (ksteps + steps - 1) / steps;
  const size_t part = splits > 1 ? (size_t)splits * M * N * sizeof(float) : 0;
  if (part && (workspace_bytes < part || !aligned16(workspace))) {
    set_error("pk_gemm_plan_ex: %zu aligned bytes of workspace required, got %zu", part, workspace_bytes);
    return PK_ERR_WORKSPACE;
  }
  if (stream_kernel && gemm_vec_ok(g) && stream_shape_ok(M, N, K)) {
    for (const StreamVariant &v : kStream)
      if (16 * v.mt == plan->block_m && 16 * v.nt == plan->block_n)
        return stream_run(epi, g, StreamPlan{&v, splits, steps, (N + 16 * v.nt - 1) / (16 * v.nt)}, workspace,
                          (hipStream_t)stream);
  } else if (plan->kernel == PK_PLAN_RING && gemm_vec_ok(g) && ring_shape_ok(N, K, 2)) {
    for (int i = 0; i < (int)(sizeof kRing / sizeof kRing[0]); ++i) {
      const int64_t units = (((int64_t)M + 32 * kRing[i].fm - 1) / (32 * kRing[i].fm)) *
                            (((int64_t)N + 64 * kRing[i].wn - 1) / (64 * kRing[i].wn)) * splits;
      if (32 * kRing[i].fm == plan->block_m && 64 * kRing[i].wn == plan->block_n && units <= INT32_MAX / 2)
        return ring_run(epi, g, RingChoice{i, splits, steps, (int)units, 0}, workspace, (hipStream_t)stream);
    }
  }
  set_error("pk_gemm_plan_ex: kernel %d with %d x %d blocks does not take M=%d N=%d K=%d with these operands",
            plan->kernel, plan->block_m, plan->block_n, M, N, K);
  return PK_ERR_UNSUPPORTED;
}

}  // extern "C"
