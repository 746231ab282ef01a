// gemm_ring.hpp -- the bf16 GEMM of prompt-sized calls (more rows than
// gemm_stream.hpp takes, too few tiles for the 256 x 256 kernel to fill the
// chip): C[M,N] = A[M,K] @ B[K,N] with the epilogues of gemm_kernels.hpp.
//
// What bounds it: with one tile per CU, the latency of each k-step and the LDS
// traffic of a small tile.  The register-staged 128 x 128 kernel spends 1.3 us
// on a 64-deep k-step (load, wait, LDS store, barrier, reads, MFMA in series:
// [501, 8192, 2048] 43 us, 0.4 PFLOP/s).  Here k-tiles of 64 come through a
// STAGES-deep LDS ring filled by buffer_load ... lds, and the 8 waves split the
// tile WN ways along N and KG ways along K instead of along M: each wave owns
// BM x 64 outputs (FM x 2 MFMA blocks of 32 x 32) over the 16-row substeps
// kg, kg + KG, ... of every k-tile.  That keeps a wave's fragment reads at
// FM + 2 per 2 FM MFMAs -- a 2 x 4 grid of 64 x 32 outputs would need 3 per 2 --
// and two waves on every SIMD, and lets BM be any multiple of 32, so a ragged
// M pads little (777 rows: 5 x 160).  The KG partial tiles are added in LDS at
// the end, 32 rows at a time.
//
// One barrier per k-tile: iteration t waits for its own loads of tile t+1,
// passes the barrier (everyone's loads of t+1 landed, everyone's reads of tile
// t are done), then runs the MFMAs of tile t between the fragment reads of
// t+1 and the loads of tile t+STAGES into the slot of t.
//
// Measured (us, best tile against the best of the 64, 128 and 256 tiles): [501,
// 8192, 2048] 22.6 / 34.2, [501, 2048, 8192] 28.9 / 73.8 (K split in 4), [777,
// 12288, 4096] 73.6 / 87, [1024, 4096, 4096] 37.0 / 60.5, [128, 4096, 4096]
// 15.2 / 38.9, [1278, 16128, 4032] 148 / 201.  Timing-only builds of the 128 x
// 128 tile at [1024, 4096, 4096]: MFMA alone 25.7, loads alone 28.7, all 37.6, each
// with 7.9 of launch, first loads and epilogue.  Without those the tiles' 537 MB
// come at 26 TB/s, and half of the MFMA time runs beside them.  Counters: MFMA busy
// on 37 % of the cycles there, 50 % at [777, 12288, 4096], no bank conflicts.
//
// Like the streaming kernel it can split K over workgroups (fp32 partials,
// gemm_reduce_body, or int8_stream.hpp's reduction).  Needs K % 8 == 0, N % 8 == 0, 16-byte aligned A and B;
// rows, columns and k past the end are clamped onto valid memory, and the k
// past K zeroed in registers.
#pragma once

#include "gemm_stream.hpp"
#include "int8_stream.hpp"

namespace pk {
namespace gk {

constexpr int GR_BK = 64, GR_WAVES = 8, GR_THREADS = GR_WAVES * 64;

struct GemmRingArgs {
  GemmArgs g;
  float *partial;   // [splits][M][N] fp32, splits > 1
  int splits;
  int split_tiles;  // k-tiles per split
  const int8_t *W8;    // INT8: weights [K][N] and their per-column scale [N]
  const float *scale;  // (g.B and g.bias are then unused)
};

// Workgroup -> (split, tile row, tile column): each XCD takes a contiguous run
// of units, a split's tiles in groups of 8 tile rows.
__device__ __forceinline__ void ring_unit(int bid, int total, int tm, int tn, int &split, int &mt, int &nt) {
  const int b = xcd_unit(bid, total);
  split = b / (tm * tn);
  const int r = b - split * tm * tn;
  const int group = r / (8 * tn), first = group * 8;
  const int rows = min(tm - first, 8);
  const int in = r - first * tn;
  mt = first + in % rows;
  nt = in / rows;
}

// 32-byte-unit XOR of int8 weight row k: the 8 rows of 32 columns that one
// 32-lane pass of ds_read_b64_tr_b8 reads then cover all 64 banks once.
template <int BN>
__device__ __forceinline__ int swz_w8(int k) {
  return BN == 128 ? (k >> 1) & 3 : k & 7;
}

// INT8: the weights are int8, widened exactly to bf16 in registers; EPI is then
// an Int8Epi, applied to the sums times the column's scale.
template <int FM, int WN, int STAGES, int EPI, bool INT8 = false>
__device__ __forceinline__ void gemm_ring_body(const GemmRingArgs &a) {
  constexpr int KG = GR_WAVES / WN;          // k groups
  constexpr int SUB = 4 / KG;                // 16-k substeps of a k-tile per wave
  static_assert(KG * WN == GR_WAVES && SUB * KG == 4, "waves split N and K");
  constexpr int BM = 32 * FM, BN = 64 * WN;
  constexpr int WB1 = INT8 ? 1 : 2;          // bytes of a weight
  constexpr int BCH = BN * WB1 / 16;         // 16-byte chunks of a weight row
  constexpr int A_BYTES = BM * GR_BK * 2, STAGE = A_BYTES + GR_BK * BN * WB1;
  constexpr int NA = BM / 8, NB = BCH;       // 1 KiB loads per k-tile
  constexpr bool GELU = INT8 ? EPI == I8_GELU : EPI == EPI_BIAS_GELU;
  constexpr int HI = (NA + NB + 7) / 8, LO = (NA + NB) / 8;  // per wave: the first waves may have one more
  constexpr int HEAVY = (NA + NB) % 8;       // waves with HI loads (0: all have LO)
  constexpr int NM = 2 * FM, NU = FM + 2;    // MFMAs and fragment-read units per substep
  __shared__ __attribute__((aligned(1024))) uint8_t ring[STAGES * STAGE];
  const GemmArgs &g = a.g;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wid % WN, kg = wid / WN;
  const int tm = (g.M + BM - 1) / BM, tn = (g.N + BN - 1) / BN;
  int split, mt, nt;
  ring_unit(blockIdx.x, tm * tn * a.splits, tm, tn, split, mt, nt);
  const int m0 = mt * BM, n0 = nt * BN;
  const int ktiles = (g.K + GR_BK - 1) / GR_BK;
  const int kt0 = split * a.split_tiles;
  const int KT = min(ktiles, kt0 + a.split_tiles) - kt0;  // k-tiles of this unit
  const int k_tail = g.K - (ktiles - 1) * GR_BK;          // valid k of the matrix's last k-tile
  const bool ragged = k_tail < GR_BK && kt0 + KT == ktiles;

  // ---- loads: load i of a k-tile (i < NA: 8 rows of A; else rows of B) goes
  // to wave i % 8 as its load i / 8, with a loop-invariant lane offset and the
  // k-tile in the scalar offset
  const pk_u32x4 a_rsrc = rsrc_words(g.A + (size_t)m0 * g.K, (uint32_t)((size_t)min(g.M - m0, BM) * g.K * 2));
  const void *w_base = INT8 ? static_cast<const void *>(a.W8 + n0) : static_cast<const void *>(g.B + n0);
  const pk_u32x4 b_rsrc = rsrc_words(w_base, (uint32_t)(((size_t)g.K * g.N - n0) * WB1));
  constexpr int BROWS = 64 / BCH;  // rows of B per load
  const auto w_col = [](int r, int p) {  // column of physical chunk p of row r
    if constexpr (INT8) return 32 * ((p >> 1) ^ swz_w8<BN>(r)) + 16 * (p & 1);
    else return 8 * (p ^ swz_b<BN>(r));
  };
  uint32_t off[HI];
#pragma unroll
  for (int j = 0; j < HI; ++j) {
    const int i = 8 * j + wid;
    if (8 * j + 7 < NA || (8 * j < NA && i < NA)) {
      const int r = 8 * i + (lane >> 3);
      off[j] = (uint32_t)(min(r, g.M - 1 - m0) * g.K + 8 * ((lane & 7) ^ swz_a64(r))) * 2u;
    } else {
      const int r = (i - NA) * BROWS + lane / BCH;
      off[j] = (uint32_t)(r * g.N + min(w_col(r, lane % BCH), g.N - 16 / WB1 - n0)) * WB1;
    }
  }
  auto issue_one = [&](int slot, int t, int j) __attribute__((always_inline)) {
    const int i = 8 * j + wid;
    if (HEAVY && j == HI - 1 && wid >= HEAVY) return;
    uint8_t *dst = ring + slot * STAGE + 1024 * i;
    const int kt = kt0 + min(t, KT - 1);  // past the end: the last tile again, into a slot nobody reads
    const bool tail = ragged && kt == ktiles - 1;
    if (i < NA) {
      uint32_t o = off[j];
      if (tail) o -= 16u * max(0, ((lane & 7) ^ swz_a64(8 * i + (lane >> 3))) - (k_tail / 8 - 1));
      dma_lds16(a_rsrc, dst, o, (uint32_t)kt * (GR_BK * 2));
    } else {
      uint32_t o = off[j];
      if (tail) o -= WB1 * (uint32_t)g.N * max(0, (i - NA) * BROWS + lane / BCH - (k_tail - 1));
      dma_lds16(b_rsrc, dst, o, (uint32_t)kt * (GR_BK * WB1) * (uint32_t)g.N);
    }
  };
  auto issue = [&](int slot, int t) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < HI; ++j) issue_one(slot, t, j);
  };
  // at most n k-tiles and `more` of this wave's loads outstanding
  auto wait_tiles = [&](auto n_c, auto more_c) __attribute__((always_inline)) {
    constexpr int n = decltype(n_c)::value, more = decltype(more_c)::value;
    if (HEAVY == 0 || wid >= HEAVY) vm_wait<n * LO + more>();
    else vm_wait<n * HI + more>();
  };

  // ---- fragment reads: substep s of a slot, A blocks then B blocks
  const int grp = lane >> 4, gi = lane & 15, hi = lane >> 5;
  int a_rd[SUB], b_rd[SUB][2];
#pragma unroll
  for (int u = 0; u < SUB; ++u) {
    const int s = kg + KG * u, row = lane & 31;
    a_rd[u] = row * 128 + 16 * ((2 * s + hi) ^ swz_a64(row));
#pragma unroll
    for (int fn = 0; fn < 2; ++fn) {
      if constexpr (INT8) {
        const int k = 16 * s + 8 * hi + (gi >> 1);
        b_rd[u][fn] = A_BYTES + k * BN + 32 * ((wn * 2 + fn) ^ swz_w8<BN>(k)) + 16 * (grp & 1) + 8 * (gi & 1);
      } else {
        const int k = 16 * s + 8 * hi + (gi >> 2);
        const int col = wn * 64 + fn * 32 + 16 * (grp & 1) + 4 * (gi & 3);
        b_rd[u][fn] = A_BYTES + k * (2 * BN) + 16 * ((col >> 3) ^ swz_b<BN>(k)) + 2 * (col & 7);
      }
    }
  }
  struct Frag {
    bf16x8 a[FM], b[2];
    i8s::v2i32 w[2];  // INT8: the weights as read, widened to b by the substep that uses them
  };
  auto read_unit = [&](Frag &f, int slot, int u, int i) __attribute__((always_inline)) {
    const uint8_t *base = ring + slot * STAGE;
    if (i < 2) {
      const uint8_t *p = base + b_rd[u][i];
      if constexpr (INT8) {
        f.w[i] = __builtin_amdgcn_ds_read_tr8_b64_v2i32((i8s::lds_v2i32 *)p);
        return;
      }
      const i16x4 h0 = lds_read_tr(reinterpret_cast<const uint16_t *>(p));
      const i16x4 h1 = lds_read_tr(reinterpret_cast<const uint16_t *>(p + 4 * (2 * BN)));
      f.b[i] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(h0, h1, 0, 1, 2, 3, 4, 5, 6, 7));
    } else {
      f.a[i - 2] = lds_read_a(reinterpret_cast<const uint16_t *>(base + a_rd[u] + (i - 2) * 32 * 128));
    }
  };
  f32x16 acc[FM][2];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  // W as the first operand: lane l holds 4 consecutive columns of output row
  // 32 fm + l % 32.  INT8 takes a column block's MFMAs together, so that the
  // second block is widened between those of the first.
  auto mfma_one = [&](Frag &f, int i) __attribute__((always_inline)) {
    const int fm = INT8 ? i % FM : i >> 1, fn = INT8 ? i / FM : i & 1;
    if constexpr (INT8) {
      if (i == 0) f.b[0] = i8s::widen8(f.w[0]);
      if (i == 1) f.b[1] = i8s::widen8(f.w[1]);
    }
    acc[fm][fn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.b[fn], f.a[fm], acc[fm][fn], 0, 0, 0);
  };
  // the lane's 8 k of a substep lie past K on the last k-tile: zero both operands
  auto mask_tail = [&](Frag &f, int u, int t) __attribute__((always_inline)) {
    if (ragged && t == KT - 1 && 16 * (kg + KG * u) + 8 * hi >= k_tail) {
      const bf16x8 z = __builtin_bit_cast(bf16x8, u32x4{0, 0, 0, 0});
#pragma unroll
      for (int i = 0; i < FM; ++i) f.a[i] = z;
      if constexpr (!INT8) f.b[0] = f.b[1] = z;  // (an int8 weight is finite)
    }
  };

  // the GELU table, loaded ahead of the first DMA and copied to LDS at the end
  constexpr int TAB_W = (GELU_TABLE_SIZE + 1) / 2, TAB_PT = (TAB_W + GR_THREADS - 1) / GR_THREADS;
  uint32_t tab_pre[GELU ? TAB_PT : 1];
  if constexpr (GELU) {
#pragma unroll
    for (int j = 0; j < TAB_PT; ++j) {
      const int i = tid + j * GR_THREADS;
      tab_pre[j] = i < TAB_W ? reinterpret_cast<const uint32_t *>(g.gelu_tab)[i] : 0u;
    }
  }

  // ---- pipeline
  using Ahead = std::integral_constant<int, STAGES - 2>;
  constexpr int H1 = SUB == 1 ? LO : (HI + 1) / 2;  // loads of a k-tile's first part
#pragma unroll
  for (int t = 0; t < STAGES - 1; ++t) issue(t, t);
#pragma unroll
  for (int j = 0; j < H1; ++j) issue_one(STAGES - 1, STAGES - 1, j);
  wait_tiles(Ahead{}, std::integral_constant<int, H1>{});
  if constexpr (SUB == 1) {
#pragma unroll
    for (int j = H1; j < HI; ++j) issue_one(STAGES - 1, STAGES - 1, j);
  }
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");  // no LDS access moves above the barrier
  Frag f0, f1;
#pragma unroll
  for (int i = 0; i < NU; ++i) read_unit(f0, 0, 0, i);
  // MFMAs of one substep with the reads of the next one spread over them, and
  // loads [j0, j1) of k-tile lt behind every second MFMA
  auto substep = [&](Frag &f, Frag &nx, int nslot, int nu, int lslot, int lt, int j0, int j1)
      __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NM; ++i) {
      if (SUB > 1 && i < NU) read_unit(nx, nslot, nu, i);  // ahead of the MFMA: 3 % faster at SUB 2, slower at SUB 1
      mfma_one(f, i);
      if (SUB == 1 && i < NU) read_unit(nx, nslot, nu, i);
      if ((i & 1) == 1 && j0 + (i >> 1) < j1) issue_one(lslot, lt, j0 + (i >> 1));
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int j = j0 + NM / 2; j < j1; ++j) issue_one(lslot, lt, j);
  };
  auto sync = [&]() __attribute__((always_inline)) {
    lgkm_wait0();  // this wave's reads of the slot about to be refilled
    wait_tiles(Ahead{}, std::integral_constant<int, 0>{});
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  int slot = 0;
  auto next = [&](int s) __attribute__((always_inline)) { return s == STAGES - 1 ? 0 : s + 1; };
  auto tile1 = [&](Frag &f, Frag &nx, int t) __attribute__((always_inline)) {  // SUB == 1
    sync();
    mask_tail(f, 0, t);
    const int n = next(slot);
    substep(f, nx, n, 0, slot, t + STAGES, 0, HI);
    slot = n;
  };
  if constexpr (SUB == 1) {
    int t = 0;
    for (; t + 2 <= KT; t += 2) {
      tile1(f0, f1, t);
      tile1(f1, f0, t + 1);
    }
    if (t < KT) tile1(f0, f1, t);
  } else {
    // the loads of tile t+STAGES in two parts, behind the barrier of tile t
    // and in the first substep of t+1
    int prev = STAGES - 1;
    for (int t = 0; t < KT; ++t) {
      mask_tail(f0, 0, t);
      substep(f0, f1, slot, SUB - 1, prev, t + STAGES - 1, H1, HI);
      sync();
      mask_tail(f1, SUB - 1, t);
      const int n = next(slot);
      substep(f1, f0, n, 0, slot, t + STAGES, 0, H1);
      prev = slot;
      slot = n;
    }
  }
  vm_wait<0>();  // repeated tail loads may still be landing
  lgkm_wait0();
  __syncthreads();

  // ---- add the KG tiles of each column group in group order and finish, 32
  // rows a pass: every wave stores its 32 x 64 block, then each thread sums and
  // finishes 8 columns.  LD spreads the 16 rows of a 16-byte store over all banks.
  constexpr int LD = 68, WB = 32 * LD * 4;
  static_assert(GR_WAVES * WB + GELU_TABLE_SIZE * 2 + 16 <= STAGES * STAGE, "staging fits the ring");
  uint16_t *tab = reinterpret_cast<uint16_t *>(ring + GR_WAVES * WB);
  if constexpr (GELU) {
#pragma unroll
    for (int j = 0; j < TAB_PT; ++j)
      if (tid + j * GR_THREADS < TAB_W) reinterpret_cast<uint32_t *>(tab)[tid + j * GR_THREADS] = tab_pre[j];
  }
  float *mine = reinterpret_cast<float *>(ring + wid * WB);
#pragma unroll
  for (int fm = 0; fm < FM; ++fm) {
    if (fm) __syncthreads();  // the previous pass is read
#pragma unroll
    for (int fn = 0; fn < 2; ++fn)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<f32x4 *>(mine + (lane & 31) * LD + fn * 32 + 8 * q + 4 * hi) =
            f32x4{acc[fm][fn][4 * q], acc[fm][fn][4 * q + 1], acc[fm][fn][4 * q + 2], acc[fm][fn][4 * q + 3]};
    __syncthreads();
    constexpr int C8 = BN / 8;
#pragma unroll
    for (int it = 0; it < 32 * C8; it += GR_THREADS) {
      const int r = (it + tid) / C8, c = 8 * ((it + tid) % C8);
      const int m = m0 + 32 * fm + r, n = n0 + c;
      if (m >= g.M || n >= g.N) continue;
      const float *p = reinterpret_cast<const float *>(ring + (c / 64) * WB) + r * LD + c % 64;
      f32x4 v0 = *reinterpret_cast<const f32x4 *>(p), v1 = *reinterpret_cast<const f32x4 *>(p + 4);
#pragma unroll
      for (int k = 1; k < KG; ++k) {
        const float *q = p + k * WN * (WB / 4);
        v0 += *reinterpret_cast<const f32x4 *>(q);
        v1 += *reinterpret_cast<const f32x4 *>(q + 4);
      }
      if (a.splits > 1) {
        float *o = a.partial + ((size_t)split * g.M + m) * g.N + n;
        *reinterpret_cast<f32x4 *>(o) = v0;
        *reinterpret_cast<f32x4 *>(o + 4) = v1;
      } else if constexpr (INT8) {
        i8s::int8_epilogue8<EPI>(v0, v1, m, n, g.N, a.scale, g.R, tab, g.C);
      } else {
        gemm_finish8<EPI>(v0, v1, m, n, g, tab);
      }
    }
  }
}

}  // namespace gk
}  // namespace pk
