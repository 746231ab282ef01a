// attention_decode.hpp -- attention of 1 to 4 queries per head over a long key
// cache, with the KV append fused (D 64 or 128).
//
// What bounds it: K and V are read once and used for at most 4 queries, so the
// time is that of streaming them from HBM.  The flash kernel's 64- or 128-query
// tile spends a whole MFMA and LDS step per key tile on one live query and
// takes one workgroup per CU (B 8, H 32, D 128, 2047 + 1 keys: 50 us for 268 MB,
// 5.4 TB/s, behind two append launches of 1.9 us).  Here a row of K or V is read
// straight into registers by D / 8 lanes (16 bytes each), 64 / (D / 8) rows per
// load instruction; each lane multiplies its 8 dims in fp32, DPP adds the
// score over the row's lanes, and every group of D / 8 lanes keeps its own
// online softmax state (raw-score max, sum, 8 dims of the output per lane), so
// the loop has no LDS access and no barrier.  U row loads of K and U of V are
// in flight per lane: the next K rows are requested as soon as the scores are
// formed, the next V rows after the products.  Scores, weights and products
// are fp32 throughout.
//
// A workgroup's 8 waves take interleaved batches of rows of one (b, h) and one
// key split; their states are merged in LDS.  Split states go to the flash
// kernel's partial layout and fa_combine_body.
#pragma once

#include "attention_kernels.hpp"

namespace pk {
namespace att {

constexpr int AD_WAVES = 8, AD_THREADS = AD_WAVES * 64, AD_U = 8, AD_MAX_Q = 4;

// Sum over the 8 or 16 lanes that share a row, in every one of them.
template <int LANES>
__device__ __forceinline__ float row_lane_sum(float v) {
  auto dpp = [](float x, auto ctrl) __attribute__((always_inline)) {
    return __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(x), decltype(ctrl)::value, 0xF, 0xF, true));
  };
  v += dpp(v, std::integral_constant<int, 0xB1>{});   // quad_perm [1,0,3,2]: lane ^ 1
  v += dpp(v, std::integral_constant<int, 0x4E>{});   // quad_perm [2,3,0,1]: lane ^ 2
  v += dpp(v, std::integral_constant<int, 0x141>{});  // row_half_mirror: the other quad of 8
  if constexpr (LANES == 16) v += dpp(v, std::integral_constant<int, 0x140>{});  // row_mirror: the other 8 of 16
  return v;
}

// The merge over a wave's groups (lanes l, l ^ LPR, l ^ 2 LPR, ... up to l ^ 32)
// by the two lane swaps and, for 8 lanes per row, a rotation by 8 in each 16.
// With shuffles (LDS permutes) of every value it was most of a short call of
// four queries: 1 head of 8 keys at D 64 8.2 us.
__device__ __forceinline__ void xor16_pair(float a, float b, float &lo, float &hi) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  lo = __uint_as_float(r[0]);
  hi = __uint_as_float(r[1]);
}
__device__ __forceinline__ float row_ror8(float v) {
  return __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0x128, 0xF, 0xF, true));
}
// f over the groups, in every lane.
template <int LPR, typename F>
__device__ __forceinline__ float group_combine(float v, F &&f) {
  static_assert(LPR == 8 || LPR == 16, "lanes per row");
  float lo, hi;
  xor32_pair(v, lo, hi);
  v = f(lo, hi);
  xor16_pair(v, v, lo, hi);
  v = f(lo, hi);
  if constexpr (LPR == 8) v = f(v, row_ror8(v));
  return v;
}
// Sums of v[0..7] over the groups: a swap of two values adds both at once, each
// in one half of the lanes, so the lanes of 16-lane row r (0-3) end up with the
// sums of v[4 (r / 2) + 2 (r % 2)] and the value after it.
template <int LPR>
__device__ __forceinline__ void group_sum8(const float (&v)[8], float &s0, float &s1) {
  float h[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[e]), __float_as_uint(v[e + 4]), false, false);
    h[e] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  float lo, hi;
  xor16_pair(h[0], h[2], lo, hi);
  s0 = lo + hi;
  xor16_pair(h[1], h[3], lo, hi);
  s1 = lo + hi;
  if constexpr (LPR == 8) {
    s0 += row_ror8(s0);
    s1 += row_ror8(s1);
  }
}

template <int D, int NQ>
__device__ __forceinline__ void att_decode_body(FaArgs g) {
  constexpr int LPR = D / 8;             // lanes per row
  constexpr int GROUPS = 64 / LPR;       // rows per load, states per wave
  constexpr int BATCH = GROUPS * AD_U;   // keys of a wave's batch
  __shared__ float so[AD_WAVES][NQ][D];
  __shared__ float sml[AD_WAVES][NQ][2];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int bh = blockIdx.x / g.splits, split = blockIdx.x % g.splits;
  const int grp = lane / LPR, d0 = 8 * (lane % LPR);
  const bool fused = g.Kn != nullptr;
  const int S_new = g.S_kv - g.S_cache;
  const uint16_t *Kp = g.K + (size_t)bh * g.kv_rows * D + d0;
  const uint16_t *Vp = g.V + (size_t)bh * g.kv_rows * D + d0;
  const uint16_t *Knp = fused ? g.Kn + (size_t)bh * S_new * D + d0 : Kp;
  const uint16_t *Vnp = fused ? g.Vn + (size_t)bh * S_new * D + d0 : Vp;

  // this head's new rows -> cache (rows nobody reads there)
  if (fused && split == 0) {
    uint16_t *kc = g.Kc + ((size_t)bh * g.kv_rows + g.S_cache) * D, *vc = g.Vc + ((size_t)bh * g.kv_rows + g.S_cache) * D;
    const uint16_t *kn = g.Kn + (size_t)bh * S_new * D, *vn = g.Vn + (size_t)bh * S_new * D;
    for (int u = tid; u < S_new * (D / 8); u += AD_THREADS) {
      *reinterpret_cast<u32x4 *>(kc + 8 * u) = *reinterpret_cast<const u32x4 *>(kn + 8 * u);
      *reinterpret_cast<u32x4 *>(vc + 8 * u) = *reinterpret_cast<const u32x4 *>(vn + 8 * u);
    }
  }

  float q[NQ][8], acc[NQ][8], m_run[NQ], l_run[NQ];
  int limit[NQ];  // last visible key
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    const int qi = min(i, g.S_q - 1);
    const u32x4 v = *reinterpret_cast<const u32x4 *>(g.Q + ((size_t)bh * g.S_q + qi) * D + d0);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      q[i][2 * e] = lo_bf(v[e]);
      q[i][2 * e + 1] = hi_bf(v[e]);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[i][e] = 0.f;
    m_run[i] = -INFINITY;
    l_run[i] = 0.f;
    limit[i] = g.causal ? g.S_kv - g.S_q + qi : g.S_kv - 1;
  }
  const float c2 = g.scale * 1.4426950408889634f;  // scale * log2(e)

  // batches of this split, interleaved over the waves
  const int batches = (g.S_kv + BATCH - 1) / BATCH;
  const int per = (batches + g.splits - 1) / g.splits;
  const int b_end = min(batches, (split + 1) * per);
  u32x4 kr[AD_U], vr[AD_U];
  // the batch's rows: all in one source, or the last rows clamped and taken
  // from the cache or the new rows (clamped rows are masked)
  auto load = [&](u32x4 (&r)[AD_U], const uint16_t *cache, const uint16_t *neu, int b) __attribute__((always_inline)) {
    const int k0 = b * BATCH + grp;
    if ((b + 1) * BATCH <= g.S_cache) {
#pragma unroll
      for (int u = 0; u < AD_U; ++u)
        r[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(cache + (size_t)(k0 + GROUPS * u) * D));
    } else {
#pragma unroll
      for (int u = 0; u < AD_U; ++u) {
        const int k = min(k0 + GROUPS * u, g.S_kv - 1);
        const uint16_t *p = k < g.S_cache ? cache + (size_t)k * D : neu + (size_t)(k - g.S_cache) * D;
        r[u] = *reinterpret_cast<const u32x4 *>(p);
      }
    }
  };
  int b = split * per + wid;
  if (b < b_end) {
    load(kr, Kp, Knp, b);
    load(vr, Vp, Vnp, b);
  }
  for (; b < b_end; b += AD_WAVES) {
    float s[NQ][AD_U];
#pragma unroll
    for (int u = 0; u < AD_U; ++u) {
      float k[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        k[2 * e] = lo_bf(kr[u][e]);
        k[2 * e + 1] = hi_bf(kr[u][e]);
      }
#pragma unroll
      for (int i = 0; i < NQ; ++i) {
        float t = q[i][0] * k[0];
#pragma unroll
        for (int e = 1; e < 8; ++e) t = fmaf(q[i][e], k[e], t);
        s[i][u] = row_lane_sum<LPR>(t);
      }
    }
    const int nb = b + AD_WAVES;
    if (nb < b_end) load(kr, Kp, Knp, nb);
    // mask only in batches that reach past a query's last visible key
    if ((b + 1) * BATCH - 1 > limit[0]) {
#pragma unroll
      for (int i = 0; i < NQ; ++i)
#pragma unroll
        for (int u = 0; u < AD_U; ++u)
          if (b * BATCH + grp + GROUPS * u > limit[i]) s[i][u] = -INFINITY;
    }
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      float m = s[i][0];
#pragma unroll
      for (int u = 1; u < AD_U; ++u) m = fmaxf(m, s[i][u]);
      const float m_new = fmaxf(m_run[i], m);
      const float mc = m_new == -INFINITY ? 0.f : m_new * c2;
      const float alpha = __builtin_amdgcn_exp2f(fmaf(m_run[i], c2, -mc));  // 0 for m_run = -inf
      m_run[i] = m_new;
      float sum = 0.f;
#pragma unroll
      for (int u = 0; u < AD_U; ++u) {
        s[i][u] = __builtin_amdgcn_exp2f(fmaf(s[i][u], c2, -mc));
        sum += s[i][u];
      }
      l_run[i] = fmaf(l_run[i], alpha, sum);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[i][e] *= alpha;
    }
#pragma unroll
    for (int u = 0; u < AD_U; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float v0 = lo_bf(vr[u][e]), v1 = hi_bf(vr[u][e]);
#pragma unroll
        for (int i = 0; i < NQ; ++i) {
          acc[i][2 * e] = fmaf(s[i][u], v0, acc[i][2 * e]);
          acc[i][2 * e + 1] = fmaf(s[i][u], v1, acc[i][2 * e + 1]);
        }
      }
    if (nb < b_end) load(vr, Vp, Vnp, nb);
  }

  // ---- merge the states of the wave's groups, then of the waves in LDS, in wave
  // order; a wave without a batch has nothing to merge
  auto weight = [&](float m, float M) __attribute__((always_inline)) {
    return m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m - M) * c2);
  };
  const bool any = split * per + wid < b_end;
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    float M = -INFINITY, l = 0.f, s0 = 0.f, s1 = 0.f;
    if (any) {
      M = group_combine<LPR>(m_run[i], [](float a, float b) __attribute__((always_inline)) { return fmaxf(a, b); });
      const float w = weight(m_run[i], M);
      l = group_combine<LPR>(l_run[i] * w, [](float a, float b) __attribute__((always_inline)) { return a + b; });
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = acc[i][e] * w;
      group_sum8<LPR>(v, s0, s1);
    }
    const int r = lane >> 4;
    if (LPR == 16 || !(lane & 8)) {
      float *o = &so[wid][i][d0 + 4 * (r >> 1) + 2 * (r & 1)];
      o[0] = s0;
      o[1] = s1;
    }
    if (lane == 0) {
      sml[wid][i][0] = M;
      sml[wid][i][1] = l;
    }
  }
  __syncthreads();
  // two neighbouring dims of a query per thread
  for (int t = tid; t < NQ * (D / 2); t += AD_THREADS) {
    const int i = t / (D / 2), d = 2 * (t % (D / 2));
    if (i >= g.S_q) break;
    float M = -INFINITY, L = 0.f, v0 = 0.f, v1 = 0.f;
#pragma unroll
    for (int w = 0; w < AD_WAVES; ++w) M = fmaxf(M, sml[w][i][0]);
#pragma unroll
    for (int w = 0; w < AD_WAVES; ++w) {
      const float f = weight(sml[w][i][0], M);
      L += sml[w][i][1] * f;
      v0 += so[w][i][d] * f;
      v1 += so[w][i][d + 1] * f;
    }
    const size_t row = (size_t)bh * g.S_q + i;
    if (g.splits == 1) {
      const float inv = 1.0f / L;
      *reinterpret_cast<uint32_t *>(g.O + row * D + d) = pack_bf(v0 * inv, v1 * inv);
    } else {
      const size_t prow = (size_t)split * g.BH * g.S_q + row;
      g.part_o[prow * D + d] = v0;
      g.part_o[prow * D + d + 1] = v1;
      if (d == 0) {
        g.part_ml[prow * 2] = M;
        g.part_ml[prow * 2 + 1] = L;
      }
    }
  }
}

}  // namespace att
}  // namespace pk
