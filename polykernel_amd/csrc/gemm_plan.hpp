// gemm_plan.hpp -- tile and K-split choice of the ring kernel (gemm_ring.hpp)
// for the bf16 and the int8 GEMM.  Host only.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdint>

namespace pk {

// A tile of 32 fm x 64 wn outputs; `us` is the time of one 64-deep k-tile with
// a tile on every CU.
struct RingTile {
  int fm, wn;
  double us;
};

// Coefficients of the time model (us, bytes per us): launch and first loads,
// each round of 256 workgroups, the slowdown of k-tiles in launches of three
// rounds or more (the clock falls), the memory rate of a full grid, and the
// launch and rate of the split reduction.
struct RingModel {
  double launch, round, slow, mem, reduce, reduce_rate;
};

struct RingChoice {
  int tile = -1;  // index, or -1: the kernel does not take the shape
  int splits = 1, split_tiles = 0, units = 0;
  double us = 0;
};

// Whether the ring kernel takes the shape (16-byte aligned operands).
inline bool ring_shape_ok(int N, int K, int weight_bytes) {
  return N % (16 / weight_bytes) == 0 && K % 8 == 0 && (size_t)K * N * weight_bytes < (size_t(1) << 31) &&
         (size_t)160 * K * 2 < (size_t(1) << 31);
}

// Splits use at most `scratch` bytes of fp32 partials.
inline RingChoice ring_choose(const RingTile *tiles, int ntiles, const RingModel &c, int M, int N, int K,
                              int weight_bytes, size_t scratch) {
  RingChoice best;
  if (!ring_shape_ok(N, K, weight_bytes)) return best;
  const int ktiles = (K + 63) / 64;
  const double bytes = (double)N * K * weight_bytes + 2.0 * ((double)M * K + (double)M * N);
  for (int i = 0; i < ntiles; ++i) {
    const RingTile &v = tiles[i];
    const int64_t grid = (((int64_t)M + 32 * v.fm - 1) / (32 * v.fm)) * (((int64_t)N + 64 * v.wn - 1) / (64 * v.wn));
    for (int s : {1, 2, 3, 4, 6, 8}) {
      const int steps = (ktiles + s - 1) / s;
      if (s > 1 && steps < 4) break;
      const int splits = (ktiles + steps - 1) / steps;
      const size_t part = splits > 1 ? (size_t)splits * M * N * sizeof(float) : 0;
      const int64_t units = grid * splits;
      if (part > scratch || units > INT32_MAX / 2 || (splits > 1 && units > 1024)) break;
      const double rounds = std::ceil(units / 256.0);
      const double k_us = steps * v.us * (1.0 + c.slow * std::min(1.0, (rounds - 1) / 2));
      double us = c.launch + rounds * c.round + std::max(rounds * k_us, bytes / (c.mem * std::min(1.0, units / 256.0)));
      if (splits > 1) us += c.reduce + 2.0 * part / c.reduce_rate;
      if (best.tile < 0 || us < best.us * (1 - 1e-9)) best = RingChoice{i, splits, steps, (int)units, us};
    }
  }
  return best;
}

// A thread's last plans, by shape and scratch (a plan depends on nothing else):
// a program's layers come back to the same few shapes, and a plan costs 0.5-1.2
// us of a call whose kernels may take 5.
template <typename Plan, int SLOTS = 16>
class PlanMemo {
 public:
  template <typename F>
  const Plan &get(int M, int N, int K, size_t scratch, int kind, F &&make) {
    const uint32_t h = (uint32_t)M * 0x9E3779B1u ^ (uint32_t)N * 0x85EBCA6Bu ^ (uint32_t)K * 0xC2B2AE35u ^
                       (uint32_t)(scratch >> 8) * 0x27D4EB2Fu ^ (uint32_t)kind;
    Slot &s = slots_[(h ^ h >> 15) % SLOTS];
    if (!s.set || s.M != M || s.N != N || s.K != K || s.scratch != scratch || s.kind != kind)
      s = Slot{true, M, N, K, kind, scratch, make()};
    return s.plan;
  }

 private:
  struct Slot {
    bool set = false;
    int M, N, K, kind;
    size_t scratch;
    Plan plan;
  };
  Slot slots_[SLOTS];
};

}  // namespace pk
