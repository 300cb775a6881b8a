// Wave tree: an implicit 64-ary tree over the leaves in Morton order, for
// traversals that run one wave per query.
//
// Group g of level 0 is the leaves [64 g, 64 g + 64), group g of level l the
// groups [64 g, 64 g + 64) of level l - 1; three levels (262 144 leaves per
// top group).  A wave tests the 64 children of a group at once, one per lane,
// and a ballot is the list of children to visit, so a traversal needs no
// stack, and a group of leaves is read with coalesced loads.  What this
// replaces is one thread per query on the binary tree: a chain of dependent
// node loads as long as the traversal, with 1/64 of a small launch's lanes
// busy.
//
// Boxes are exact FP64 and distances to them FP64, so the pruning is as fine as
// the points lie, wherever and however unevenly that is.  In FP32 relative to
// the cloud's centre a single far outlier left no bit of the others' places:
// 200 000 points with one at 10^6 times their extent, 8 neighbours each,
// 35 ms, now 2.7 ms (EMST 129 and 4.2 ms); 50 000 lattice points, 32
// neighbours, 1.27 and 1.25 ms.
#pragma once

#include "common.hpp"
#include "traverse.hpp"

namespace mhgp {

// Bound for boxes that a ball of squared radius r2 can meet.
__device__ inline double wave_bound(double r2) { return r2 * (1.0 + kSlack) + kSlackAbs; }

// A point as the centre of a traversal.
struct WaveQuery {
  double q[3];
  __device__ WaveQuery(double x, double y, double z) : q{x, y, z} {}
  __device__ double d2(const GroupBox &b) const { return box_d2(q, b.lo, b.hi); }
};

// A point of the cloud and an offset, whose sum would round away far from the
// origin.
struct WaveOffsetQuery {
  double q[3], off[3];
  __device__ WaveOffsetQuery(double x, double y, double z, double dx, double dy, double dz)
      : q{x, y, z}, off{dx, dy, dz} {}
  __device__ double d2(const GroupBox &b) const {
    double s = 0.0;
    for (int a = 0; a < 3; ++a) {
      const double d = fmax(fmax((b.lo[a] - q[a]) - off[a], off[a] - (b.hi[a] - q[a])), 0.0);
      s += d * d;
    }
    return s;
  }
};

// Calls leaf(g) for every level-0 group whose box lies within the squared
// bound `most`, which leaf may shrink as it goes (pending groups are tested
// against it again), and whose ancestors and itself pass keep(level, group).
// Uniform over the wave: every lane makes the call with the same query and
// bound, and leaf(g) runs with all lanes active.
template <class Q_, class K, class F>
__device__ inline void wave_tree_visit(const WaveTree &T, const Q_ &Q, double &most, K &&keep, F &&leaf) {
  const uint32_t lane = threadIdx.x & 63u;
  for (uint32_t b2 = 0; b2 < T.c2; b2 += 64) {
    const uint32_t i2 = b2 + lane;
    // a single top group holds every leaf: nothing to test
    uint64_t m2 = T.c2 == 1 ? 1ull : __ballot(i2 < T.c2 && keep(2, min(i2, T.c2 - 1)) && !(Q.d2(T.l2[min(i2, T.c2 - 1)]) > most));
    while (m2) {
      const uint32_t g2 = b2 + (uint32_t)(__ffsll((long long)m2) - 1);
      m2 &= m2 - 1;
      const uint32_t i1 = g2 * 64 + lane;
      const double d1 = Q.d2(T.l1[min(i1, T.c1 - 1)]);
      uint64_t rem1 = __ballot(i1 < T.c1 && keep(1, min(i1, T.c1 - 1)));
      for (uint64_t m1 = __ballot(!(d1 > most)) & rem1; m1; m1 = __ballot(!(d1 > most)) & rem1) {
        const int k1 = __ffsll((long long)m1) - 1;
        rem1 &= ~((2ull << k1) - 1ull);  // this one is taken; the ones before it lie outside the bound
        const uint32_t g1 = g2 * 64 + (uint32_t)k1, i0 = g1 * 64 + lane;
        const double d0 = Q.d2(T.l0[min(i0, T.c0 - 1)]);
        uint64_t rem0 = __ballot(i0 < T.c0 && keep(0, min(i0, T.c0 - 1)));
        for (uint64_t m0 = __ballot(!(d0 > most)) & rem0; m0; m0 = __ballot(!(d0 > most)) & rem0) {
          const int k0 = __ffsll((long long)m0) - 1;
          rem0 &= ~((2ull << k0) - 1ull);
          leaf(g1 * 64 + (uint32_t)k0);
        }
      }
    }
  }
}

template <class Q_, class F>
__device__ inline void wave_tree_visit(const WaveTree &T, const Q_ &Q, double &most, F &&leaf) {
  wave_tree_visit(T, Q, most, [](int, uint32_t) { return true; }, leaf);
}

// A level-0 group near the query (the nearest box under the nearest level-1
// box), where a search bound starts out tight.  Uniform over the wave.
__device__ inline uint32_t wave_near_group(const WaveTree &T, const WaveQuery &Q) {
  const uint32_t lane = threadIdx.x & 63u;
  double d = INFINITY;
  uint32_t g = 0;
  for (uint32_t i = lane; i < T.c1; i += 64) {
    const double e = Q.d2(T.l1[i]);
    if (e < d) {
      d = e;
      g = i;
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const double e = __shfl_xor(d, o);
    const uint32_t h = __shfl_xor(g, o);
    if (e < d || (e == d && h < g)) {
      d = e;
      g = h;
    }
  }
  uint32_t i = min(g * 64 + lane, T.c0 - 1);
  d = Q.d2(T.l0[i]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const double e = __shfl_xor(d, o);
    const uint32_t h = __shfl_xor(i, o);
    if (e < d || (e == d && h < i)) {
      d = e;
      i = h;
    }
  }
  return __builtin_amdgcn_readfirstlane(i);
}

// Value of lane `src` (uniform) in every lane.
__device__ inline uint32_t lane_u32(uint32_t v, int src) { return __builtin_amdgcn_readlane(v, src); }
__device__ inline double lane_f64(double v, int src) {
  const uint64_t b = (uint64_t)__double_as_longlong(v);
  const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)b, src), hi = __builtin_amdgcn_readlane((uint32_t)(b >> 32), src);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

}  // namespace mhgp
