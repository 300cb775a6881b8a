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
// Boxes are FP32, relative to a centre of the cloud and rounded outward, so
// the precision of the pruning does not depend on where the cloud lies.
#pragma once

#include "common.hpp"

namespace mhgp {

// Query point in the boxes' frame, with the largest magnitude of its FP32
// coordinates (their rounding stays below 1e-7 of it).
struct WaveQuery {
  float q[3], qmax;
  // (x, y, z) + (dx, dy, dz): a point near a cloud far from the origin is given
  // by one of the cloud's own and an offset, whose sum would round away
  __device__ WaveQuery(const WaveTree &T, double x, double y, double z, double dx = 0.0, double dy = 0.0,
                       double dz = 0.0) {
    q[0] = (float)((x - T.centre[0]) + dx);
    q[1] = (float)((y - T.centre[1]) + dy);
    q[2] = (float)((z - T.centre[2]) + dz);
    qmax = fmaxf(fmaxf(fabsf(q[0]), fabsf(q[1])), fabsf(q[2]));
  }
  // Squared FP32 bound for boxes that a ball of squared radius r2 can meet:
  // inflated past the rounding of the query, of the box distance and of this
  // arithmetic; the absolute term keeps the squares of tiny radii in the
  // normal range, and a bound beyond FP32 prunes nothing.
  __device__ float bound(double r2) const {
    const float r = __builtin_amdgcn_sqrtf((float)r2) * (1.0f + 2e-6f) + qmax * 1e-6f + 1e-18f;
    const float b = r * r * (1.0f + 1e-5f);
    return b < 3.0e38f ? b : INFINITY;
  }
  __device__ float d2(const GroupBox &b) const {
    const float4 *v = reinterpret_cast<const float4 *>(&b);
    const float4 lo = v[0], hi = v[1];
    const float dx = fmaxf(fmaxf(lo.x - q[0], q[0] - hi.x), 0.f);
    const float dy = fmaxf(fmaxf(lo.y - q[1], q[1] - hi.y), 0.f);
    const float dz = fmaxf(fmaxf(lo.z - q[2], q[2] - hi.z), 0.f);
    return dx * dx + dy * dy + dz * dz;
  }
};

// Calls leaf(g) for every level-0 group whose box lies within the squared
// bound Tf, which leaf may shrink as it goes (pending groups are tested
// against it again), and whose ancestors and itself pass keep(level, group).
// Uniform over the wave: every lane makes the call with the same query and
// bound, and leaf(g) runs with all lanes active.
template <class K, class F>
__device__ inline void wave_tree_visit(const WaveTree &T, const WaveQuery &Q, float &Tf, K &&keep, F &&leaf) {
  const uint32_t lane = threadIdx.x & 63u;
  for (uint32_t b2 = 0; b2 < T.c2; b2 += 64) {
    const uint32_t i2 = b2 + lane;
    // a single top group holds every leaf: nothing to test
    uint64_t m2 = T.c2 == 1 ? 1ull : __ballot(i2 < T.c2 && keep(2, min(i2, T.c2 - 1)) && !(Q.d2(T.l2[min(i2, T.c2 - 1)]) > Tf));
    while (m2) {
      const uint32_t g2 = b2 + (uint32_t)(__ffsll((long long)m2) - 1);
      m2 &= m2 - 1;
      const uint32_t i1 = g2 * 64 + lane;
      const float d1 = Q.d2(T.l1[min(i1, T.c1 - 1)]);
      uint64_t rem1 = __ballot(i1 < T.c1 && keep(1, min(i1, T.c1 - 1)));
      for (uint64_t m1 = __ballot(!(d1 > Tf)) & rem1; m1; m1 = __ballot(!(d1 > Tf)) & rem1) {
        const int k1 = __ffsll((long long)m1) - 1;
        rem1 &= ~((2ull << k1) - 1ull);  // this one is taken; the ones before it lie outside the bound
        const uint32_t g1 = g2 * 64 + (uint32_t)k1, i0 = g1 * 64 + lane;
        const float d0 = Q.d2(T.l0[min(i0, T.c0 - 1)]);
        uint64_t rem0 = __ballot(i0 < T.c0 && keep(0, min(i0, T.c0 - 1)));
        for (uint64_t m0 = __ballot(!(d0 > Tf)) & rem0; m0; m0 = __ballot(!(d0 > Tf)) & rem0) {
          const int k0 = __ffsll((long long)m0) - 1;
          rem0 &= ~((2ull << k0) - 1ull);
          leaf(g1 * 64 + (uint32_t)k0);
        }
      }
    }
  }
}

template <class F>
__device__ inline void wave_tree_visit(const WaveTree &T, const WaveQuery &Q, float &Tf, F &&leaf) {
  wave_tree_visit(T, Q, Tf, [](int, uint32_t) { return true; }, leaf);
}

// A level-0 group near the query (the nearest box under the nearest level-1
// box), where a search bound starts out tight.  Uniform over the wave.
__device__ inline uint32_t wave_near_group(const WaveTree &T, const WaveQuery &Q) {
  const uint32_t lane = threadIdx.x & 63u;
  float d = INFINITY;
  uint32_t g = 0;
  for (uint32_t i = lane; i < T.c1; i += 64) {
    const float e = Q.d2(T.l1[i]);
    if (e < d) {
      d = e;
      g = i;
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float e = __shfl_xor(d, o);
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
    const float e = __shfl_xor(d, o);
    const uint32_t h = __shfl_xor(i, o);
    if (e < d || (e == d && h < i)) {
      d = e;
      i = h;
    }
  }
  return __builtin_amdgcn_readfirstlane(i);
}

// Value of lane `src` (uniform) in every lane, and the value of the lane
// below (lane 0 keeps its own).
__device__ inline uint32_t lane_u32(uint32_t v, int src) { return __builtin_amdgcn_readlane(v, src); }
__device__ inline double lane_f64(double v, int src) {
  const uint64_t b = (uint64_t)__double_as_longlong(v);
  const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)b, src), hi = __builtin_amdgcn_readlane((uint32_t)(b >> 32), src);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

}  // namespace mhgp
