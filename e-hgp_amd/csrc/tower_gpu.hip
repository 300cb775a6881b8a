// Device arm resolution for the hgp_reduced tower.
//
// For order k the minima are the catalogue records of closed rank k and the
// saddles those of closed rank k+1.  Every strict arm (closed label minus one
// shell point) is resolved to the minimum of its component:
//  * the labels of the minima live in an open-addressing hash table;
//  * an arm that is not a minimum descends: the FP64 miniball of the facet has
//    its support and containment certified with the predicates of
//    predicates.hpp, the points of the closed ball come from a
//    neighbour list or an LBVH ball query, and the facet trades its least
//    support point for the least point strictly inside (the miniball strictly
//    shrinks);
//  * anything the certified filters cannot decide is flagged for the host's
//    exact descent.
#include <chrono>
#include <cstdio>
#include <cstdlib>

#include "pipeline.hpp"
#include "predicates.hpp"
#include "scan.hpp"
#include "supports.hpp"
#include "traverse.hpp"
#include "tower_gpu.hpp"
#include "tower_state.hpp"
#include "wave.hpp"

namespace mhgp {

namespace {

constexpr int kMaxLabel = 11;

// Hash of a facet: the sum of its points' mixes, so that the hash of a
// saddle's label minus one point is a subtraction.  The low word picks the
// slot, the high word (made odd) is the tag stored beside the value.
__device__ inline uint64_t point_mix(uint32_t id) {
  uint32_t a = id * 0x9e3779b1u, b = (id ^ 0x5bd1e995u) * 0x85ebca77u;
  a ^= a >> 15;
  b ^= b >> 13;
  a *= 0x2c1b3c6du;
  b *= 0xc2b2ae3du;
  return ((uint64_t)(b ^ (b >> 16)) << 32) | (a ^ (a >> 13));
}
__device__ inline uint64_t hash_slot(uint64_t h, uint64_t mask) { return (h ^ (h >> 19)) & mask & 0xffffffffull; }
__device__ inline unsigned long long hash_tag(uint64_t h) { return (unsigned long long)((h >> 32) | 1ull) << 32; }

__device__ inline int rank_of(const EventRec &e) { return (e.meta >> 8) & 0xff; }

// Sorted closed label (L points) of a record: the interior is sorted and
// padded with kInvalid, each support point is bubbled in (static indices, the
// label stays in registers).  members: bit q set when label[q] is a support
// point; support ids ascend, so arm j drops the j-th of them.
template <int L>
__device__ inline void sorted_label(const EventRec &e, uint32_t (&a)[L], uint32_t &members) {
#pragma unroll
  for (int q = 0; q < L; ++q) a[q] = q < kMaxInterior ? e.interior[q] : kInvalid;
  uint32_t sup[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    sup[i] = e.ids[i];
    uint32_t x = sup[i];
#pragma unroll
    for (int q = 0; q < L; ++q) {
      const uint32_t lo = min(a[q], x);
      x = max(a[q], x);
      a[q] = lo;
    }
  }
  members = 0;
#pragma unroll
  for (int q = 0; q < L; ++q) {
    bool in = false;
#pragma unroll
    for (int i = 0; i < 4; ++i) in |= a[q] == sup[i];
    members |= (uint32_t)(in && a[q] != kInvalid) << q;
  }
}

// Position of the j-th set bit.
__device__ inline int nth_bit(uint32_t m, int j) {
  for (int i = 0; i < j; ++i) m &= m - 1;
  return __ffs(m) - 1;
}

// Slots of this thread in a global append list, count of them per thread:
// one atomic per workgroup (a single counter takes about 10 ns per atomic, so
// one per wave bound the kernels below).  Every thread of the workgroup calls.
template <int WAVES>
__device__ inline unsigned long long block_append(uint32_t count, unsigned long long *counter) {
  __shared__ uint32_t tot[WAVES];
  __shared__ unsigned long long base;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t x = count;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t y = __shfl_up(x, (unsigned)d);
    if (lane >= d) x += y;
  }
  if (lane == 63) tot[wave] = x;
  __syncthreads();
  uint32_t before = 0, all = 0;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) {
    before += w < wave ? tot[w] : 0u;
    all += tot[w];
  }
  if (threadIdx.x == 0 && all) base = atomicAdd(counter, (unsigned long long)all);
  __syncthreads();
  const unsigned long long at = all ? base + before + x - count : 0ull;
  __syncthreads();  // the shared words serve the next call
  return at;
}

// Records grouped by closed rank, canonical order kept inside each rank:
// key = rank (0xff for a degenerate record), value = sorted position.
__global__ void k_rank_keys(const EventRec *__restrict__ ev, const uint32_t *__restrict__ order, int64_t n,
                            uint64_t *keys, uint32_t *vals) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const EventRec &e = ev[order[i]];
  keys[i] = ((e.meta >> 24) & 1) ? 0xffull : (uint64_t)rank_of(e);
  vals[i] = (uint32_t)i;
}

__global__ void k_rank_bounds(const uint64_t *__restrict__ keys, int64_t n, uint32_t *lo, uint32_t *hi) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint64_t key = keys[i];
  if (i == 0 || keys[i - 1] != key) lo[key] = (uint32_t)i;
  if (i == n - 1 || keys[i + 1] != key) hi[key] = (uint32_t)(i + 1);
}

// Minima of an order: labels (K ids each) and the hash table, whose slots
// hold tag << 32 | minimum (0: empty).
struct MinimaTable {
  unsigned long long *slots;
  uint64_t mask;
  uint32_t *labels;
};

template <int K>
__global__ void k_insert_minima(const EventRec *__restrict__ ev, const uint32_t *__restrict__ order,
                                const uint32_t *__restrict__ pos, int64_t count, MinimaTable T) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  uint32_t lab[K], members;
  sorted_label<K>(ev[order[pos[i]]], lab, members);
  uint64_t h = 0;
#pragma unroll
  for (int q = 0; q < K; ++q) {
    T.labels[(size_t)i * K + q] = lab[q];
    h += point_mix(lab[q]);
  }
  uint64_t slot = hash_slot(h, T.mask);
  const unsigned long long mine = hash_tag(h) | (unsigned long long)(uint32_t)i;
  while (atomicCAS(&T.slots[slot], 0ull, mine) != 0ull) slot = (slot + 1) & T.mask;
}

// The minimum with facet F (sorted, hash h), or -1.
template <int K>
__device__ inline int64_t lookup(const MinimaTable &T, const uint32_t (&F)[K], uint64_t h) {
  uint64_t slot = hash_slot(h, T.mask);
  const unsigned long long tag = hash_tag(h);
  while (true) {
    const unsigned long long s = T.slots[slot];
    if (s == 0ull) return -1;
    if ((s & 0xffffffff00000000ull) == tag) {
      const uint32_t v = (uint32_t)s;
      bool same = true;
#pragma unroll
      for (int q = 0; q < K; ++q) same &= T.labels[(size_t)v * K + q] == F[q];
      if (same) return v;
    }
    slot = (slot + 1) & T.mask;
  }
}

// Saddles of an order, read once from their records: sorted labels (K + 1
// ids), support members, arm counts, exact class and level.
struct Saddles {
  uint32_t *label;      // K + 1 per saddle
  uint16_t *members;
  uint32_t *base;       // first arm (after the scan of the arm counts)
};

template <int K>
__global__ void k_saddles(const EventRec *__restrict__ ev, const uint32_t *__restrict__ order,
                          const uint32_t *__restrict__ cls, const uint32_t *__restrict__ pos, int64_t count, Saddles D,
                          uint32_t *sizes, uint32_t *out_cls, double *out_level) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  const EventRec &e = ev[order[pos[i]]];
  uint32_t lab[K + 1], members;
  sorted_label<K + 1>(e, lab, members);
#pragma unroll
  for (int q = 0; q <= K; ++q) D.label[(size_t)i * (K + 1) + q] = lab[q];
  D.members[i] = (uint16_t)members;
  sizes[i] = e.meta & 0xff;
  out_cls[i] = cls[pos[i]];
  out_level[i] = e.level;
}

// Facet of an arm: the saddle's label without position `at`.
template <int K>
__device__ inline void drop_point(const uint32_t (&L)[K + 1], int at, uint32_t (&F)[K]) {
#pragma unroll
  for (int q = 0; q < K; ++q) F[q] = q < at ? L[q] : L[q + 1];
}

template <int K>
__device__ inline void load_label(const Saddles &D, uint32_t s, uint32_t (&L)[K + 1]) {
#pragma unroll
  for (int q = 0; q <= K; ++q) L[q] = D.label[(size_t)s * (K + 1) + q];
}

struct ArmParams {
  Saddles sad;
  int64_t saddles;
  MinimaTable table;
  const double *X, *Y, *Z;
  const WideNode *wide;
  const double *LX, *LY, *LZ;
  const uint32_t *leaf_id;
  const uint32_t *leaf_pos;
  uint32_t *carrier;  // per arm: minimum index, or kInvalid (host)
  // nearest neighbours of every PointId (a row of kNearRow ids, nearest first,
  // kInvalid past the list) and the FP64 squared distance to the last of them
  // (infinite when the list holds every other point); nn == nullptr: none
  const uint32_t *nn;
  const double *nn_d2;
};

constexpr int kNearK = 63;    // a wave's neighbour list without its tie probe
constexpr int kNearRow = 64;

// Facets to descend, deduplicated: a slot holds tag << 32 | saddle << 2 | arm
// of the saddle; an arm whose facet equals a stored one takes that arm's
// carrier after the descents.  The probe length is bounded; an arm that finds
// no slot simply descends itself.
struct FacetSet {
  unsigned long long *slots;
  uint64_t mask;
  uint32_t *alias_arm, *alias_rep;
  unsigned long long *alias_count;
};

// One thread per saddle: each arm's facet is a minimum (hash hit), equals a
// facet already claimed, or is queued for the descents (saddle << 2 | arm, with
// the Morton position of its least point, so that the descents run in spatial
// order).  Bound by the random reads of the tables; a thread per arm built
// every label up to four times and its two appends per wave serialised on
// their counters (order 10 of the
// 50 000-point tower, 20.6 M arms: 6.9 ms, 2.1 here).
constexpr int kArmBlock = 256;
template <int K>
__global__ void __launch_bounds__(kArmBlock) k_arm_lookup(ArmParams A, FacetSet D, uint32_t *queue, uint64_t *qkey,
                                                          unsigned long long *qcount) {
  const int64_t s = (int64_t)blockIdx.x * kArmBlock + threadIdx.x;
  uint32_t ndesc = 0, nalias = 0, desc = 0, rep[4] = {}, key[4] = {}, base = 0;
  uint32_t alias = 0;
  if (s < A.saddles) {
    base = A.sad.base[s];
    uint32_t L[K + 1];
    load_label<K>(A.sad, (uint32_t)s, L);
    const uint32_t members = A.sad.members[s];
    uint64_t whole = 0;
#pragma unroll
    for (int q = 0; q <= K; ++q) whole += point_mix(L[q]);
    uint32_t left = members;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (!left) continue;
      const int at = __ffs(left) - 1;
      left &= left - 1;
      uint32_t F[K];
      drop_point<K>(L, at, F);
      if (K == 1) {  // order one: the arm is a point, its own minimum
        A.carrier[base + j] = F[0];
        continue;
      }
      uint32_t gone = L[0];
#pragma unroll
      for (int q = 1; q <= K; ++q) gone = q == at ? L[q] : gone;
      const uint64_t h = whole - point_mix(gone);
      const int64_t hit = lookup<K>(A.table, F, h);
      A.carrier[base + j] = hit >= 0 ? (uint32_t)hit : kInvalid;
      if (hit >= 0) continue;
      // claim the facet
      const unsigned long long tag = hash_tag(h), mine = tag | (unsigned long long)((uint32_t)s << 2 | (uint32_t)j);
      uint64_t slot = hash_slot(h, D.mask);
      bool same = false;
      uint32_t other = 0;
      for (int probe = 0; probe < 64; ++probe) {
        const unsigned long long cur = atomicCAS(&D.slots[slot], 0ull, mine);
        if (cur == 0ull) break;
        if ((cur & 0xffffffff00000000ull) == tag) {
          other = (uint32_t)cur;
          uint32_t M[K + 1], G[K];
          load_label<K>(A.sad, other >> 2, M);
          drop_point<K>(M, nth_bit(A.sad.members[other >> 2], (int)(other & 3u)), G);
          same = true;
#pragma unroll
          for (int q = 0; q < K; ++q) same &= G[q] == F[q];
          if (same) break;
        }
        slot = (slot + 1) & D.mask;
      }
      if (same) {
        alias |= 1u << j;
        rep[j] = A.sad.base[other >> 2] + (other & 3u);
        nalias++;
      } else {
        desc |= 1u << j;
        key[j] = A.leaf_pos[F[0]];
        ndesc++;
      }
    }
  }
  if (K == 1) return;
  unsigned long long ai = block_append<kArmBlock / 64>(nalias, D.alias_count);
  unsigned long long di = block_append<kArmBlock / 64>(ndesc, qcount);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if ((alias >> j) & 1u) {
      D.alias_arm[ai] = base + j;
      D.alias_rep[ai] = rep[j];
      ai++;
    }
    if ((desc >> j) & 1u) {
      queue[di] = (uint32_t)s << 2 | (uint32_t)j;
      qkey[di] = key[j];
      di++;
    }
  }
}

__global__ void k_alias_carriers(const uint32_t *__restrict__ alias_arm, const uint32_t *__restrict__ alias_rep,
                                 uint64_t count, uint32_t *carrier) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < count) carrier[alias_arm[i]] = carrier[alias_rep[i]];
}

__device__ inline V3 P3(const double *X, const double *Y, const double *Z, uint32_t id) { return {X[id], Y[id], Z[id]}; }

// Sphere of a miniball support (2..4 points) in one form for every size: the
// scaled power a p.p - p.b of a point relative to the first support point, with
// its magnitude bound (predicates.hpp), and the centre.
struct SupSphere {
  double a, aA;
  V3 b, bA;
  V3 off;  // centre relative to the first support point
  // certified well-centred support of m points (relative to the first)
  __device__ bool init(int m, const V3 &p1, const V3 &p2, const V3 &p3) {
    if (m == 2) {
      a = aA = 1.0;
      b = p1;
      bA = vabs(p1);
      if (!(dot(p1, p1) > 0)) return false;
    } else if (m == 3) {
      TriSphere t;
      if (t.init(p1, p2) <= 0) return false;
      a = t.D;
      aA = t.DA;
      b = t.g;
      bA = t.gA;
    } else if (m == 4) {
      TetSphere t;
      if (t.init(p1, p2, p3) <= 0) return false;
      a = t.V;
      aA = t.VA;
      b = t.N;
      bA = t.NA;
    } else {
      return false;
    }
    const double h = 0.5 / a;
    off = {b.x * h, b.y * h, b.z * h};
    return true;
  }
  // certified position of a point relative to the first support point
  __device__ int side(const V3 &p) const {
    const double pp = dot(p, p);
    const int s = cert_sign(a * pp - dot(p, b), aA * pp + dot(vabs(p), bA));
    return a > 0 ? s : -s;
  }
};

// 1 / x: the hardware's estimate, in FP64 (about 24 bits of it) with one Newton
// step.
__device__ inline float reciprocal(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ inline double reciprocal(double x) {
  const double r = __builtin_amdgcn_rcp(x);
  return __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
}
__device__ inline float at_least_0(float x) { return fmaxf(x, 0.0f); }
__device__ inline double at_least_0(double x) { return fmax(x, 0.0); }

// Support of the smallest ball holding K points, by walking a centre: T are
// points on the ball's boundary; the centre moves towards its projection onto
// their affine hull (the ball shrinks) until another point is met, which joins
// T, or the projection is reached; there the point of T with the most negative
// barycentric coordinate leaves, and without one the ball is the smallest.
// (K. Fischer, B. Gaertner, M. Kutz, Fast Smallest-Enclosing-Ball Computation in
// High Dimensions, ESA 2003.)  Every lane does the same work per move, unlike
// Welzl's nested restarts.  The result is a proposal, certified by the caller.
// T: float first, whose supports of nearly cospherical facets fail the
// certificate (a 1 000-point lattice displaced by 1e-7 of its spacing: 4 645 of
// 25 496 steps); those walk again in double.  In double at once k_descend takes
// 225 instead of 168 VGPRs at order 10 and 1.3 times as long.
// Returns the size of the support (positions in at[]), 0 when the walk does not
// settle.
template <int K, class T>
__device__ inline int walk_miniball(const T (&x)[K], const T (&y)[K], const T (&z)[K], int (&at)[4]) {
  T cx = 0, cy = 0, cz = 0;
#pragma unroll
  for (int i = 0; i < K; ++i) {
    cx += x[i];
    cy += y[i];
    cz += z[i];
  }
  cx *= (T)(1.0 / K);
  cy *= (T)(1.0 / K);
  cz *= (T)(1.0 / K);
  T far = -1;
  T tx[4] = {}, ty[4] = {}, tz[4] = {};
#pragma unroll
  for (int i = 0; i < K; ++i) {
    const T dx = x[i] - cx, dy = y[i] - cy, dz = z[i] - cz, d = dx * dx + dy * dy + dz * dz;
    const bool take = d > far;
    far = take ? d : far;
    at[0] = take ? i : at[0];
    tx[0] = take ? x[i] : tx[0];
    ty[0] = take ? y[i] : ty[0];
    tz[0] = take ? z[i] : tz[0];
  }
  int m = 1;
  uint32_t in = 1u << at[0];
#pragma unroll 1
  for (int it = 0; it < 24; ++it) {
    const T wx = cx - tx[0], wy = cy - ty[0], wz = cz - tz[0];
    T la = 0, lb = 0, lc = 0;
    const T ux = tx[1] - tx[0], uy = ty[1] - ty[0], uz = tz[1] - tz[0];
    const T vx = tx[2] - tx[0], vy = ty[2] - ty[0], vz = tz[2] - tz[0];
    T qx = tx[0], qy = ty[0], qz = tz[0];
    if (m == 2) {
      la = (wx * ux + wy * uy + wz * uz) * reciprocal(ux * ux + uy * uy + uz * uz);
    } else if (m >= 3) {
      // solved with the normal of the first three points
      const T nx = uy * vz - uz * vy, ny = uz * vx - ux * vz, nz = ux * vy - uy * vx;
      if (m == 3) {
        const T in2 = reciprocal(nx * nx + ny * ny + nz * nz);
        // w x v . n and u x w . n
        la = ((wy * vz - wz * vy) * nx + (wz * vx - wx * vz) * ny + (wx * vy - wy * vx) * nz) * in2;
        lb = ((uy * wz - uz * wy) * nx + (uz * wx - ux * wz) * ny + (ux * wy - uy * wx) * nz) * in2;
      } else {
        const T ex = tx[3] - tx[0], ey = ty[3] - ty[0], ez = tz[3] - tz[0];
        const T id = reciprocal(ex * nx + ey * ny + ez * nz);
        lc = (wx * nx + wy * ny + wz * nz) * id;
        const T rx = wx - lc * ex, ry = wy - lc * ey, rz = wz - lc * ez;
        const T in2 = reciprocal(nx * nx + ny * ny + nz * nz);
        la = ((ry * vz - rz * vy) * nx + (rz * vx - rx * vz) * ny + (rx * vy - ry * vx) * nz) * in2;
        lb = ((uy * rz - uz * ry) * nx + (uz * rx - ux * rz) * ny + (ux * ry - uy * rx) * nz) * in2;
      }
    }
    T step = 1;
    int hit = -1;
    T hx = 0, hy = 0, hz = 0;
    if (m < 4) {
      qx += la * ux + lb * vx;
      qy += la * uy + lb * vy;
      qz += la * uz + lb * vz;
      const T dx = qx - cx, dy = qy - cy, dz = qz - cz;
      const T ww = wx * wx + wy * wy + wz * wz;
#pragma unroll
      for (int i = 0; i < K; ++i) {
        const T px = cx - x[i], py = cy - y[i], pz = cz - z[i];
        // 2 d . (t0 - p), the rate at which p nears the boundary
        const T rate = 2 * (dx * (px - wx) + dy * (py - wy) + dz * (pz - wz));
        const T gap = ww - (px * px + py * py + pz * pz);
        const T t = at_least_0(gap) * reciprocal(rate);
        const bool take = rate > 0 && t < step && !((in >> i) & 1u);
        step = take ? t : step;
        hit = take ? i : hit;
        hx = take ? x[i] : hx;
        hy = take ? y[i] : hy;
        hz = take ? z[i] : hz;
      }
      cx += step * dx;
      cy += step * dy;
      cz += step * dz;
    }
    if (hit >= 0) {
#pragma unroll
      for (int q = 1; q < 4; ++q) {
        const bool here = q == m;
        tx[q] = here ? hx : tx[q];
        ty[q] = here ? hy : ty[q];
        tz[q] = here ? hz : tz[q];
        at[q] = here ? hit : at[q];
      }
      in |= 1u << hit;
      m++;
      continue;
    }
    const T l[4] = {1 - la - lb - lc, la, lb, lc};
    T least = sizeof(T) == 4 ? (T)-1e-5 : (T)-1e-12;
    int out = -1;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const bool take = q < m && l[q] < least;
      least = take ? l[q] : least;
      out = take ? q : out;
    }
    if (out < 0) return m;
    // the last of T takes the place of the one that leaves
    T ex = tx[0], ey = ty[0], ez = tz[0];
    int ei = at[0], oi = at[0];
#pragma unroll
    for (int q = 1; q < 4; ++q) {
      const bool last = q == m - 1;
      ex = last ? tx[q] : ex;
      ey = last ? ty[q] : ey;
      ez = last ? tz[q] : ez;
      ei = last ? at[q] : ei;
      oi = q == out ? at[q] : oi;
    }
    in &= ~(1u << oi);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const bool here = q == out;
      tx[q] = here ? ex : tx[q];
      ty[q] = here ? ey : ty[q];
      tz[q] = here ? ez : tz[q];
      at[q] = here ? ei : at[q];
    }
    m--;
  }
  return 0;
}

// Descents advance one or more steps per round for every arm still
// descending.  Item state lives in SoA arrays of capacity cap: facet ids
// F[q * cap + i] (sorted, not a minimum) and origin arm.
struct DescentItems {
  uint32_t *F, *origin;
  uint64_t cap;
};
// counters of a round: what still descends, what FP32 leaves open, the steps
// taken, what FP64 leaves open
enum { D_OUT = 0, D_OPEN = 1, D_STEPS = 2, D_SLOW = 3 };

// One descent step of facet F (sorted ids): F := F - y + x, where x is the
// least point strictly inside the facet's miniball and y its least support
// point (the miniball strictly shrinks).  Points inside come from the
// neighbour list of the facet point nearest the centre: every point of the
// ball lies within sqrt(R2) + |c - f| of f, so the list holds them all when
// that radius stays below the distance to its last entry (with margins far
// above the FP64 rounding), and its walk ends at the first entry beyond it.
// False: the certified filters or the list cannot decide the step.
template <int K, class T>
__device__ inline bool descent_step(const ArmParams &A, uint32_t (&F)[K]) {
  int at[4] = {0, 0, 0, 0};
  int m;
  {
    const V3 o = P3(A.X, A.Y, A.Z, F[0]);
    T x[K], y[K], z[K];
#pragma unroll
    for (int i = 0; i < K; ++i) {
      const V3 p = sub(P3(A.X, A.Y, A.Z, F[i]), o);
      x[i] = (T)p.x;
      y[i] = (T)p.y;
      z[i] = (T)p.z;
    }
    m = walk_miniball<K, T>(x, y, z, at);
  }
  if (m < 2) return false;
  uint32_t sid[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    sid[j] = F[0];
#pragma unroll
    for (int i = 1; i < K; ++i) sid[j] = at[j] == i ? F[i] : sid[j];
    if (j >= m) sid[j] = kInvalid;
  }
  const V3 o = P3(A.X, A.Y, A.Z, sid[0]);
  const V3 p1 = sub(P3(A.X, A.Y, A.Z, sid[1]), o);
  const V3 p2 = m > 2 ? sub(P3(A.X, A.Y, A.Z, sid[2]), o) : p1;
  const V3 p3 = m > 3 ? sub(P3(A.X, A.Y, A.Z, sid[3]), o) : p1;
  SupSphere S;
  if (!S.init(m, p1, p2, p3)) return false;
  // every facet point must be certainly inside, or a support point
  bool ok = true;
  double best = INFINITY;
  uint32_t f = F[0];
#pragma unroll
  for (int i = 0; i < K; ++i) {
    const V3 p = sub(P3(A.X, A.Y, A.Z, F[i]), o);
    bool on = false;
#pragma unroll
    for (int j = 0; j < 4; ++j) on |= sid[j] == F[i];
    ok = ok && (on || S.side(p) < 0);
    const V3 d = sub(p, S.off);
    const double d2 = dot(d, d);
    f = d2 < best ? F[i] : f;
    best = fmin(best, d2);
  }
  if (!ok || !A.nn) return false;
  const double R2 = dot(S.off, S.off) * (1.0 + 1e-9) + 1e-300;
  const double rho = (sqrt(R2) + sqrt(best)) * (1.0 + 1e-9) + 1e-150, rho2 = rho * rho;
  if (!(rho2 < A.nn_d2[f] * (1.0 - 1e-9))) return false;
  uint32_t xin = kInvalid;
  bool undecided = false;
  const V3 pf = sub(P3(A.X, A.Y, A.Z, f), o);
  const uint4 *row = reinterpret_cast<const uint4 *>(A.nn + (size_t)f * kNearRow);
  bool more = true;
#pragma unroll 1
  for (int j = 0; more && j < kNearRow / 4; ++j) {
    const uint4 r = row[j];
    const uint32_t id4[4] = {r.x, r.y, r.z, r.w};
    V3 p4[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) p4[q] = sub(P3(A.X, A.Y, A.Z, id4[q] == kInvalid ? f : id4[q]), o);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t id = id4[q];
      const V3 e = sub(p4[q], pf), d = sub(p4[q], S.off);
      more = more && id != kInvalid && !(dot(e, e) > rho2 * (1.0 + 1e-9));  // ascending from here on
      if (id == kInvalid || dot(d, d) > R2) continue;
      bool member = false;
#pragma unroll
      for (int i = 0; i < K; ++i) member |= F[i] == id;
      if (member) continue;
      const int sd = S.side(p4[q]);
      xin = sd < 0 ? min(xin, id) : xin;
      undecided |= sd == 0;
    }
  }
  if (undecided || xin == kInvalid) return false;
  uint32_t y = sid[0];
#pragma unroll
  for (int j = 1; j < 4; ++j) y = min(y, sid[j]);
  // F - y + xin, kept sorted: close the gap, bubble xin in
  bool gone = false;
#pragma unroll
  for (int q = 0; q + 1 < K; ++q) {
    gone |= F[q] == y;
    F[q] = gone ? F[q + 1] : F[q];
  }
  F[K - 1] = kInvalid;
#pragma unroll
  for (int q = 0; q < K; ++q) {
    const uint32_t lo = min(F[q], xin);
    xin = max(F[q], xin);
    F[q] = lo;
  }
  return true;
}

// One round of the descents: up to `steps` steps per item, each followed by
// the lookup of the new facet; what still descends goes to `out`, what the
// step leaves open to `slow`.  T = float, then double over what that left open
// (one step).  queue != nullptr: the first round, whose items
// are queued arms.  Bound by the gathers of the neighbours' coordinates and
// the FP64 predicates; Welzl's miniball and a tree traversal per step, with
// the facet in scratch memory, took 66 ms of the 50 000-point tower at 0.22
// lane utilisation (order 10: 28 ms, 7 here).
constexpr int kDescentBlock = 256;
template <int K, class T>
__global__ void __launch_bounds__(kDescentBlock) k_descend(ArmParams A, const uint32_t *queue, DescentItems in,
                                                           uint32_t n_in, DescentItems out, DescentItems slow,
                                                           int steps, unsigned long long *counters) {
  constexpr int kLeft = sizeof(T) == 4 ? D_OPEN : D_SLOW;
  const uint64_t i = (uint64_t)blockIdx.x * kDescentBlock + threadIdx.x;
  bool next = false, open = false;
  uint32_t F[K], origin = 0, done = 0;
  if (i < n_in) {
    if (queue) {
      const uint32_t code = queue[i], s = code >> 2;
      uint32_t L[K + 1];
      load_label<K>(A.sad, s, L);
      drop_point<K>(L, nth_bit(A.sad.members[s], (int)(code & 3u)), F);
      origin = A.sad.base[s] + (code & 3u);
    } else {
      origin = in.origin[i];
#pragma unroll
      for (int q = 0; q < K; ++q) F[q] = in.F[q * in.cap + i];
    }
    next = true;
#pragma unroll 1
    for (int t = 0; next && t < steps; ++t) {
      if (!descent_step<K, T>(A, F)) {
        next = false;
        open = true;
        break;
      }
      done++;
      uint64_t h = 0;
#pragma unroll
      for (int q = 0; q < K; ++q) h += point_mix(F[q]);
      const int64_t hit = lookup<K>(A.table, F, h);
      if (hit >= 0) {
        A.carrier[origin] = (uint32_t)hit;
        next = false;
      }
    }
  }
  const unsigned long long at = block_append<kDescentBlock / 64>(next ? 1u : 0u, counters + D_OUT);
  if (next) {
#pragma unroll
    for (int q = 0; q < K; ++q) out.F[q * out.cap + at] = F[q];
    out.origin[at] = origin;
  }
  (void)block_append<kDescentBlock / 64>(done, counters + D_STEPS);
  const unsigned long long sl = block_append<kDescentBlock / 64>(open ? 1u : 0u, counters + kLeft);
  if (open) {
#pragma unroll
    for (int q = 0; q < K; ++q) slow.F[q * slow.cap + sl] = F[q];
    slow.origin[sl] = origin;
  }
}

// The steps the fast path leaves open, one thread each with the facet in
// scratch memory: Welzl's miniball in FP64, certified containment, and an LBVH
// ball query for the points inside.
struct Ball {
  V3 c;
  double r2;
  int m;
  uint32_t sup[4];  // indices into the facet
};

// circumball of 0..4 facet points with centre in their affine hull (FP64);
// point i of the facet is pts[i * stride]
__device__ bool ball_from(const V3 *pts, int stride, const uint32_t *R, int r, Ball &b) {
  b.m = r;
  for (int i = 0; i < r; ++i) b.sup[i] = R[i];
  if (r == 0) { b.c = {0, 0, 0}; b.r2 = -1; return true; }
  const V3 p0 = pts[R[0] * stride];
  if (r == 1) { b.c = p0; b.r2 = 0; return true; }
  const V3 a = sub(pts[R[1] * stride], p0);
  V3 off;
  if (r == 2) {
    off = {0.5 * a.x, 0.5 * a.y, 0.5 * a.z};
  } else if (r == 3) {
    const V3 bb = sub(pts[R[2] * stride], p0);
    double aa = dot(a, a), b2 = dot(bb, bb), ab = dot(a, bb);
    double D = aa * b2 - ab * ab;
    if (!(D > 1e-14 * (aa * b2 + ab * ab))) return false;
    double al = b2 * (aa - ab), be = aa * (b2 - ab);
    off = {(al * a.x + be * bb.x) / (2 * D), (al * a.y + be * bb.y) / (2 * D), (al * a.z + be * bb.z) / (2 * D)};
  } else {
    const V3 bb = sub(pts[R[2] * stride], p0), d = sub(pts[R[3] * stride], p0);
    V3 bxd = cross(bb, d), dxa = cross(d, a), axb = cross(a, bb);
    double V = dot(a, bxd);
    if (!(fabs(V) > 1e-14 * adot(vabs(a), across(bb, d)))) return false;
    double aa = dot(a, a), b2 = dot(bb, bb), dd = dot(d, d);
    off = {(aa * bxd.x + b2 * dxa.x + dd * axb.x) / (2 * V), (aa * bxd.y + b2 * dxa.y + dd * axb.y) / (2 * V),
           (aa * bxd.z + b2 * dxa.z + dd * axb.z) / (2 * V)};
  }
  b.c = {p0.x + off.x, p0.y + off.y, p0.z + off.z};
  b.r2 = dot(off, off);
  return true;
}

__device__ inline bool in_ball(const Ball &b, const V3 &p) {
  if (b.r2 < 0) return false;
  V3 d = sub(p, b.c);
  return dot(d, d) <= b.r2 * (1.0 + 1e-12) + 1e-300;
}

// Welzl's miniball in its fixed-dimension loop form: level r of the loop nest
// is the recursion level with r boundary points (at most 4 in 3-D), visited in
// the same order as the recursive algorithm.  No recursion, so the kernel's
// private stack has a static size.
__device__ bool welzl(const V3 *pts, int stride, int n, Ball &out) {
  uint32_t R[4];
  Ball b;
  ball_from(pts, stride, R, 0, b);
  for (int i = 0; i < n; ++i) {
    if (in_ball(b, pts[i * stride])) continue;
    R[0] = (uint32_t)i;
    if (!ball_from(pts, stride, R, 1, b)) return false;
    for (int j = 0; j < i; ++j) {
      if (in_ball(b, pts[j * stride])) continue;
      R[1] = (uint32_t)j;
      if (!ball_from(pts, stride, R, 2, b)) return false;
      for (int l = 0; l < j; ++l) {
        if (in_ball(b, pts[l * stride])) continue;
        R[2] = (uint32_t)l;
        if (!ball_from(pts, stride, R, 3, b)) return false;
        for (int q = 0; q < l; ++q) {
          if (in_ball(b, pts[q * stride])) continue;
          R[3] = (uint32_t)q;
          if (!ball_from(pts, stride, R, 4, b)) return false;
        }
      }
    }
  }
  out = b;
  return true;
}

// Sphere of a miniball support (1..4 canonical ids), built once per descent
// step; side() is the certified position of a point (0: on a support point
// or undecided, which sends the arm to the host).
struct SlowSphere {
  int m;
  uint32_t sid[4];
  V3 o;
  union {
    PairSphere ps;
    TriSphere ts;
    TetSphere tt;
  };
  // certified well-centring: +1 yes, -1 no, 0 undecided
  __device__ int init(const double *X, const double *Y, const double *Z, const uint32_t *ids, int mm) {
    m = mm;
    for (int i = 0; i < 4; ++i) sid[i] = i < m ? ids[i] : kInvalid;
    o = P3(X, Y, Z, sid[0]);
    if (m == 2) { ps.init(sub(P3(X, Y, Z, sid[1]), o)); return 1; }
    if (m == 3) return ts.init(sub(P3(X, Y, Z, sid[1]), o), sub(P3(X, Y, Z, sid[2]), o));
    if (m == 4)
      return tt.init(sub(P3(X, Y, Z, sid[1]), o), sub(P3(X, Y, Z, sid[2]), o), sub(P3(X, Y, Z, sid[3]), o));
    return 1;
  }
  __device__ int side(const double *X, const double *Y, const double *Z, uint32_t q) const {
    for (int i = 0; i < m; ++i)
      if (sid[i] == q) return 0;
    if (m == 1) return 1;
    const V3 p = sub(P3(X, Y, Z, q), o);
    if (m == 2) return ps.side(p);
    if (m == 3) return ts.side(p);
    return tt.side(p);
  }
};

constexpr int kSlowBlock = 64;
constexpr int kSlowStack = 40;  // LBVH depth is 18 at 50k points, 32 at 200k; overflow goes to the host

// Trade the miniball's least support point for the least point strictly
// inside; false leaves the arm to the host (shell points, or no point inside:
// a minimum missing from the table).
__device__ bool finish_step(const Ball &b, const uint32_t *sid, int k, uint32_t *F, uint32_t xin, bool undecided) {
  if (undecided || xin == kInvalid) return false;
  uint32_t y = sid[0];
  for (int i = 1; i < b.m; ++i) y = min(y, sid[i]);
  // F := F - y + xin, kept sorted
  int w = 0;
  uint32_t G[kMaxLabel];
  bool placed = false;
  for (int i = 0; i < k; ++i) {
    if (F[i] == y) continue;
    if (!placed && xin < F[i]) { G[w++] = xin; placed = true; }
    G[w++] = F[i];
  }
  if (!placed) G[w++] = xin;
  for (int i = 0; i < k; ++i) F[i] = G[i];
  return true;
}

// stk is the lane's traversal stack in LDS (stride kSlowBlock).  False: the
// certified filters cannot decide the step (the host descends the arm).
__device__ bool slow_step(const ArmParams &A, int k, uint32_t *F, uint32_t *stk, int lane) {
  V3 pts[kMaxLabel];
  for (int i = 0; i < k; ++i) pts[i] = P3(A.X, A.Y, A.Z, F[i]);
  Ball b;
  if (!welzl(pts, 1, k, b)) return false;
  uint32_t sid[4];
  for (int i = 0; i < b.m; ++i) sid[i] = F[b.sup[i]];
  SlowSphere S;
  if (S.init(A.X, A.Y, A.Z, sid, b.m) <= 0) return false;
  // every facet point must be certainly inside, or a support point
  bool ok = true;
  for (int i = 0; i < k && ok; ++i) {
    bool on_support = false;
    for (int q = 0; q < b.m; ++q) on_support |= sid[q] == F[i];
    if (!on_support) ok = S.side(A.X, A.Y, A.Z, F[i]) < 0;
  }
  if (!ok) return false;
  // closed-ball points outside the facet
  uint32_t xin = kInvalid;
  bool undecided = false;
  const double q[3] = {b.c.x, b.c.y, b.c.z};
  const double R2 = b.r2 * (1.0 + 1e-9) + 1e-300;
  // FP32 pruning against outward-rounded child boxes: the radius is
  // inflated by the rounding of the query point and of the FP32 arithmetic
  // (a non-finite bound prunes nothing)
  const float qf[3] = {(float)q[0], (float)q[1], (float)q[2]};
  const double qmax = fmax(fmax(fabs(q[0]), fabs(q[1])), fabs(q[2]));
  const double rb = sqrt(R2) * (1.0 + 1e-6) + qmax * 1e-6 + 1e-30;
  float Tf = (float)(rb * rb * (1.0 + 1e-5));
  if (!(Tf < 3.0e38f)) Tf = INFINITY;
  int sp = 0;
  stk[lane] = 0;
  sp = 1;
  while (sp && !undecided) {
    const WideNode &N = A.wide[stk[(--sp) * kSlowBlock + lane]];
    for (int c = 0; c < 4; ++c) {
      float d2 = 0.f;
      for (int a = 0; a < 3; ++a) {
        const float d = fmaxf(fmaxf(N.lo[c][a] - qf[a], qf[a] - N.hi[c][a]), 0.f);
        d2 += d * d;
      }
      const uint32_t x = N.child[c];
      if (d2 > Tf || x == kInvalid) continue;
      if (x & kLeafBit) {
        const uint32_t lp = x & ~kLeafBit;
        const double dx = A.LX[lp] - q[0], dy = A.LY[lp] - q[1], dz = A.LZ[lp] - q[2];
        if (dx * dx + dy * dy + dz * dz > R2) continue;
        const uint32_t id = A.leaf_id[lp];
        bool inF = false;
        for (int i = 0; i < k; ++i) inF |= F[i] == id;
        if (inF) continue;
        const int sd = S.side(A.X, A.Y, A.Z, id);
        if (sd < 0) xin = min(xin, id);
        else if (sd == 0) undecided = true;
      } else if (sp < kSlowStack) {
        stk[(sp++) * kSlowBlock + lane] = x;
      } else {
        undecided = true;
      }
    }
  }
  return finish_step(b, sid, k, F, xin, undecided);
}

template <int K>
__global__ void __launch_bounds__(kSlowBlock) k_descend_slow(ArmParams A, DescentItems in, DescentItems out,
                                                             unsigned long long *counters) {
  __shared__ uint32_t stk[kSlowStack * kSlowBlock];
  const uint64_t n_in = counters[D_SLOW];  // the launch has threads for more
  const int lane = threadIdx.x;
  const uint64_t i = (uint64_t)blockIdx.x * kSlowBlock + lane;
  bool next = false, stepped = false;
  uint32_t origin = 0, F[K];
  if (i < n_in) {
    origin = in.origin[i];
    uint32_t G[K];
    for (int q = 0; q < K; ++q) G[q] = in.F[q * in.cap + i];
    stepped = slow_step(A, K, G, stk, lane);
    if (stepped) {
      uint64_t h = 0;
      for (int q = 0; q < K; ++q) {
        F[q] = G[q];
        h += point_mix(F[q]);
      }
      const int64_t hit = lookup<K>(A.table, F, h);
      if (hit >= 0) A.carrier[origin] = (uint32_t)hit;
      else next = true;
    } else {
      A.carrier[origin] = kInvalid;  // the host descends this arm
    }
  }
  const unsigned long long at = wave_append(next, counters + D_OUT);
  if (next) {
    for (int q = 0; q < K; ++q) out.F[q * out.cap + at] = F[q];
    out.origin[at] = origin;
  }
  (void)wave_append(stepped, counters + D_STEPS);
}

__global__ void k_arm_owner(uint32_t *__restrict__ base, const uint32_t *__restrict__ sizes_incl,
                            int64_t count, uint32_t *arm_saddle) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  const uint32_t b = i ? sizes_incl[i - 1] : 0u, e = sizes_incl[i];
  base[i] = b;
  for (uint32_t a = b; a < e; ++a) arm_saddle[a] = (uint32_t)i;
}

// Closed labels (support then interior, kInvalid padded to 11) and supports
// of the saddles, for the host's exact descents.
__global__ void k_saddle_labels(const EventRec *__restrict__ ev, const uint32_t *__restrict__ order,
                                const uint32_t *__restrict__ pos, int64_t count, uint32_t *labels,
                                uint32_t *sup) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  const EventRec &e = ev[order[pos[i]]];
  const int m = e.meta & 0xff, ni = (e.meta >> 16) & 0xff;
  int t = 0;
  for (int q = 0; q < m; ++q) labels[(size_t)i * kMaxLabel + t++] = e.ids[q];
  for (int q = 0; q < ni; ++q) labels[(size_t)i * kMaxLabel + t++] = e.interior[q];
  while (t < kMaxLabel) labels[(size_t)i * kMaxLabel + t++] = kInvalid;
  for (int q = 0; q < 4; ++q) sup[4 * i + q] = e.ids[q];
}

// Reduction of an order's saddles before the level-ordered contraction.
//
// first[m] is the least saddle with an arm at minimum m.  A carrier m of
// saddle s is fresh when first[m] == s (an untouched one-minimum component),
// owned otherwise (its component already has a reduced root; order one has
// no fresh minima, every point is born at level zero).
//  * Attachment: every fresh carrier joins, from its first saddle on, the
//    component of that saddle's first owned carrier, or of its first fresh
//    carrier when it has none.  The attachment pointers form a forest (a
//    pointer goes to a minimum first touched strictly earlier, or to a root)
//    and its roots are the representatives.
//  * Owned carriers of one saddle on distinct representatives give star
//    edges, keyed by arm index (level order).  A Boruvka spanning forest over
//    them counts, per saddle, the components its owned carriers join beyond
//    the first.
//  * A saddle at an unshared level with owned carriers and no such forest edge
//    changes no root (silent growth or no new connection) and is dropped; the
//    others (births, multifusions, shared levels) go to the host with their
//    carriers replaced by representatives.
__global__ void k_fill_u32(uint32_t *p, int64_t n, uint32_t v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

__global__ void k_fill_u64(uint64_t *p, int64_t n, uint64_t v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}


__global__ void k_first_touch(const uint32_t *__restrict__ arm_saddle, const uint32_t *__restrict__ carrier,
                              int64_t arms, int64_t minima, uint32_t *first, uint32_t *invalid) {
  int64_t a = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (a >= arms) return;
  const uint32_t c = carrier[a];
  if (c == kInvalid || c >= minima) {
    *invalid = 1u;
    return;
  }
  // arms come in saddle order, so a plain read first spares most atomics
  const uint32_t s = arm_saddle[a];
  if (s < first[c]) atomicMin(&first[c], s);
}

__device__ inline bool carrier_owned(const uint32_t *first, uint32_t c, uint32_t s, int all_owned) {
  return all_owned || first[c] < s;
}

__global__ void k_attach(int64_t S, const uint32_t *__restrict__ base, const uint32_t *__restrict__ incl,
                         const uint32_t *__restrict__ carrier, const uint32_t *__restrict__ first, int all_owned,
                         uint32_t *attach) {
  int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= S) return;
  const uint32_t b = base[s], e = incl[s];
  uint32_t target = kInvalid, fresh0 = kInvalid;
  for (uint32_t a = b; a < e; ++a) {
    const uint32_t c = carrier[a];
    if (carrier_owned(first, c, (uint32_t)s, all_owned)) { target = c; break; }
    if (fresh0 == kInvalid) fresh0 = c;
  }
  if (target == kInvalid) target = fresh0;
  for (uint32_t a = b; a < e; ++a) {
    const uint32_t c = carrier[a];
    if (c != target && !carrier_owned(first, c, (uint32_t)s, all_owned)) attach[c] = target;
  }
}

// Star edges of a saddle, in arm order: from the representative of its first
// owned carrier to each other representative of an owned carrier.  f(r0, r);
// returns their number (at most 3).
//
// A thread per saddle reads each of its up to four carriers once.  A thread
// per arm had to look through the arms before it again, 3.6 arms a saddle, and
// the scan ran over the arms: for 20.6 million arms 1.5 ms,
// now 1.2 ms.
template <class F>
__device__ inline uint32_t star_edges(const uint32_t *base, const uint32_t *incl, const uint32_t *carrier,
                                      const uint32_t *first, const uint32_t *rep, uint32_t s, int all_owned, F f) {
  const uint32_t b = base[s], e = incl[s];
  uint32_t seen[4], n = 0;
#pragma unroll
  for (uint32_t q = 0; q < 4; ++q) {
    if (b + q >= e) continue;
    const uint32_t c = carrier[b + q];
    if (!carrier_owned(first, c, s, all_owned)) continue;
    const uint32_t r = rep[c];
    bool known = false;
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) known |= k < n && seen[k] == r;
    if (known) continue;
    if (n) f(seen[0], r, n - 1);
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) seen[k] = k == n ? r : seen[k];
    n++;
  }
  return n ? n - 1 : 0;
}

__global__ void k_edge_counts(int64_t S, const uint32_t *__restrict__ base, const uint32_t *__restrict__ incl,
                              const uint32_t *__restrict__ carrier, const uint32_t *__restrict__ first,
                              const uint32_t *__restrict__ rep, int all_owned, uint32_t *count) {
  const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= S) return;
  count[s] = star_edges(base, incl, carrier, first, rep, (uint32_t)s, all_owned, [](uint32_t, uint32_t, uint32_t) {});
}

// scan: the saddles' edge counts, inclusive
__global__ void k_edge_list(int64_t S, const uint32_t *__restrict__ base, const uint32_t *__restrict__ incl,
                            const uint32_t *__restrict__ carrier, const uint32_t *__restrict__ first,
                            const uint32_t *__restrict__ rep, int all_owned, const uint32_t *__restrict__ scan,
                            uint32_t *eu, uint32_t *ev, uint32_t *es) {
  const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= S) return;
  const uint32_t at = s ? scan[s - 1] : 0u;
  if (scan[s] == at) return;
  star_edges(base, incl, carrier, first, rep, (uint32_t)s, all_owned, [&](uint32_t r0, uint32_t r, uint32_t j) {
    eu[at + j] = r0;
    ev[at + j] = r;
    es[at + j] = (uint32_t)s;
  });
}

// Edge lists from this length on contract their first quarter first: forest of
// 6.4 million edges (order 10 of a 50 000-point lattice) 5.0 -> 3.0 ms; a
// twelfth or a sixteenth and a quarter first were slower (tower 45.9, 46.9 and
// 48.3 ms).  Shorter lists are bound by launches and waits: three launches a
// round and two rounds a wait, 70 000 edges 0.55 -> 0.27 ms.
constexpr uint32_t kMsfSplit = 1u << 20;

// Counters of one Boruvka round
struct MsfRound {
  unsigned long long live;  // edges that still joined two components
  uint32_t changed, cyclic;
};
constexpr int kMsfRounds = 256;

__global__ void k_msf_init(int64_t M, int64_t E, int64_t S, uint32_t *comp, uint32_t *best, uint32_t *msf,
                           uint32_t *mcount, MsfRound *rounds) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < M) {
    comp[i] = (uint32_t)i;
    best[i] = kInvalid;
  }
  if (i < E) msf[i] = 0u;
  if (i < S) mcount[i] = 0u;
  if (i < kMsfRounds) rounds[i] = MsfRound{0ull, 0u, 0u};
}

// Boruvka round, part 1: least edge (by index) leaving each component.  The
// edges still joining two components are appended to the next round's list.
// The list holds L edges, or *live of them when given (at most L); li ==
// nullptr: it is the edge list from `base` on, edge i at base + i.
constexpr int kMsfBlock = 1024;
__global__ void __launch_bounds__(kMsfBlock) k_msf_best(int64_t L, const unsigned long long *live_in, const uint32_t *__restrict__ lu,
                           const uint32_t *__restrict__ lv, const uint32_t *__restrict__ li, uint32_t base,
                           const uint32_t *__restrict__ comp, uint32_t *best, uint32_t *ou, uint32_t *ov, uint32_t *oi,
                           MsfRound *round) {
  if (live_in) L = min(L, (int64_t)*live_in);
  if ((int64_t)blockIdx.x * kMsfBlock >= L) return;
  const int64_t i = (int64_t)blockIdx.x * kMsfBlock + threadIdx.x;
  uint32_t u = 0, v = 0, idx = 0, cu = 0, cv = 0;
  if (i < L) {
    u = lu[i];
    v = lv[i];
    idx = li ? li[i] : base + (uint32_t)i;
    cu = comp[u];
    cv = comp[v];
  }
  const bool live = i < L && cu != cv;
  if (live) {
    // the list runs in increasing index order, so a plain read first lets most
    // edges of a large component skip an atomic that cannot win
    if (idx < best[cu]) atomicMin(&best[cu], idx);
    if (idx < best[cv]) atomicMin(&best[cv], idx);
  }
  const uint64_t pos = block_append<kMsfBlock / 64>(live ? 1u : 0u, &round->live);
  if (live) {
    ou[pos] = u;
    ov[pos] = v;
    oi[pos] = idx;
  }
}

// Part 2: every component root hooks along its least edge, which is a forest
// edge; of a pair choosing the same edge the smaller root stays a root.  next
// takes the hook forest over all minima.
__global__ void k_msf_hook(int64_t M, const uint32_t *__restrict__ eu, const uint32_t *__restrict__ ev,
                           const uint32_t *__restrict__ comp, const uint32_t *__restrict__ best, uint32_t *next,
                           uint32_t *msf, MsfRound *round) {
  const int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= M) return;
  uint32_t to = comp[m];
  if (to == (uint32_t)m) {
    const uint32_t i = best[m];
    if (i != kInvalid) {
      const uint32_t cu = comp[eu[i]], cv = comp[ev[i]];
      const uint32_t other = cu == (uint32_t)m ? cv : cu;
      msf[i] = 1u;
      if (best[other] != i || (uint32_t)m > other) {
        to = other;
        round->changed = 1u;
      }
    }
  }
  next[m] = to;
}

// Root of m in a forest of parent pointers (a root points to itself, or
// holds kInvalid when nil_root); path halving.  Concurrent threads only ever
// store an ancestor of a node into it, so the forest keeps its roots; the
// roots themselves go to another array.  The walk is bounded by the node
// count: a longer one (a cycle, which a correct forest cannot hold) raises
// *err and returns kInvalid.
__device__ inline uint32_t forest_root(uint32_t *parent, uint32_t m, bool nil_root, int64_t nodes, uint32_t *err) {
  uint32_t x = m;
  for (int64_t step = 0;; ++step) {
    if (step > nodes) {
      *err = 1u;
      return kInvalid;
    }
    const uint32_t p = parent[x];
    if (nil_root ? p == kInvalid : p == x) break;
    const uint32_t g = parent[p];
    if (nil_root ? g == kInvalid : g == p) { x = p; break; }
    parent[x] = g;
    x = g;
  }
  return x;
}

// Part 3: roots of the hook forest into the component array; the least edges
// start again.
__global__ void k_msf_flatten(int64_t M, uint32_t *hooks, uint32_t *comp, uint32_t *best, MsfRound *round) {
  const int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= M) return;
  comp[m] = forest_root(hooks, (uint32_t)m, false, M, &round->cyclic);
  best[m] = kInvalid;
}

__global__ void k_msf_count(int64_t E, const uint32_t *__restrict__ msf, const uint32_t *__restrict__ es,
                            uint32_t *mcount) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < E && msf[i]) atomicAdd(&mcount[es[i]], 1u);
}

// Whether arm a's contraction element (its carrier's representative; the
// carrier itself without representatives) differs from those of the saddle's
// arms before it: the others join nothing new, the host never sees them.
__device__ inline bool first_of_class(const uint32_t *carrier, const uint32_t *rep, uint32_t b, uint32_t a) {
  const uint32_t c = rep ? rep[carrier[a]] : carrier[a];
  for (uint32_t x = b; x < a; ++x)
    if ((rep ? rep[carrier[x]] : carrier[x]) == c) return false;
  return true;
}

__global__ void k_reduce_saddles(int64_t S, const uint32_t *__restrict__ base, const uint32_t *__restrict__ incl,
                                 const uint32_t *__restrict__ carrier, const uint32_t *__restrict__ cls,
                                 const uint32_t *__restrict__ first, const uint32_t *__restrict__ mcount,
                                 const uint32_t *__restrict__ rep, int all_owned, uint32_t *keep,
                                 uint32_t *kept_arms) {
  int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= S) return;
  const uint32_t b = base[s], e = incl[s];
  const uint32_t c = cls[s];
  const bool shared = (s > 0 && cls[s - 1] == c) || (s + 1 < S && cls[s + 1] == c);
  bool k = true;
  if (!shared && mcount[s] == 0) {
    bool any_owned = false;
    for (uint32_t a = b; a < e; ++a) any_owned |= carrier_owned(first, carrier[a], (uint32_t)s, all_owned);
    k = !any_owned;  // no owned carrier: a birth
  }
  keep[s] = k ? 1u : 0u;
  uint32_t distinct = 0;
  for (uint32_t a = b; k && a < e; ++a) distinct += first_of_class(carrier, rep, b, a);
  kept_arms[s] = distinct;
}

__global__ void k_attach_roots(int64_t M, uint32_t *attach, uint32_t *rep, uint32_t *err) {
  int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (m < M) rep[m] = forest_root(attach, (uint32_t)m, true, M, err);
}

// Minima met by a kept saddle get dense ids (flag, then an inclusive scan).
__global__ void k_flag_used(int64_t S, const uint32_t *__restrict__ keep, const uint32_t *__restrict__ base,
                            const uint32_t *__restrict__ incl, const uint32_t *__restrict__ carrier,
                            const uint32_t *__restrict__ rep, uint32_t *used) {
  int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= S || !keep[s]) return;
  for (uint32_t a = base[s]; a < incl[s]; ++a) used[rep[carrier[a]]] = 1u;
}

__global__ void k_compact_saddles(int64_t S, const uint32_t *__restrict__ kpos, const uint32_t *__restrict__ kinc,
                                  const uint32_t *__restrict__ base, const uint32_t *__restrict__ incl,
                                  const uint32_t *__restrict__ carrier, const uint32_t *__restrict__ scls,
                                  const double *__restrict__ slev, const uint32_t *__restrict__ rep,
                                  const uint32_t *__restrict__ dense, uint32_t *o_cls, double *o_lev, uint32_t *o_base,
                                  uint32_t *o_car) {
  int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= S) return;
  const uint32_t prev = s ? kpos[s - 1] : 0u;
  if (kpos[s] == prev) return;  // dropped
  const uint32_t b = base[s], e = incl[s];
  const uint32_t p = prev;
  uint32_t nb = s ? kinc[s - 1] : 0u;
  o_cls[p] = scls[s];
  o_lev[p] = slev[s];
  o_base[p] = nb;
  for (uint32_t a = b; a < e; ++a)
    if (first_of_class(carrier, rep, b, a)) o_car[nb++] = rep ? dense[rep[carrier[a]]] - 1u : carrier[a];
}

// Vertical maps: the order-k contraction element (dense representative id;
// the minimum itself for order one or when the host descends) of the first
// arm's carrier of every order-k saddle, stored at the saddle's rank-index
// position, which is also its position as a minimum of order k + 1.
__global__ void k_vm_elem(int64_t S, const uint32_t *__restrict__ base, const uint32_t *__restrict__ carrier,
                          const uint32_t *__restrict__ rep, const uint32_t *__restrict__ dense, uint32_t *out) {
  int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= S) return;
  const uint32_t c = carrier[base[s]];
  out[s] = (rep && c != kInvalid) ? dense[rep[c]] - 1u : c;
}

// Raw minimum of every dense representative id (the inverse of dense - 1).
__global__ void k_raw_of_dense(int64_t M, const uint32_t *__restrict__ dense, uint32_t *out) {
  int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= M) return;
  const uint32_t prev = m ? dense[m - 1] : 0u;
  if (dense[m] != prev) out[prev] = (uint32_t)m;
}

// FP64 squared distance from every point to the last of its `listed`
// neighbours; infinite when the list holds every other point.
__global__ void k_nn_last_d2(int64_t n, int listed, const uint32_t *__restrict__ nn, const double *__restrict__ X,
                             const double *__restrict__ Y, const double *__restrict__ Z, double *d2) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const uint32_t q = nn[p * kNearRow + listed - 1];
  if (listed == n - 1 || q >= (uint64_t)n) {
    d2[p] = q >= (uint64_t)n ? 0.0 : INFINITY;  // 0: never used
    return;
  }
  const double dx = X[q] - X[p], dy = Y[q] - Y[p], dz = Z[q] - Z[p];
  d2[p] = dx * dx + dy * dy + dz * dz;
}

__global__ void k_give_up(const uint32_t *__restrict__ origin, uint32_t n, uint32_t *carrier) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) carrier[origin[i]] = kInvalid;
}

// Vertical maps of a large order pair: targets by ancestor doubling.  up[0] is
// the parent of every node of the order below (-1: none); level j holds the
// 2^j-th ancestor.
__global__ void k_double_up(int64_t n, const int32_t *__restrict__ below, int32_t *above) {
  const int64_t x = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= n) return;
  const int32_t p = below[x];
  above[x] = p < 0 ? -1 : below[p];
}

// Node i (level class L) starts at the node that first owned the class of
// its element and climbs to that node's highest ancestor at or below L
// (levels never decrease towards a root).
struct VerticalPair {
  const int64_t *s_cls;      // order o: level class per node
  const int32_t *s_rep;      // representative element per node
  const uint32_t *s_raw;     // raw minimum of each element (null: identity)
  int64_t s_nodes, s_raws;
  uint32_t base, span;       // rank-index range of order o's minima
  const uint32_t *elem;      // element of the order below per rank-index position
  const int64_t *t_cls;      // order o - 1
  const int32_t *t_acq;      // per element: node that first owned its class
  const int64_t *t_acq_cls;  // and its level class
  int64_t t_nodes, t_elems;
  const int32_t *up;         // levels x t_nodes
  int levels;
};

__global__ void k_vertical(VerticalPair V, int64_t *target, uint32_t *error) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= V.s_nodes) return;
  const int64_t L = V.s_cls[i];
  int64_t x = -1;
  const int32_t r = V.s_rep[i];
  if (r >= 0 && (!V.s_raw || r < V.s_raws)) {
    const uint32_t raw = V.s_raw ? V.s_raw[r] : (uint32_t)r;
    if (raw < V.span) {
      const uint32_t e = V.elem[V.base + raw];
      if (e < (uint64_t)V.t_elems && V.t_acq[e] >= 0 && V.t_acq[e] < V.t_nodes && V.t_acq_cls[e] <= L) x = V.t_acq[e];
    }
  }
  if (x < 0) {
    *error = 1u;
    return;
  }
  for (int j = V.levels - 1; j >= 0; --j) {
    const int32_t a = V.up[(int64_t)j * V.t_nodes + x];
    if (a >= 0 && V.t_cls[a] <= L) x = a;
  }
  target[i] = x;
}

__global__ void k_gather_u32(const uint32_t *__restrict__ src, const uint32_t *__restrict__ idx, int64_t n,
                             uint32_t *out) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = src[idx[i]];
}

}  // namespace

void tower_vm_gather(Context &c, const std::vector<uint32_t> &pos, std::vector<uint32_t> &out) {
  TowerWork &R = *c.tower_work;
  const int64_t q = (int64_t)pos.size();
  out.assign(q, kInvalid);
  if (!q) return;
  if (!R.vm_stream) MHGP_HIP(hipStreamCreateWithFlags(&R.vm_stream, hipStreamNonBlocking));
  hipStream_t s = R.vm_stream;
  R.vm_idx.ensure(q);
  R.vm_out.ensure(q);
  MHGP_HIP(hipMemcpyAsync(R.vm_idx.p, pos.data(), q * 4, hipMemcpyHostToDevice, s));
  hipLaunchKernelGGL(k_gather_u32, dim3(blocks_for(q, 256)), dim3(256), 0, s, R.vm_elem.p, R.vm_idx.p, q, R.vm_out.p);
  MHGP_LAUNCH_CHECK();
  copy_wait(out.data(), R.vm_out.p, q * 4, hipMemcpyDeviceToHost, s);
}

bool tower_vm_targets(Context &c, const Forest &S, const Forest &T, uint32_t base, uint32_t span,
                      std::vector<int64_t> &target) {
  const int64_t m = (int64_t)S.order.size(), tm = (int64_t)T.order.size(), te = (int64_t)T.acq_node.size();
  if (m < kVerticalOnDevice || tm < 2) return false;
  TowerWork &R = *c.tower_work;
  if (!R.vm_stream) MHGP_HIP(hipStreamCreateWithFlags(&R.vm_stream, hipStreamNonBlocking));
  hipStream_t s = R.vm_stream;
  int levels = 1;
  while ((1ll << levels) < tm) ++levels;
  const int64_t raws = (int64_t)S.raw_of_dense.size();
  // eight-byte words, then four-byte ones
  R.vm_long.ensure((size_t)(2 * m + tm + te));
  R.vm_int.ensure((size_t)(m + raws + te + levels * tm + 1));
  int64_t *s_cls = R.vm_long.p, *d_target = s_cls + m, *t_cls = d_target + m, *t_acq_cls = t_cls + tm;
  int32_t *s_rep = R.vm_int.p, *s_raw = s_rep + m, *t_acq = s_raw + raws, *up = t_acq + te, *err = up + levels * tm;
  auto put = [&](void *d, const void *h, size_t bytes) {
    if (bytes) MHGP_HIP(hipMemcpyAsync(d, h, bytes, hipMemcpyHostToDevice, s));
  };
  put(s_cls, S.level_class.data(), m * 8);
  put(t_cls, T.level_class.data(), tm * 8);
  put(t_acq_cls, T.acq_cls.data(), te * 8);
  put(s_rep, S.rep_elem.data(), m * 4);
  put(s_raw, S.raw_of_dense.data(), raws * 4);
  put(t_acq, T.acq_node.data(), te * 4);
  put(up, T.parent.data(), tm * 4);
  hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(64), 0, s, (uint32_t *)err, (int64_t)1, 0u);
  for (int j = 1; j < levels; ++j)
    hipLaunchKernelGGL(k_double_up, dim3(blocks_for(tm, 256)), dim3(256), 0, s, tm, up + (int64_t)(j - 1) * tm,
                       up + (int64_t)j * tm);
  const VerticalPair V{s_cls, s_rep, raws ? (const uint32_t *)s_raw : nullptr, m, raws, base, span, R.vm_elem.p,
                       t_cls, t_acq, t_acq_cls, tm, te, up, levels};
  hipLaunchKernelGGL(k_vertical, dim3(blocks_for(m, 256)), dim3(256), 0, s, V, d_target, (uint32_t *)err);
  MHGP_LAUNCH_CHECK();
  target.resize(m);
  uint32_t bad = 0;
  MHGP_HIP(hipMemcpyAsync(&bad, err, 4, hipMemcpyDeviceToHost, s));
  copy_wait(target.data(), d_target, m * 8, hipMemcpyDeviceToHost, s);
  if (bad) throw std::runtime_error("vertical map: the order below holds no owned class at the node's level");
  return true;
}

void tower_vm_store(Context &c, hipStream_t s, uint32_t first_pos, const std::vector<uint32_t> &elems) {
  if (elems.empty()) return;
  copy_wait(c.tower_work->vm_elem.p + first_pos, elems.data(), elems.size() * 4, hipMemcpyHostToDevice, s);
}

void tower_prefetch_neighbours(Context &c) {
  if (c.n < 2) return;
  const int listed = (int)std::min<int64_t>(kNearK, c.n - 1);
  if (!c.tower_work) c.tower_work = std::make_unique<TowerWork>();
  TowerWork &W = *c.tower_work;
  if (!W.vm_stream) MHGP_HIP(hipStreamCreateWithFlags(&W.vm_stream, hipStreamNonBlocking));
  if (!W.nn_start) {
    MHGP_HIP(hipEventCreateWithFlags(&W.nn_start, hipEventDisableTiming));
    MHGP_HIP(hipEventCreateWithFlags(&W.nn_done, hipEventDisableTiming));
  }
  W.nn.ensure((size_t)c.n * kNearRow);
  W.nn_d2.ensure(c.n);
  W.nn_flags.ensure(c.n);
  // the side stream starts after the context stream's work so far (the LBVH)
  MHGP_HIP(hipEventRecord(W.nn_start, c.stream));
  MHGP_HIP(hipStreamWaitEvent(W.vm_stream, W.nn_start, 0));
  knn_all(c, listed, W.nn.p, W.nn_flags.p, W.vm_stream, kNearRow);
  hipLaunchKernelGGL(k_nn_last_d2, dim3(blocks_for(c.n, 256)), dim3(256), 0, W.vm_stream, c.n, listed, W.nn.p,
                     c.X.p, c.Y.p, c.Z.p, W.nn_d2.p);
  MHGP_LAUNCH_CHECK();
  MHGP_HIP(hipEventRecord(W.nn_done, W.vm_stream));
  W.nn_pending = true;
}

void tower_rank_index(Context &c) {
  CatalogBuffers &B = *c.catalog;
  hipStream_t s = c.stream;
  const int64_t n = B.count;
  if (!c.tower_work) c.tower_work = std::make_unique<TowerWork>();
  TowerWork &W = *c.tower_work;
  std::fill(W.rank_lo, W.rank_lo + 256, 0u);
  std::fill(W.rank_hi, W.rank_hi + 256, 0u);
  if (n == 0) return;
  W.rank_keys.ensure(n);
  W.rank_vals.ensure(n);
  W.vm_elem.ensure(n);
  // neighbour lists of the points, for the descents' ball queries: started
  // beside the level order, or computed here
  W.nn_ready = false;
  if (c.n >= 2) {
    if (!W.nn_pending) tower_prefetch_neighbours(c);
    MHGP_HIP(hipStreamWaitEvent(s, W.nn_done, 0));
    W.nn_pending = false;
    W.nn_ready = true;
  }
  W.rank_bounds.ensure(512);
  hipLaunchKernelGGL(k_rank_keys, dim3(blocks_for(n, 256)), dim3(256), 0, s, B.events.p, B.order.p, n,
                     W.rank_keys.p, W.rank_vals.p);
  c.sorter.sort(W.rank_keys.p, W.rank_vals.p, n, 0, 8, s);
  hipLaunchKernelGGL(k_fill_u32, dim3(2), dim3(256), 0, s, W.rank_bounds.p, (int64_t)512, 0u);
  hipLaunchKernelGGL(k_rank_bounds, dim3(blocks_for(n, 256)), dim3(256), 0, s, W.rank_keys.p, n, W.rank_bounds.p,
                     W.rank_bounds.p + 256);
  uint32_t h[512];
  copy_wait(h, W.rank_bounds.p, sizeof h, hipMemcpyDeviceToHost, s);
  std::copy(h, h + 256, W.rank_lo);
  std::copy(h + 256, h + 512, W.rank_hi);
  for (int r = 0; r < 256; ++r)
    if (W.rank_lo[r] > W.rank_hi[r] || W.rank_hi[r] > (uint64_t)n) throw std::runtime_error("malformed rank index");
}

// Calls f.template operator()<K>() for K = k.
template <class F>
void with_order(int k, F &&f) {
  switch (k) {
    case 1: f(std::integral_constant<int, 1>{}); break;
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 3: f(std::integral_constant<int, 3>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 5: f(std::integral_constant<int, 5>{}); break;
    case 6: f(std::integral_constant<int, 6>{}); break;
    case 7: f(std::integral_constant<int, 7>{}); break;
    case 8: f(std::integral_constant<int, 8>{}); break;
    case 9: f(std::integral_constant<int, 9>{}); break;
    case 10: f(std::integral_constant<int, 10>{}); break;
    default: throw std::logic_error("tower order beyond 10");
  }
}

void tower_order_device(Context &c, TowerWork &W, const TowerWork &R, int k, TowerOrderData &out) {
  CatalogBuffers &B = *c.catalog;
  hipStream_t s = W.stream;
  out = TowerOrderData{};
  // host clock at the synchronisations that end each phase (MHGP_TIMING)
  using clk = std::chrono::steady_clock;
  clk::time_point ph[8];
  for (auto &x : ph) x = clk::now();
  // minima of order k (k >= 2) and saddles of order k: records of closed
  // rank k and k + 1, as runs of the rank index
  const uint32_t M = R.rank_hi[k] - R.rank_lo[k], S = R.rank_hi[k + 1] - R.rank_lo[k + 1];
  const uint32_t *minima_pos = R.rank_vals.p + R.rank_lo[k], *saddle_pos = R.rank_vals.p + R.rank_lo[k + 1];
  out.minima = M;
  uint64_t cap = 1;
  while (cap < 2ull * M + 16) cap <<= 1;
  auto &slots = W.slots;
  auto &labels = W.labels;
  slots.ensure(cap);
  labels.ensure((size_t)M * k + 1);
  const MinimaTable table{(unsigned long long *)slots.p, cap - 1, labels.p};
  hipLaunchKernelGGL(k_fill_u64, dim3(blocks_for((int64_t)cap, 256)), dim3(256), 0, s, slots.p, (int64_t)cap, 0ull);
  if (M)
    with_order(k, [&](auto K) {
      hipLaunchKernelGGL((k_insert_minima<K.value>), dim3(blocks_for(M, 256)), dim3(256), 0, s, B.events.p, B.order.p,
                         minima_pos, (int64_t)M, table);
    });
  out.saddles = S;
  if (S == 0) return;
  if (S >= (1u << 30)) throw CapacityError("an order of the tower has more saddles than the arm codes hold");
  auto &sizes = W.sizes, &carrier = W.carrier, &scls = W.scls;
  auto &slev = W.slev;
  sizes.ensure(S);
  scls.ensure(S);
  slev.ensure(S);
  W.members.ensure(S);
  // the saddles' labels; the pool's words serve the spanning forest later
  auto &base = W.base;
  base.ensure(S);
  const Saddles sad{W.slab.ensure((size_t)S * (k + 1)), W.members.p, base.p};
  with_order(k, [&](auto K) {
    hipLaunchKernelGGL((k_saddles<K.value>), dim3(blocks_for(S, 256)), dim3(256), 0, s, B.events.p, B.order.p, B.cls.p,
                       saddle_pos, (int64_t)S, sad, sizes.p, scls.p, slev.p);
  });
  W.scanner.inclusive(sizes.p, S, s);
  uint32_t arms = 0;
  copy_wait(&arms, sizes.p + S - 1, 4, hipMemcpyDeviceToHost, s);
  ph[1] = ph[2] = ph[3] = clk::now();
  carrier.ensure(arms);
  auto &arm_saddle = W.arm_saddle;
  arm_saddle.ensure(arms);
  // exclusive bases (the inclusive scan shifted by one) and the arms' saddles
  hipLaunchKernelGGL(k_arm_owner, dim3(blocks_for(S, 256)), dim3(256), 0, s, base.p, sizes.p, (int64_t)S,
                     arm_saddle.p);
  ArmParams A{};
  A.sad = sad;
  A.saddles = S;
  A.table = table;
  A.X = c.X.p; A.Y = c.Y.p; A.Z = c.Z.p;
  A.wide = c.wide.p; A.LX = c.LX.p; A.LY = c.LY.p; A.LZ = c.LZ.p; A.leaf_id = c.leaf_id.p; A.leaf_pos = c.leaf_pos.p;
  A.carrier = carrier.p;
  A.nn = R.nn_ready ? R.nn.p : nullptr;
  A.nn_d2 = R.nn_ready ? R.nn_d2.p : nullptr;
  auto &queue = W.queue;
  queue.ensure(arms);
  W.clock.start(s);
  auto &qkey = W.qkey;
  qkey.ensure(arms);
  // distinct facets of the arms to descend (load factor below 1/2)
  uint64_t fcap = 1;
  while (fcap < 2ull * arms + 16) fcap <<= 1;
  W.facet_slots.ensure(fcap);
  W.alias_arm.ensure(arms);
  W.alias_rep.ensure(arms);
  W.dcount.ensure(4);
  hipLaunchKernelGGL(k_fill_u64, dim3(blocks_for((int64_t)fcap, 256)), dim3(256), 0, s, W.facet_slots.p,
                     (int64_t)fcap, 0ull);
  hipLaunchKernelGGL(k_fill_u64, dim3(1), dim3(64), 0, s, W.dcount.p, (int64_t)4, 0ull);
  unsigned long long *counters = (unsigned long long *)W.dcount.p;
  const FacetSet D{(unsigned long long *)W.facet_slots.p, fcap - 1, W.alias_arm.p, W.alias_rep.p, counters + 1};
  with_order(k, [&](auto K) {
    hipLaunchKernelGGL((k_arm_lookup<K.value>), dim3(blocks_for(S, kArmBlock)), dim3(kArmBlock), 0, s, A, D, queue.p,
                       qkey.p, counters);
  });
  uint64_t got[4] = {0, 0, 0, 0};
  copy_wait(got, W.dcount.p, 16, hipMemcpyDeviceToHost, s);
  const uint64_t nq = got[0], na = got[1];
  ph[2] = ph[3] = clk::now();
  if (nq > 1) {  // spatial order: neighbouring lanes read neighbouring lists
    int bits = 8;
    while (bits < 32 && (1ll << bits) < c.n) bits += 8;
    W.sorter.sort(qkey.p, queue.p, (int64_t)nq, 0, bits, s);
  }
  uint64_t steps_total = 0, slow_total = 0;
  if (nq && k >= 2) {
    DescentItems items[3];  // two rounds' items, and what FP32 leaves open
    for (int q = 0; q < 3; ++q) {
      W.dF[q].ensure((size_t)k * nq);
      W.dO[q].ensure(nq);
      items[q] = DescentItems{W.dF[q].p, W.dO[q].p, nq};
    }
    uint32_t active = (uint32_t)nq;
    for (int round = 0; active > 0; ++round) {
      const int q = round & 1;
      if (round > 4096) {  // the host descends what is left
        hipLaunchKernelGGL(k_give_up, dim3(blocks_for(active, 256)), dim3(256), 0, s, items[q ^ 1].origin, active,
                           carrier.p);
        break;
      }
      // a small round is bound by its launch and wait, not by idle lanes:
      // several steps in one
      const int steps = active <= 1u << 17 ? 8 : 1;
      hipLaunchKernelGGL(k_fill_u64, dim3(1), dim3(64), 0, s, W.dcount.p, (int64_t)4, 0ull);
      with_order(k, [&](auto K) {
        hipLaunchKernelGGL((k_descend<K.value, float>), dim3(blocks_for(active, kDescentBlock)), dim3(kDescentBlock), 0,
                           s, A, round == 0 ? queue.p : nullptr, items[q ^ 1], active, items[q], items[2], steps, counters);
      });
      copy_wait(got, W.dcount.p, sizeof got, hipMemcpyDeviceToHost, s);
      if (const uint32_t open = (uint32_t)got[D_OPEN]) {
        // the round's input is done: its list takes what FP64 leaves open too
        with_order(k, [&](auto K) {
          hipLaunchKernelGGL((k_descend<K.value, double>), dim3(blocks_for(open, kDescentBlock)), dim3(kDescentBlock), 0, s,
                             A, nullptr, items[2], open, items[q], items[q ^ 1], 1, counters);
          hipLaunchKernelGGL((k_descend_slow<K.value>), dim3(blocks_for(open, kSlowBlock)), dim3(kSlowBlock), 0, s, A,
                             items[q ^ 1], items[q], counters);
        });
        copy_wait(got, W.dcount.p, sizeof got, hipMemcpyDeviceToHost, s);
        slow_total += got[D_SLOW];
      }
      steps_total += got[D_STEPS];
      active = (uint32_t)got[D_OUT];
    }
    ph[3] = clk::now();
  }
  if (na)
    hipLaunchKernelGGL(k_alias_carriers, dim3(blocks_for(na, 256)), dim3(256), 0, s, W.alias_arm.p, W.alias_rep.p,
                       na, carrier.p);
  W.clock.stop(s);
  MHGP_LAUNCH_CHECK();
  W.arm_ms += W.clock.ms();
  W.arm_launches++;
  // algorithmic bytes: each saddle record and its order/position entries read
  // once, each arm's carrier written once and one hash probe (key + value)
  W.arm_bytes += (int64_t)S * ((int64_t)sizeof(EventRec) + 8) + (int64_t)arms * (4 + 12);
  // drop the saddles that cannot change the contraction (unless the host
  // must descend some arms: then every saddle goes down as it is)
  const int64_t minima_n = k == 1 ? c.n : (int64_t)M;
  auto &first = W.first, &keep = W.keep, &kept = W.kept, &flag1 = W.flag1;
  first.ensure(minima_n);
  keep.ensure(S);
  kept.ensure(S);
  flag1.ensure(1);
  MHGP_HIP(hipMemsetAsync(flag1.p, 0, 4, s));
  hipLaunchKernelGGL(k_fill_u32, dim3(blocks_for(minima_n, 256)), dim3(256), 0, s, first.p, minima_n, kInvalid);
  hipLaunchKernelGGL(k_first_touch, dim3(blocks_for(arms, 256)), dim3(256), 0, s, arm_saddle.p, carrier.p,
                     (int64_t)arms, minima_n, first.p, flag1.p);
  uint32_t any_invalid = 0;
  copy_wait(&any_invalid, flag1.p, 4, hipMemcpyDeviceToHost, s);
  ph[4] = ph[5] = ph[6] = clk::now();
  uint32_t S2 = S, arms2 = arms;
  const uint32_t *d_cls = scls.p, *d_base = base.p, *d_car = carrier.p;
  const double *d_lev = slev.p;
  auto &c_cls = W.c_cls, &c_base = W.c_base, &c_car = W.c_car;
  auto &c_lev = W.c_lev;
  uint32_t msf_edges = 0;
  int msf_rounds = 0;
  if (!any_invalid) {
    const dim3 tb(256);
    const int all_owned = k == 1 ? 1 : 0;
    const dim3 gm(blocks_for(minima_n, 256)), gs(blocks_for(S, 256));
    // attachment forest of the fresh minima and its representatives
    auto &attach = W.attach, &rep = W.rep, &dense = W.dense, &err = W.err;
    attach.ensure(minima_n);
    rep.ensure(minima_n);
    err.ensure(1);
    hipLaunchKernelGGL(k_fill_u32, dim3(1), tb, 0, s, err.p, (int64_t)1, 0u);
    hipLaunchKernelGGL(k_fill_u32, gm, tb, 0, s, attach.p, minima_n, kInvalid);
    hipLaunchKernelGGL(k_attach, gs, tb, 0, s, (int64_t)S, base.p, sizes.p, carrier.p, first.p, all_owned, attach.p);
    hipLaunchKernelGGL(k_attach_roots, gm, tb, 0, s, minima_n, attach.p, rep.p, err.p);
    // star edges between the representatives of owned carriers, in arm (= level) order
    auto &eflag = W.eflag;
    eflag.ensure(S);
    hipLaunchKernelGGL(k_edge_counts, gs, tb, 0, s, (int64_t)S, base.p, sizes.p, carrier.p, first.p, rep.p, all_owned,
                       eflag.p);
    W.scanner.inclusive(eflag.p, S, s);
    uint32_t E = 0, bad = 0;
    MHGP_HIP(hipMemcpyAsync(&bad, err.p, 4, hipMemcpyDeviceToHost, s));
    copy_wait(&E, eflag.p + S - 1, 4, hipMemcpyDeviceToHost, s);
    if (bad) throw std::runtime_error("tower attachment forest is cyclic");
    ph[5] = ph[6] = clk::now();
    // edges and two rounds' lists, in the pool that held the saddles' labels
    uint32_t *pool = W.slab.ensure(9 * (size_t)E);
    uint32_t *eu = pool, *ev = eu + E, *es = ev + E;
    uint32_t *Lu[2] = {es + E, es + 4 * (size_t)E}, *Lv[2] = {Lu[0] + E, Lu[1] + E}, *Li[2] = {Lv[0] + E, Lv[1] + E};
    hipLaunchKernelGGL(k_edge_list, gs, tb, 0, s, (int64_t)S, base.p, sizes.p, carrier.p, first.p, rep.p, all_owned,
                       eflag.p, eu, ev, es);
    // Boruvka spanning forest of the minima over the star edges.  Edges are in
    // level order, so of a long list a prefix is contracted first: most of the
    // rest then lies within components and only passes the filter once,
    // instead of through several rounds.  Two rounds share a wait; the second
    // takes its list's length from the device.
    auto &comp = W.comp, &hooks = W.comp2, &best = W.best, &msf = W.msf;
    auto &mcount = W.mcount;
    auto &rounds = W.rounds;
    rounds.ensure(kMsfRounds * sizeof(MsfRound));
    MsfRound *slot = reinterpret_cast<MsfRound *>(rounds.p);
    comp.ensure(minima_n);
    hooks.ensure(minima_n);
    best.ensure(minima_n);
    msf.ensure(E + 1);
    mcount.ensure(S);
    const dim3 ge(blocks_for(E + 1, 256));
    hipLaunchKernelGGL(k_msf_init, dim3(blocks_for(std::max<int64_t>({minima_n, E, S, kMsfRounds}), 256)), tb, 0, s,
                       minima_n, (int64_t)E, (int64_t)S, comp.p, best.p, msf.p, mcount.p, slot);
    msf_edges = E;
    const uint32_t prefix = E >= kMsfSplit ? E / 4 : E;
    int used = 0;
    for (uint32_t lo = 0, hi = prefix; lo < E; lo = hi, hi = E) {
      const uint32_t *lu = eu + lo, *lv = ev + lo, *li = nullptr;
      uint32_t live = hi - lo;
      while (live > 0) {
        if (used + 2 > kMsfRounds) throw std::runtime_error("spanning forest of the tower did not converge");
        for (int q = 0; q < 2; ++q) {
          MsfRound *r = slot + used + q;
          hipLaunchKernelGGL(k_msf_best, dim3(blocks_for(live, kMsfBlock)), dim3(kMsfBlock), 0, s, (int64_t)live,
                             q ? &r[-1].live : nullptr, lu, lv, li, lo, comp.p, best.p, Lu[q], Lv[q], Li[q], r);
          hipLaunchKernelGGL(k_msf_hook, gm, tb, 0, s, minima_n, eu, ev, comp.p, best.p, hooks.p, msf.p, r);
          hipLaunchKernelGGL(k_msf_flatten, gm, tb, 0, s, minima_n, hooks.p, comp.p, best.p, r);
          lu = Lu[q];
          lv = Lv[q];
          li = Li[q];
        }
        MsfRound got[2];
        copy_wait(got, slot + used, sizeof got, hipMemcpyDeviceToHost, s);
        used += 2;
        if (got[0].cyclic || got[1].cyclic) throw std::runtime_error("spanning forest of the tower: cyclic hook forest");
        if (!got[0].changed || !got[1].changed) break;
        live = (uint32_t)got[1].live;
      }
    }
    msf_rounds = used;
    ph[6] = clk::now();
    if (E) hipLaunchKernelGGL(k_msf_count, ge, tb, 0, s, (int64_t)E, msf.p, es, mcount.p);
    // keep births, multifusions and shared levels
    const uint32_t *d_rep = k >= 2 ? rep.p : nullptr, *d_dense = nullptr;  // order one keeps point ids: every point is born
    hipLaunchKernelGGL(k_reduce_saddles, gs, tb, 0, s, (int64_t)S, base.p, sizes.p, carrier.p, scls.p, first.p,
                       mcount.p, d_rep, all_owned, keep.p, kept.p);
    uint32_t Mdense = (uint32_t)minima_n;
    if (k >= 2) {
      dense.ensure(minima_n);
      hipLaunchKernelGGL(k_fill_u32, gm, tb, 0, s, dense.p, minima_n, 0u);
      hipLaunchKernelGGL(k_flag_used, gs, tb, 0, s, (int64_t)S, keep.p, base.p, sizes.p, carrier.p, rep.p, dense.p);
      W.scanner.inclusive(dense.p, minima_n, s);
      copy_wait(&Mdense, dense.p + minima_n - 1, 4, hipMemcpyDeviceToHost, s);
      d_dense = dense.p;
      // dense id -> raw minimum, for the vertical maps out of this order
      W.raw_dense.ensure(Mdense + 1);
      hipLaunchKernelGGL(k_raw_of_dense, gm, tb, 0, s, minima_n, dense.p, W.raw_dense.p);
      out.raw_of_dense.resize(Mdense);
      if (Mdense) copy_wait(out.raw_of_dense.data(), W.raw_dense.p, (size_t)Mdense * 4, hipMemcpyDeviceToHost, s);
    }
    hipLaunchKernelGGL(k_vm_elem, gs, tb, 0, s, (int64_t)S, base.p, carrier.p, d_rep, d_dense,
                       R.vm_elem.p + R.rank_lo[k + 1]);
    W.scanner.inclusive(keep.p, S, s);
    W.scanner.inclusive(kept.p, S, s);
    MHGP_HIP(hipMemcpyAsync(&S2, keep.p + S - 1, 4, hipMemcpyDeviceToHost, s));
    MHGP_HIP(hipMemcpyAsync(&arms2, kept.p + S - 1, 4, hipMemcpyDeviceToHost, s));
    MHGP_HIP(hipStreamSynchronize(s));
    c_cls.ensure(S2);
    c_lev.ensure(S2);
    c_base.ensure(S2);
    c_car.ensure(arms2);
    hipLaunchKernelGGL(k_compact_saddles, dim3(blocks_for(S, 256)), tb, 0, s, (int64_t)S, keep.p, kept.p, base.p,
                       sizes.p, carrier.p, scls.p, slev.p, d_rep, d_dense, c_cls.p, c_lev.p, c_base.p, c_car.p);
    d_cls = c_cls.p;
    d_lev = c_lev.p;
    d_base = c_base.p;
    d_car = c_car.p;
    if (k >= 2) out.minima = Mdense;
  }
  // page-locked results: cls | arm_base | carrier | level
  const size_t o_base = (size_t)S2 * 4, o_car = o_base + ((size_t)S2 + 1) * 4;
  const size_t o_lev = (o_car + (size_t)arms2 * 4 + 7) & ~(size_t)7;
  char *h = (char *)c.tower_pinned[k].ensure(o_lev + (size_t)S2 * 8 + 8);
  uint32_t *h_cls = (uint32_t *)h, *h_base = (uint32_t *)(h + o_base), *h_car = (uint32_t *)(h + o_car);
  double *h_lev = (double *)(h + o_lev);
  if (S2) {
    MHGP_HIP(hipMemcpyAsync(h_cls, d_cls, (size_t)S2 * 4, hipMemcpyDeviceToHost, s));
    MHGP_HIP(hipMemcpyAsync(h_base, d_base, (size_t)S2 * 4, hipMemcpyDeviceToHost, s));
    MHGP_HIP(hipMemcpyAsync(h_car, d_car, (size_t)arms2 * 4, hipMemcpyDeviceToHost, s));
    MHGP_HIP(hipMemcpyAsync(h_lev, d_lev, (size_t)S2 * 8, hipMemcpyDeviceToHost, s));
  }
  const uint64_t st = steps_total;
  MHGP_HIP(hipStreamSynchronize(s));
  ph[7] = clk::now();
  h_base[S2] = arms2;
  out.saddles = S2;
  out.cls = h_cls;
  out.arm_base = h_base;
  out.carrier = h_car;
  out.level = h_lev;
  out.arms = arms2;
  out.steps = (int64_t)st;
  if (std::getenv("MHGP_TIMING"))
    std::fprintf(stderr,
                 "[mhgp] arms order %2d: %u saddles, %u arms, %llu descending, %llu steps (%llu slow), %u forest edges in %d "
                 "rounds, %u kept | ms: setup %.2f lookup %.2f descents %.2f first %.2f edges %.2f forest %.2f "
                 "tail %.2f\n",
                 k, S, arms, (unsigned long long)nq, (unsigned long long)st, (unsigned long long)slow_total, msf_edges, msf_rounds, S2,
                 std::chrono::duration<double, std::milli>(ph[1] - ph[0]).count(),
                 std::chrono::duration<double, std::milli>(ph[2] - ph[1]).count(),
                 std::chrono::duration<double, std::milli>(ph[3] - ph[2]).count(),
                 std::chrono::duration<double, std::milli>(ph[4] - ph[3]).count(),
                 std::chrono::duration<double, std::milli>(ph[5] - ph[4]).count(),
                 std::chrono::duration<double, std::milli>(ph[6] - ph[5]).count(),
                 std::chrono::duration<double, std::milli>(ph[7] - ph[6]).count());
  const bool need_labels = any_invalid != 0;  // then the saddles were not filtered
  out.vm_first_pos = R.rank_lo[k + 1];
  if (need_labels) {
    // the host descends unresolved arms; it needs the saddle labels, their
    // supports and the minima labels
    out.minima_labels.resize((size_t)M * k);
    if (M) copy_wait(out.minima_labels.data(), labels.p, (size_t)M * k * 4, hipMemcpyDeviceToHost, s);
    auto &slab = W.slab, &ssup = W.ssup;
    slab.ensure((size_t)S * kMaxLabel);
    ssup.ensure(4 * (size_t)S);
    hipLaunchKernelGGL(k_saddle_labels, dim3(blocks_for(S, 256)), dim3(256), 0, s, B.events.p, B.order.p,
                       saddle_pos, (int64_t)S, slab.p, ssup.p);
    out.saddle_labels.resize((size_t)S * kMaxLabel);
    out.sup.resize(4 * (size_t)S);
    MHGP_HIP(hipMemcpyAsync(out.saddle_labels.data(), slab.p, (size_t)S * kMaxLabel * 4, hipMemcpyDeviceToHost, s));
    copy_wait(out.sup.data(), ssup.p, 4 * (size_t)S * 4, hipMemcpyDeviceToHost, s);
  }
}

}  // namespace mhgp
