// Canonical cloud and Morton LBVH on gfx950.
//
// Canonical PointIds (reference morsehgp3d/src/cpu/spatial/point_cloud.cpp:40-95):
// lexicographic order of the three binary64 total-order keys, -0 -> +0,
// duplicates rejected.  Morton codes (reference lbvh.cpp:78-90, 237-298):
// 21 bits per axis, q = floor(2^21 (x - l) / (u - l)) exactly, certified here
// with error-free FP64 transforms.  Tree: the reference's top-down
// highest-differing-bit split with midpoint splits inside runs of equal codes
// (lbvh.cpp:831-906), built in one pass with Karras' radix-tree construction
// over the augmented key (code, midpoint path bits).  Boxes carry PointId
// witnesses with the reference's tie rule (lbvh.cpp:46-76).
#include <algorithm>
#include <cmath>

#include "context.hpp"
#include "exact_device.hpp"

namespace mhgp {

namespace {

// Cloud bounds, per workgroup (lower x, y, z, upper x, y, z).
constexpr int kBoundBlocks = 64;
constexpr int kBoundBlock = 256;
__global__ void __launch_bounds__(kBoundBlock) k_bounds(const double *__restrict__ src, int64_t n, double *part) {
  __shared__ double red[kBoundBlock / 64][6];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double v[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
  for (int64_t i = (int64_t)blockIdx.x * kBoundBlock + threadIdx.x; i < n; i += (int64_t)kBoundBlocks * kBoundBlock)
    for (int a = 0; a < 3; ++a) {
      const double x = src[3 * i + a] + 0.0;  // -0 -> +0
      v[a] = fmin(v[a], x);
      v[3 + a] = fmax(v[3 + a], x);
    }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
    for (int a = 0; a < 3; ++a) {
      v[a] = fmin(v[a], __shfl_xor(v[a], o));
      v[3 + a] = fmax(v[3 + a], __shfl_xor(v[3 + a], o));
    }
  if (lane == 0)
    for (int a = 0; a < 6; ++a) red[wave][a] = v[a];
  __syncthreads();
  if (threadIdx.x < 6) {
    double x = red[0][threadIdx.x];
    for (int w = 1; w < kBoundBlock / 64; ++w)
      x = threadIdx.x < 3 ? fmin(x, red[w][threadIdx.x]) : fmax(x, red[w][threadIdx.x]);
    part[6 * blockIdx.x + threadIdx.x] = x;
  }
}

__global__ void __launch_bounds__(64) k_bounds_all(const double *__restrict__ part, double *bounds) {
  static_assert(kBoundBlocks == 64, "one partial per lane");
  double v[6];
  for (int a = 0; a < 6; ++a) v[a] = part[6 * threadIdx.x + a];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
    for (int a = 0; a < 3; ++a) {
      v[a] = fmin(v[a], __shfl_xor(v[a], o));
      v[3 + a] = fmax(v[3 + a], __shfl_xor(v[3 + a], o));
    }
  if (threadIdx.x == 0)
    for (int a = 0; a < 6; ++a) bounds[a] = v[a];
}

// Canonical order by one sort: a coarse key of 22 + 21 + 21 bits (the
// coordinates' places between the bounds, monotone in each coordinate), and
// then the exact lexicographic order within runs of equal x bits.  Points of
// different x bits are in order; inside a run the key has ordered equal x by
// y and z already, so only adjacent inversions, which differing x values cause,
// need the repair below.  Three sorts of the full coordinates (24 passes)
// remain for clouds with longer runs.
//
// Such a run sets status bit kLongRun, and the build's kernels behind the sort
// return at once: their results would be thrown away, and with 25 000 equal codes
// the leaf kernel's walk alone is 2.4 of a build's 3.2 ms.
constexpr int kCoarseShift = 42;
constexpr int kRunMost = 64;
constexpr uint32_t kRunMark = 0x80000000u;
constexpr uint32_t kLongRun = 4u;

__device__ inline uint64_t coarse(double x, double lo, double hi, double most) {
  const double e = hi - lo, s = e > 0.0 && e < INFINITY ? most / e : 0.0;
  return (uint64_t)fmin(fmax((x - lo) * s, 0.0), most);
}

__global__ void k_coarse_keys(const double *__restrict__ src, int64_t n, const double *__restrict__ b, uint64_t *key,
                              uint32_t *perm) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  key[i] = coarse(src[3 * i] + 0.0, b[0], b[3], 4194303.0) << kCoarseShift |
           coarse(src[3 * i + 1] + 0.0, b[1], b[4], 2097151.0) << 21 |
           coarse(src[3 * i + 2] + 0.0, b[2], b[5], 2097151.0);
  perm[i] = (uint32_t)i;
}

// Exact lexicographic order of two source points, equal points by index.
__device__ inline bool source_less(const double *src, uint32_t a, uint32_t b) {
  for (int k = 0; k < 3; ++k) {
    const uint64_t x = order_key(dbits(src[3 * (size_t)a + k])), y = order_key(dbits(src[3 * (size_t)b + k]));
    if (x != y) return x < y;
  }
  return a < b;
}

// Marks the start of every run that holds an adjacent inversion; a run beyond
// kRunMost points sets kLongRun.  LESS(a, b): the exact order of values.
template <class LESS>
__device__ inline void mark_run(const uint64_t *key, int shift, uint32_t *val, int64_t n, int64_t i, uint32_t *status,
                                LESS &&less) {
  if (i <= 0 || i >= n) return;
  const uint64_t r = key[i] >> shift;
  if (key[i - 1] >> shift != r) return;
  volatile uint32_t *v = val;  // marks come and go in the top bit
  if (!less(v[i] & ~kRunMark, v[i - 1] & ~kRunMark)) return;
  int64_t s = i - 1;
  while (s > 0 && i - s < kRunMost && key[s - 1] >> shift == r) --s;
  int64_t e = i + 1;
  while (e < n && e - s <= kRunMost && key[e] >> shift == r) ++e;
  if (e - s > kRunMost || (s > 0 && key[s - 1] >> shift == r)) {
    atomicOr(status, kLongRun);
    return;
  }
  atomicOr(&val[s], kRunMark);
}

__global__ void k_mark_runs(const double *__restrict__ src, const uint64_t *__restrict__ key, uint32_t *perm, int64_t n,
                            uint32_t *status) {
  mark_run(key, kCoarseShift, perm, n, (int64_t)blockIdx.x * blockDim.x + threadIdx.x, status,
           [&](uint32_t a, uint32_t b) { return source_less(src, a, b); });
}

__global__ void k_sort_runs(const double *__restrict__ src, const uint64_t *__restrict__ key, uint32_t *perm,
                            int64_t n) {
  const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n || !(perm[s] & kRunMark)) return;
  perm[s] &= ~kRunMark;
  const uint64_t r = key[s] >> kCoarseShift;
  for (int64_t i = s + 1; i < n && i < s + kRunMost && key[i] >> kCoarseShift == r; ++i) {
    const uint32_t v = perm[i];
    int64_t j = i;
    for (; j > s && source_less(src, v, perm[j - 1]); --j) perm[j] = perm[j - 1];
    perm[j] = v;
  }
}

__global__ void k_order_keys(const double *__restrict__ src, int64_t n, uint64_t *k0,
                             uint64_t *k1, uint64_t *k2, uint32_t *perm) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  k0[i] = order_key(dbits(src[3 * i]));
  k1[i] = order_key(dbits(src[3 * i + 1]));
  k2[i] = order_key(dbits(src[3 * i + 2]));
  perm[i] = (uint32_t)i;
}

__global__ void k_gather_key(const uint64_t *__restrict__ from, const uint32_t *__restrict__ perm,
                             int64_t n, uint64_t *to) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) to[i] = from[perm[i]];
}

// perm lists source indices in canonical order.
__global__ void k_canonical(const double *__restrict__ src, const uint32_t *__restrict__ perm,
                            int64_t n, double *X, double *Y, double *Z, uint32_t *source_index,
                            uint32_t *status) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || (status[0] & kLongRun)) return;
  uint32_t s = perm[i];
  double x = src[3 * s] + 0.0, y = src[3 * s + 1] + 0.0, z = src[3 * s + 2] + 0.0;  // -0 -> +0
  X[i] = x;
  Y[i] = y;
  Z[i] = z;
  source_index[i] = s;
  if (i > 0) {
    uint32_t t = perm[i - 1];
    if (dbits(src[3 * t] + 0.0) == dbits(x) && dbits(src[3 * t + 1] + 0.0) == dbits(y) &&
        dbits(src[3 * t + 2] + 0.0) == dbits(z))
      atomicOr(&status[0], 1u);
  }
  double v[3] = {x, y, z};
  for (int a = 0; a < 3; ++a)
    if (!isfinite(v[a])) atomicOr(&status[0], 2u);
}

// floor(2^21 (x - l) / (u - l)), certified exactly.
__device__ uint32_t quantize(double x, double l, double u, uint32_t *fallbacks) {
  const uint32_t qmax = (1u << 21) - 1;
  if (u == l) return 0;
  if (x == u) return qmax;
  double eh, el, dh, dl;
  two_diff(u, l, eh, el);
  two_diff(x, l, dh, dl);
  double t = (dh / eh) * 2097152.0;
  int64_t q = (int64_t)floor(t);
  if (q < 0) q = 0;
  if (q > (int64_t)qmax) q = qmax;
  // accept q when q*E <= 2^21 D < (q+1)*E holds exactly
  for (int iter = 0; iter < 4; ++iter) {
    double terms[6];
    double qd = (double)q;
    double p, pe, r, re;
    two_prod(qd, eh, p, pe);
    two_prod(qd, el, r, re);
    terms[0] = dh * 2097152.0; terms[1] = dl * 2097152.0;
    terms[2] = -p; terms[3] = -pe; terms[4] = -r; terms[5] = -re;
    int lo_sign = exact_sum_sign(terms, 6);  // 2^21 D - q E
    double qd1 = (double)(q + 1);
    two_prod(qd1, eh, p, pe);
    two_prod(qd1, el, r, re);
    terms[2] = -p; terms[3] = -pe; terms[4] = -r; terms[5] = -re;
    int hi_sign = exact_sum_sign(terms, 6);  // 2^21 D - (q+1) E
    if (lo_sign >= 0 && hi_sign < 0) {
      if (iter) atomicAdd(fallbacks, 1u);
      return (uint32_t)q;
    }
    if (lo_sign < 0) q--; else q++;
    if (q < 0) q = 0;
    if (q > (int64_t)qmax) return qmax;
  }
  atomicAdd(fallbacks + 1, 1u);  // unresolved: reported to the host as a failure
  return (uint32_t)q;
}

__device__ inline uint64_t spread21(uint32_t v) {
  uint64_t x = v & 0x1fffff;
  x = (x | (x << 32)) & 0x1f00000000ffffull;
  x = (x | (x << 16)) & 0x1f0000ff0000ffull;
  x = (x | (x << 8)) & 0x100f00f00f00f00full;
  x = (x | (x << 4)) & 0x10c30c30c30c30c3ull;
  x = (x | (x << 2)) & 0x1249249249249249ull;
  return x;
}

__global__ void k_morton(const double *__restrict__ X, const double *__restrict__ Y,
                         const double *__restrict__ Z, int64_t n, const double *__restrict__ b,
                         uint64_t *codes, uint32_t *ids, uint32_t *status) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || (status[0] & kLongRun)) return;
  uint32_t qx = quantize(X[i], b[0], b[3], status + 1);
  uint32_t qy = quantize(Y[i], b[1], b[4], status + 1);
  uint32_t qz = quantize(Z[i], b[2], b[5], status + 1);
  codes[i] = (spread21(qx) << 2) | (spread21(qy) << 1) | spread21(qz);
  ids[i] = (uint32_t)i;
}

__global__ void k_leaves(const uint32_t *__restrict__ ids, const double *__restrict__ X,
                         const double *__restrict__ Y, const double *__restrict__ Z,
                         const uint64_t *__restrict__ codes, int64_t n, double *LX, double *LY,
                         double *LZ, uint32_t *leaf_pos, uint64_t *path, const uint32_t *__restrict__ status) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n || (status[0] & kLongRun)) return;
  uint32_t id = ids[p];
  LX[p] = X[id];
  LY[p] = Y[id];
  LZ[p] = Z[id];
  leaf_pos[id] = (uint32_t)p;
  // midpoint path bits inside a run of equal codes (reference find_split)
  uint64_t c = codes[p];
  uint64_t bits = 0;
  bool inrun = (p > 0 && codes[p - 1] == c) || (p + 1 < n && codes[p + 1] == c);
  if (inrun) {
    int64_t a = p, e = p + 1;
    while (a > 0 && codes[a - 1] == c) a--;
    while (e < n && codes[e] == c) e++;
    int depth = 0;
    while (e - a > 1) {
      int64_t mid = a + (e - a) / 2;
      if (p >= mid) { bits |= 1ull << (63 - depth); a = mid; } else { e = mid; }
      depth++;
    }
  }
  path[p] = bits;
}

__device__ inline int delta(const uint64_t *codes, const uint64_t *path, int64_t n, int64_t i,
                            int64_t j) {
  if (j < 0 || j >= n) return -1;
  uint64_t a = codes[i], b = codes[j];
  if (a != b) return __clzll(a ^ b);
  return 64 + __clzll(path[i] ^ path[j]);
}

__global__ void k_karras(const uint64_t *__restrict__ codes, const uint64_t *__restrict__ path,
                         int64_t n, Node *nodes, uint32_t *parent_int, uint32_t *parent_leaf,
                         const uint32_t *__restrict__ status) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n - 1 || (status[0] & kLongRun)) return;
  const int d = (delta(codes, path, n, i, i + 1) - delta(codes, path, n, i, i - 1)) >= 0 ? 1 : -1;
  const int dmin = delta(codes, path, n, i, i - d);
  int64_t lmax = 2;
  while (delta(codes, path, n, i, i + lmax * d) > dmin) lmax *= 2;
  int64_t l = 0;
  for (int64_t t = lmax / 2; t >= 1; t /= 2)
    if (delta(codes, path, n, i, i + (l + t) * d) > dmin) l += t;
  const int64_t j = i + l * d;
  const int dnode = delta(codes, path, n, i, j);
  int64_t s = 0;
  int64_t t = l;
  do {
    t = (t + 1) / 2;
    if (delta(codes, path, n, i, i + (s + t) * d) > dnode) s += t;
  } while (t > 1);
  const int64_t gamma = i + s * d + (d < 0 ? -1 : 0);
  const int64_t lo = i < j ? i : j, hi = i < j ? j : i;
  Node nd;
  nd.begin = (uint32_t)lo;
  nd.end = (uint32_t)(hi + 1);
  if (lo == gamma) { nd.left = kLeafBit | (uint32_t)gamma; parent_leaf[gamma] = (uint32_t)i; }
  else { nd.left = (uint32_t)gamma; parent_int[gamma] = (uint32_t)i; }
  if (hi == gamma + 1) { nd.right = kLeafBit | (uint32_t)(gamma + 1); parent_leaf[gamma + 1] = (uint32_t)i; }
  else { nd.right = (uint32_t)(gamma + 1); parent_int[gamma + 1] = (uint32_t)i; }
  for (int a = 0; a < 3; ++a) { nd.lo[a] = 0; nd.hi[a] = 0; }
  nodes[i] = nd;
  if (i == 0) parent_int[0] = kInvalid;
}

// Box of a set of leaves with its witnesses: per side the extremum and the
// least PointId attaining it (reference tie rule, lbvh.cpp:46-76).  Any split
// of the set gives the same box.
struct Box {
  double v[6];  // lower x, y, z, upper x, y, z
  uint32_t w[6];
  __device__ void clear() {
    for (int a = 0; a < 3; ++a) {
      v[a] = INFINITY;
      v[3 + a] = -INFINITY;
      w[a] = w[3 + a] = kInvalid;
    }
  }
  __device__ void add(int a, double x, uint32_t id) {
    const bool take = (a < 3 ? x < v[a] : x > v[a]) || (x == v[a] && id < w[a]);
    v[a] = take ? x : v[a];
    w[a] = take ? id : w[a];
  }
  __device__ void add_leaf(const double *LX, const double *LY, const double *LZ, const uint32_t *leaf_id, int64_t p) {
    const double x[3] = {LX[p], LY[p], LZ[p]};
    const uint32_t id = leaf_id[p];
    for (int a = 0; a < 3; ++a) {
      add(a, x[a], id);
      add(3 + a, x[a], id);
    }
  }
  __device__ void add_box(const Box &b) {
    for (int a = 0; a < 6; ++a) add(a, b.v[a], b.w[a]);
  }
  // over the wave, in every lane
  __device__ void reduce() {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
#pragma unroll
      for (int a = 0; a < 6; ++a) {
        const double x = __shfl_xor(v[a], o);
        const uint32_t id = __shfl_xor(w[a], o);
        add(a, x, id);
      }
  }
};

// Boxes of the wave tree's level-0 and level-1 groups, one workgroup per
// level-1 group.
constexpr int kGroupBlock = 1024;
__global__ void __launch_bounds__(kGroupBlock) k_group_boxes(int64_t n, const double *__restrict__ LX,
                                                             const double *__restrict__ LY,
                                                             const double *__restrict__ LZ,
                                                             const uint32_t *__restrict__ leaf_id, Box *l0, Box *l1,
                                                             const uint32_t *__restrict__ status) {
  __shared__ Box box[64];
  if (status[0] & kLongRun) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t c0 = (n + 63) / 64;
  for (int j = wave; j < 64; j += kGroupBlock / 64) {
    const int64_t g = (int64_t)blockIdx.x * 64 + j;
    Box b;
    b.clear();
    if (g < c0) {
      if (g * 64 + lane < n) b.add_leaf(LX, LY, LZ, leaf_id, g * 64 + lane);
      b.reduce();
    }
    if (lane == 0) {
      box[j] = b;
      if (g < c0) l0[g] = b;
    }
  }
  __syncthreads();
  if (wave == 0) {
    Box b = box[lane];
    b.reduce();
    if (lane == 0) l1[blockIdx.x] = b;
  }
}

// Boxes and witnesses of the internal nodes from their leaf ranges: short
// ranges leaf by leaf, one node per lane; longer ones by the whole wave from
// the leaves and groups that make up the range.  No node waits for another
// (a bottom-up pass with fences between siblings took 97 us at 256 points and
// 1.44 ms at 200 000).  Bound by the latency of the lane loops.
constexpr uint32_t kShortRange = 32;
__global__ void __launch_bounds__(256) k_refit(int64_t n, Node *nodes, uint32_t *wit, const double *__restrict__ LX,
                                               const double *__restrict__ LY, const double *__restrict__ LZ,
                                               const uint32_t *__restrict__ leaf_id, const Box *__restrict__ l0,
                                               const Box *__restrict__ l1, const uint32_t *__restrict__ status) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t lane = threadIdx.x & 63u;
  if (status[0] & kLongRun) return;
  const bool valid = i < n - 1;
  const uint32_t b = valid ? nodes[i].begin : 0u, e = valid ? nodes[i].end : 0u;
  auto store = [&](int64_t node, const Box &x) {
    for (int a = 0; a < 3; ++a) {
      nodes[node].lo[a] = x.v[a];
      nodes[node].hi[a] = x.v[3 + a];
    }
    for (int a = 0; a < 6; ++a) wit[6 * node + a] = x.w[a];
  };
  const bool is_short = e - b <= kShortRange;
  if (valid && is_short) {
    Box x;
    x.clear();
    for (uint32_t p = b; p < e; ++p) x.add_leaf(LX, LY, LZ, leaf_id, p);
    store(i, x);
  }
  for (uint64_t m = __ballot(valid && !is_short); m;) {
    const int k = __builtin_amdgcn_readfirstlane(__ffsll((long long)m) - 1);
    m &= m - 1;
    const uint32_t rb = __builtin_amdgcn_readlane(b, k), re = __builtin_amdgcn_readlane(e, k);
    Box x;
    x.clear();
    // whole level-0 groups [g0, g1), of these whole level-1 groups [h0, h1)
    const uint32_t g0 = (rb + 63) / 64, g1 = re / 64;
    if (g0 >= g1) {
      for (uint32_t p = rb + lane; p < re; p += 64) x.add_leaf(LX, LY, LZ, leaf_id, p);
    } else {
      if (rb + lane < g0 * 64) x.add_leaf(LX, LY, LZ, leaf_id, rb + lane);
      if (g1 * 64 + lane < re) x.add_leaf(LX, LY, LZ, leaf_id, g1 * 64 + lane);
      const uint32_t h0 = (g0 + 63) / 64, h1 = g1 / 64;
      if (h0 >= h1) {
        for (uint32_t g = g0 + lane; g < g1; g += 64) x.add_box(l0[g]);
      } else {
        if (g0 + lane < h0 * 64) x.add_box(l0[g0 + lane]);
        if (h1 * 64 + lane < g1) x.add_box(l0[h1 * 64 + lane]);
        for (uint32_t h = h0 + lane; h < h1; h += 64) x.add_box(l1[h]);
      }
    }
    x.reduce();
    if (lane == 0) store(i - lane + k, x);
  }
}

// Canonical points in the input unit (an exact power of two), interleaved.
__global__ void k_points_out(int64_t n, const double *__restrict__ X, const double *__restrict__ Y,
                             const double *__restrict__ Z, int exponent, double *out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  out[3 * i] = ldexp(X[i], exponent);
  out[3 * i + 1] = ldexp(Y[i], exponent);
  out[3 * i + 2] = ldexp(Z[i], exponent);
}

// Snapshot leaves (code, PointId) and, of the runs of equal codes, their
// number (totals[0]) and the longest (totals[1]).  Codes ascend: a run's end
// is found by doubling steps and halving.
__global__ void k_leaves_out(int64_t n, const uint64_t *__restrict__ codes, const uint32_t *__restrict__ leaf_id,
                             ulonglong2 *leaves, unsigned long long *totals) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const uint64_t c = codes[p];
  leaves[p] = make_ulonglong2(c, leaf_id[p]);
  if (p + 1 >= n || codes[p + 1] != c || (p > 0 && codes[p - 1] == c)) return;
  int64_t last = p + 1, step = 2;  // the last known position of the run
  while (last + step < n && codes[last + step] == c) {
    last += step;
    step *= 2;
  }
  for (; step > 0; step /= 2)
    if (last + step < n && codes[last + step] == c) last += step;
  atomicAdd(&totals[0], 1ull);
  atomicMax(&totals[1], (unsigned long long)(last - p + 1));
}

// Postorder index of every node (internal i < n-1, leaf n-1+p), and the
// largest depth (in the words totals[2 ..]).
constexpr int kDepthSlots = 64;
__global__ void k_postorder(int64_t n, const Node *__restrict__ nodes,
                            const uint32_t *__restrict__ parent_int,
                            const uint32_t *__restrict__ parent_leaf, uint64_t *post,
                            unsigned long long *totals) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  uint32_t dep = 0;
  if (t < 2 * n - 1) {
    const bool leaf = t >= n - 1;
    uint32_t cur = leaf ? (uint32_t)(t - (n - 1)) | kLeafBit : (uint32_t)t;
    uint32_t par = n == 1 ? kInvalid : leaf ? parent_leaf[t - (n - 1)] : parent_int[t];
    uint64_t w = 0;
    while (par != kInvalid) {
      const Node &P = nodes[par];
      if (P.right == cur) {
        w += 1;
      } else {
        uint32_t r = P.right;
        uint64_t leaves_r = (r & kLeafBit) ? 1 : (uint64_t)(nodes[r].end - nodes[r].begin);
        w += 2 * leaves_r;
      }
      dep++;
      cur = par;
      par = parent_int[par];
    }
    post[t] = (uint64_t)(2 * n - 2) - w;
  }
  // the block's largest, into one of kDepthSlots words: 6 250 waves with an
  // atomic each on one word took 60 of the kernel's 90 us (200 000 points), now 31
  __shared__ uint32_t most;
  if (threadIdx.x == 0) most = 0;
  __syncthreads();
  uint32_t x = dep;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) x = max(x, (uint32_t)__shfl_xor((int)x, d));
  if (threadIdx.x % 64 == 0) atomicMax(&most, x);
  __syncthreads();
  if (threadIdx.x == 0) atomicMax(&totals[2 + blockIdx.x % kDepthSlots], (unsigned long long)most);
}

__global__ void k_snapshot(int64_t n, const Node *__restrict__ nodes, const uint32_t *__restrict__ wit,
                           const uint32_t *__restrict__ leaf_id, const uint64_t *__restrict__ post,
                           uint64_t *out) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 2 * n - 1) return;
  if (post[t] >= (uint64_t)(2 * n - 1)) return;  // malformed tree: the host sees a zero record
  uint64_t *o = out + 10 * post[t];
  if (t >= n - 1) {
    uint64_t p = t - (n - 1);
    uint64_t id = leaf_id[p];
    for (int a = 0; a < 6; ++a) o[a] = id;
    o[6] = ~0ull; o[7] = ~0ull; o[8] = p; o[9] = p + 1;
    return;
  }
  const Node &nd = nodes[t];
  for (int a = 0; a < 6; ++a) o[a] = wit[6 * t + a];
  uint32_t l = nd.left, r = nd.right;
  o[6] = post[(l & kLeafBit) ? (n - 1) + (l & ~kLeafBit) : l];
  o[7] = post[(r & kLeafBit) ? (n - 1) + (r & ~kLeafBit) : r];
  o[8] = nd.begin;
  o[9] = nd.end;
}

// FP32 copy of the LBVH for ball queries: each internal node lists its
// grandchildren (a leaf child stands for itself) with boxes rounded outward
// (a leaf's box is its point).
__device__ inline void wide_entry(const Node *nodes, const double *LX, const double *LY, const double *LZ,
                                  uint32_t x, WideNode &w, int slot) {
  double lo[3], hi[3];
  if (x & kLeafBit) {
    const uint32_t lp = x & ~kLeafBit;
    lo[0] = hi[0] = LX[lp];
    lo[1] = hi[1] = LY[lp];
    lo[2] = hi[2] = LZ[lp];
  } else {
    for (int a = 0; a < 3; ++a) { lo[a] = nodes[x].lo[a]; hi[a] = nodes[x].hi[a]; }
  }
  for (int a = 0; a < 3; ++a) {
    w.lo[slot][a] = __double2float_rd(lo[a]);
    w.hi[slot][a] = __double2float_ru(hi[a]);
  }
  w.child[slot] = x;
}

__global__ void k_wide_nodes(int64_t m, const Node *__restrict__ nodes, const double *__restrict__ LX,
                             const double *__restrict__ LY, const double *__restrict__ LZ, WideNode *out) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m) return;
  const Node &N = nodes[i];
  WideNode w;
  int slot = 0;
  for (int c = 0; c < 2; ++c) {
    const uint32_t x = c ? N.right : N.left;
    if (x & kLeafBit) {
      wide_entry(nodes, LX, LY, LZ, x, w, slot++);
    } else {
      wide_entry(nodes, LX, LY, LZ, nodes[x].left, w, slot++);
      wide_entry(nodes, LX, LY, LZ, nodes[x].right, w, slot++);
    }
  }
  for (; slot < 4; ++slot) {  // empty slot: a box no query meets
    for (int a = 0; a < 3; ++a) { w.lo[slot][a] = INFINITY; w.hi[slot][a] = -INFINITY; }
    w.child[slot] = kInvalid;
  }
  out[i] = w;
}

// Wave-tree boxes (wave_tree.hpp) of levels 0 and 1 from the boxes with
// witnesses, in the unit 2^e.
__global__ void k_wave_boxes(int64_t count, const Box *__restrict__ in, int e, GroupBox *out) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= count) return;
  GroupBox b;
  for (int a = 0; a < 3; ++a) {
    b.lo[a] = ldexp(in[g].v[a], e);
    b.hi[a] = ldexp(in[g].v[3 + a], e);
  }
  out[g] = b;
}

// Level-2 boxes, one wave per group (clouds of more than 262 144 points).
__global__ void __launch_bounds__(64) k_group_top(uint32_t c1, const GroupBox *__restrict__ l1, GroupBox *l2) {
  const uint32_t i = blockIdx.x * 64 + threadIdx.x;
  double v[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
  if (i < c1)
    for (int a = 0; a < 3; ++a) {
      v[a] = l1[i].lo[a];
      v[3 + a] = l1[i].hi[a];
    }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      v[a] = fmin(v[a], __shfl_xor(v[a], o));
      v[3 + a] = fmax(v[3 + a], __shfl_xor(v[3 + a], o));
    }
  if (threadIdx.x == 0) l2[blockIdx.x] = GroupBox{{v[0], v[1], v[2]}, {v[3], v[4], v[5]}};
}

// Power-of-two change of unit (context.hpp, scale_exp): possible only when
// every scaled coordinate stays a normal (or zero) finite binary64.
__global__ void k_scale_check(const double *__restrict__ X, const double *__restrict__ Y,
                              const double *__restrict__ Z, int64_t n, int e, uint32_t *bad) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double v[3] = {X[i], Y[i], Z[i]};
  bool ok = true;
  for (int a = 0; a < 3; ++a) {
    const double t = fabs(ldexp(v[a], e));
    ok = ok && (v[a] == 0.0 || (t >= 0x1p-1022 && t < INFINITY));
  }
  if (!ok) atomicOr(bad, 1u);
}

__global__ void k_scale_values(double *v, int64_t n, int e) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) v[i] = ldexp(v[i], e);
}

__global__ void k_scale_nodes(Node *nodes, int64_t m, int e) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m) return;
  for (int a = 0; a < 3; ++a) {
    nodes[i].lo[a] = ldexp(nodes[i].lo[a], e);
    nodes[i].hi[a] = ldexp(nodes[i].hi[a], e);
  }
}

// Unit exponent for a cloud of extent E: none inside [2^-16, 2^16], else the
// one that brings E into [1, 2).
int scale_exponent_for(double extent) {
  if (!(extent > 0.0) || !(extent < INFINITY)) return 0;
  if (extent >= 0x1p-16 && extent <= 0x1p16) return 0;
  return -std::ilogb(extent);
}

void apply_unit_scale(Context &c, const double bounds[6]) {
  const int64_t n = c.n;
  hipStream_t s = c.stream;
  c.scale_exp = 0;
  double extent = 0.0;
  for (int a = 0; a < 3; ++a) extent = std::max(extent, bounds[3 + a] - bounds[a]);
  const int e = scale_exponent_for(extent);
  if (e == 0) return;
  MHGP_HIP(hipMemsetAsync(c.status.p + 4, 0, sizeof(uint32_t), s));
  hipLaunchKernelGGL(k_scale_check, dim3(blocks_for(n, 256)), dim3(256), 0, s, c.X.p, c.Y.p, c.Z.p, n, e,
                     c.status.p + 4);
  uint32_t bad = 0;
  copy_wait(&bad, c.status.p + 4, 4, hipMemcpyDeviceToHost, s);
  if (bad) return;  // keep the input unit: exactness first
  for (double *v : {c.X.p, c.Y.p, c.Z.p, c.LX.p, c.LY.p, c.LZ.p})
    hipLaunchKernelGGL(k_scale_values, dim3(blocks_for(n, 256)), dim3(256), 0, s, v, n, e);
  hipLaunchKernelGGL(k_scale_values, dim3(1), dim3(64), 0, s, c.bounds.p, (int64_t)6, e);
  if (n > 1)
    hipLaunchKernelGGL(k_scale_nodes, dim3(blocks_for(n - 1, 256)), dim3(256), 0, s, c.nodes.p, n - 1, e);
  MHGP_LAUNCH_CHECK();
  c.scale_exp = e;
}

}  // namespace

// Canonical order and LBVH; full_sort: by three sorts of the whole
// coordinates, whatever the runs.  Returns false when that is needed.
static bool build(Context &c, bool full_sort) {
  const int64_t n = c.n;
  hipStream_t s = c.stream;
  const int T = 256;
  const dim3 G(blocks_for(n, T)), B256(T);
  MHGP_HIP(hipMemsetAsync(c.status.p, 0, 16 * sizeof(uint32_t), s));
  hipLaunchKernelGGL(k_bounds, dim3(kBoundBlocks), dim3(kBoundBlock), 0, s, c.src.p, n, c.bounds.p + 6);
  hipLaunchKernelGGL(k_bounds_all, dim3(1), dim3(64), 0, s, c.bounds.p + 6, c.bounds.p);
  if (full_sort) {
    c.key1.ensure(n);
    c.key2.ensure(n);
    hipLaunchKernelGGL(k_order_keys, G, B256, 0, s, c.src.p, n, c.key0.p, c.key1.p, c.key2.p, c.perm.p);
    // stable LSD over (k0, k1, k2): least significant key first
    c.sorter.sort(c.key2.p, c.perm.p, n, 0, 64, s);
    hipLaunchKernelGGL(k_gather_key, G, B256, 0, s, c.key1.p, c.perm.p, n, c.key2.p);
    c.sorter.sort(c.key2.p, c.perm.p, n, 0, 64, s);
    hipLaunchKernelGGL(k_gather_key, G, B256, 0, s, c.key0.p, c.perm.p, n, c.key2.p);
    c.sorter.sort(c.key2.p, c.perm.p, n, 0, 64, s);
  } else {
    hipLaunchKernelGGL(k_coarse_keys, G, B256, 0, s, c.src.p, n, c.bounds.p, c.key0.p, c.perm.p);
    c.sorter.sort(c.key0.p, c.perm.p, n, 0, 64, s);
    hipLaunchKernelGGL(k_mark_runs, G, B256, 0, s, c.src.p, c.key0.p, c.perm.p, n, c.status.p);
    hipLaunchKernelGGL(k_sort_runs, G, B256, 0, s, c.src.p, c.key0.p, c.perm.p, n);
  }
  hipLaunchKernelGGL(k_canonical, G, B256, 0, s, c.src.p, c.perm.p, n, c.X.p, c.Y.p, c.Z.p, c.source_index.p,
                     c.status.p);
  hipLaunchKernelGGL(k_morton, G, B256, 0, s, c.X.p, c.Y.p, c.Z.p, n, c.bounds.p, c.codes.p, c.leaf_id.p,
                     c.status.p);
  c.sorter.sort(c.codes.p, c.leaf_id.p, n, 0, 63, s);
  hipLaunchKernelGGL(k_leaves, G, B256, 0, s, c.leaf_id.p, c.X.p, c.Y.p, c.Z.p, c.codes.p, n, c.LX.p, c.LY.p, c.LZ.p,
                     c.leaf_pos.p, c.path.p, c.status.p);
  const int64_t c0 = (n + 63) / 64, c1 = (c0 + 63) / 64;
  c.group_exact.ensure((c0 + c1) * sizeof(Box));
  Box *gb = reinterpret_cast<Box *>(c.group_exact.p);
  hipLaunchKernelGGL(k_group_boxes, dim3(c1), dim3(kGroupBlock), 0, s, n, c.LX.p, c.LY.p, c.LZ.p, c.leaf_id.p, gb,
                     gb + c0, c.status.p);
  if (n > 1) {
    hipLaunchKernelGGL(k_karras, dim3(blocks_for(n - 1, T)), B256, 0, s, c.codes.p, c.path.p, n, c.nodes.p,
                       c.parent_int.p, c.parent_leaf.p, c.status.p);
    hipLaunchKernelGGL(k_refit, dim3(blocks_for(n - 1, T)), B256, 0, s, n, c.nodes.p, c.wit.p, c.LX.p, c.LY.p,
                       c.LZ.p, c.leaf_id.p, gb, gb + c0, c.status.p);
  } else {
    MHGP_HIP(hipMemsetAsync(c.parent_leaf.p, 0xff, sizeof(uint32_t), s));
  }
  MHGP_LAUNCH_CHECK();
  uint32_t st[4];
  copy_wait(st, c.status.p, sizeof(st), hipMemcpyDeviceToHost, s);
  if (st[0] & kLongRun) return false;
  if (st[0] & 2u) throw std::invalid_argument("a point coordinate is not finite");
  if (st[0] & 1u) throw std::invalid_argument("the cloud contains duplicate geometric points");
  if (st[2]) throw std::runtime_error("an exact Morton bin could not be certified");
  return true;
}

void canonicalize_and_build(Context &c) {
  const int64_t n = c.n, ni = n > 1 ? n - 1 : 1;
  c.scale_exp = 0;
  hipStream_t s = c.stream;
  c.X.ensure(n); c.Y.ensure(n); c.Z.ensure(n);
  c.source_index.ensure(n);
  c.key0.ensure(n);
  c.perm.ensure(n);
  c.status.ensure(16);
  c.bounds.ensure(6 * (1 + kBoundBlocks));
  c.codes.ensure(n);
  c.leaf_id.ensure(n);
  c.leaf_pos.ensure(n);
  c.LX.ensure(n); c.LY.ensure(n); c.LZ.ensure(n);
  c.path.ensure(n);
  c.nodes.ensure(ni);
  c.parent_int.ensure(ni);
  c.parent_leaf.ensure(n);
  c.wit.ensure(6 * ni);
  if (!build(c, false) && !build(c, true)) throw std::runtime_error("the canonical order did not settle");
  double bounds[6];
  copy_wait(bounds, c.bounds.p, sizeof(bounds), hipMemcpyDeviceToHost, s);
  apply_unit_scale(c, bounds);
  const int64_t internal = std::max<int64_t>(n - 1, 0);
  c.wide.ensure(internal);
  if (internal)
    hipLaunchKernelGGL(k_wide_nodes, dim3(blocks_for(internal, 256)), dim3(256), 0, s, internal, c.nodes.p, c.LX.p,
                       c.LY.p, c.LZ.p, c.wide.p);
  const int64_t c0 = (n + 63) / 64, c1 = (c0 + 63) / 64, c2 = (c1 + 63) / 64;
  c.groups.ensure(c0 + c1 + c2);
  hipLaunchKernelGGL(k_wave_boxes, dim3(blocks_for(c0 + c1, 256)), dim3(256), 0, s, c0 + c1,
                     reinterpret_cast<const Box *>(c.group_exact.p), c.scale_exp, c.groups.p);
  if (c2 > 1)
    hipLaunchKernelGGL(k_group_top, dim3(c2), dim3(64), 0, s, (uint32_t)c1, c.groups.p + c0, c.groups.p + c0 + c1);
  MHGP_LAUNCH_CHECK();
  c.lbvh_ready = true;
}

WaveTree wave_tree(const Context &c) {
  const uint32_t n = (uint32_t)c.n, c0 = (n + 63) / 64, c1 = (c0 + 63) / 64, c2 = (c1 + 63) / 64;
  return {c.groups.p, c.groups.p + c0, c.groups.p + c0 + c1, c0, c1, c2, n,
          c.LX.p, c.LY.p, c.LZ.p, c.leaf_id.p};
}

void canonical_points(Context &c, double *xyz_out, uint32_t *source_index_out) {
  const int64_t n = c.n;
  hipStream_t s = c.stream;
  if (source_index_out)
    MHGP_HIP(hipMemcpyAsync(source_index_out, c.source_index.p, n * 4, hipMemcpyDeviceToHost, s));
  if (xyz_out && n) {
    // the uploaded points' buffer is free once the index stands
    c.src.ensure(3 * n);
    hipLaunchKernelGGL(k_points_out, dim3(blocks_for(n, 256)), dim3(256), 0, s, n, c.X.p, c.Y.p, c.Z.p, -c.scale_exp, c.src.p);
    MHGP_LAUNCH_CHECK();
    MHGP_HIP(hipMemcpyAsync(xyz_out, c.src.p, n * 24, hipMemcpyDeviceToHost, s));
  }
  MHGP_HIP(hipStreamSynchronize(s));
}

void export_snapshot(Context &c, uint64_t *leaves, uint64_t *nodes_out, uint64_t *counters) {
  const int64_t n = c.n, m = 2 * n - 1;
  hipStream_t s = c.stream;
  const int T = 256;
  // leaves, nodes, postorder, totals; kept by the context unless its device
  // memory is bounded
  DevBuf<uint64_t> own;
  DevBuf<uint64_t> &buf = c.capacity_bytes > 0 ? own : c.snapshot;
  buf.ensure(2 * n + 10 * m + m + 2 + kDepthSlots);
  uint64_t *d_leaves = buf.p, *d_nodes = d_leaves + 2 * n, *post = d_nodes + 10 * m, *totals = post + m;
  MHGP_HIP(hipMemsetAsync(totals, 0, (2 + kDepthSlots) * 8, s));
  hipLaunchKernelGGL(k_postorder, dim3(blocks_for(m, T)), dim3(T), 0, s, n, c.nodes.p, c.parent_int.p,
                     c.parent_leaf.p, post, (unsigned long long *)totals);
  hipLaunchKernelGGL(k_snapshot, dim3(blocks_for(m, T)), dim3(T), 0, s, n, c.nodes.p, c.wit.p, c.leaf_id.p, post,
                     d_nodes);
  hipLaunchKernelGGL(k_leaves_out, dim3(blocks_for(n, T)), dim3(T), 0, s, n, c.codes.p, c.leaf_id.p,
                     reinterpret_cast<ulonglong2 *>(d_leaves), (unsigned long long *)totals);
  MHGP_LAUNCH_CHECK();
  uint64_t got[2 + kDepthSlots];
  MHGP_HIP(hipMemcpyAsync(leaves, d_leaves, n * 16, hipMemcpyDeviceToHost, s));
  MHGP_HIP(hipMemcpyAsync(nodes_out, d_nodes, 10 * m * 8, hipMemcpyDeviceToHost, s));
  copy_wait(got, totals, sizeof got, hipMemcpyDeviceToHost, s);
  counters[0] = n;
  counters[1] = m;
  counters[2] = *std::max_element(got + 2, got + 2 + kDepthSlots);
  counters[3] = got[0];
  counters[4] = got[1];
}

}  // namespace mhgp
