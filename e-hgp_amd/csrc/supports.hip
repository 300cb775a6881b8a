// Critical-sphere catalogue (supports of 2..4 points, closed rank <= s_max).
//
// Observable definition (reference reference/morsehgp3d_oracle/catalog.py and
// morsehgp3d/src/cpu/hierarchy/critical_catalog.cpp): a support U of 1..4
// affinely independent points whose circumcentre c (in aff U) lies strictly
// inside conv U; interior I = points strictly inside the sphere, shell = points
// on it; an event when shell == U and |I| + |U| <= s_max, an extra-shell
// diagnostic when shell != U and |I| + |U| <= s_max.
//
// Enumeration (this backend's own method, replacing the reference's node-tuple
// branch-and-bound of pair_support_stream.cpp / higher_support_stream.cpp):
// every support is enumerated once, from its least PointId u (the anchor).
//  1. Direction-cell certificate.  For a critical sphere through u with centre
//     u + r d, every open ball of radius rho tangent at u towards d lies in
//     the open sphere when rho <= r.  The unit sphere of directions is cut
//     into 384 cube-map cells; for each cell C the radius rho_C is the
//     (s_max-1)-th smallest radius at which a gathered point lies strictly
//     inside every tangent ball of the cell.  A sphere with direction in C and
//     r >= rho_C therefore holds >= s_max-1 interior points and is not
//     critical.  Since the centre of a well-centred support lies in the
//     cloud's AABB, r is also below the AABB exit distance of the cell.
//  2. Region.  All points of a critical sphere with direction in C lie in
//     the union of closed tangent balls of radius rho'_C over C; a point's
//     mask records the cells whose union contains it.  Pairs, triangles and
//     tetrahedra through u are searched among region members only, and their
//     interior is counted over the whole region.
//  3. Tetrahedra come from faces (u, v, w) (the three least ids) by the
//     pencil of spheres through the face's circumcircle: the apex z must be
//     among the first s_max-3 points swept on its side, so only those are
//     tested.
// Every emitted record is certified with the FP64 predicates of
// predicates.hpp over the anchor's region; anything undecided goes to the
// host fallback queue with the anchor's region.
#include <algorithm>
#include <cmath>
#include <cfloat>
#include <cstdio>
#include <cstring>
#include <memory>
#include <numeric>

#include "wave.hpp"
#include "pipeline.hpp"
#include "predicates.hpp"
#include "supports.hpp"
#include "timing.hpp"
#include "wave_tree.hpp"

namespace mhgp {

int64_t catalog_device_bytes(const CatalogBuffers &b) {
  return b.radius.bytes() + b.gcount.bytes() + b.goff.bytes() + b.glist.bytes() + b.region.bytes() +
         b.lists.bytes() + b.big.bytes() + b.rescans.bytes() + b.events.bytes() + b.fallbacks.bytes() + b.fb_region.bytes() +
         b.counters.bytes() + b.cells.bytes() + b.cellf.bytes() + b.strips.bytes() + b.scratch.bytes() + b.anchors.bytes() +
         b.total.bytes() + b.run_count.bytes() + b.run_pos.bytes() + b.run_gidx.bytes() + b.run_new.bytes() +
         b.run_link.bytes() + b.run_rec.bytes();
}

namespace {

constexpr int kBlock = 256;
constexpr int kRegionCapHuge = 1023;  // the largest region enumerated in LDS

// LDS written by some lanes of a wave, then read by other lanes of it
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Lists the probes append to (B.lists, kLists rows of n entries; their lengths
// are counters[kListCount ..]).  The first four hold PointIds for a later
// pass: gathers to widen, gathers beyond the small probe, those beyond the next
// one, gathers (and regions) beyond LDS.
// The others hold the probed anchors of one launch (their index in it, which
// is also their slab's) by the size of their region.
enum { L_WIDEN = 0, L_WIDE = 1, L_WIDER = 2, L_BIG = 3, L_TINY = 4, L_LITTLE = 5, L_SMALL = 6, L_MID = 7, L_LARGE = 8, L_SLAB = 9,
       kLists = 10 };
constexpr int kListCount = 8;    // counters: list lengths
constexpr int kOpenCount = 18;   // counters: open anchors, their largest region
constexpr int kOpenLargest = 19;
constexpr int kRescanMost = 20;  // longest rescan list of a launch
constexpr int kCounters = 24;

// Regions of the global-memory path are enumerated face by face in
// O(region^3) work; beyond the context's region limit (at most this) one
// anchor would keep a workgroup busy for many seconds.  Such an anchor is not
// enumerated: the catalogue is returned complete for every other anchor with
// status conditional (a budget stop), and the anchor and its region size are
// reported.
constexpr uint32_t kBigRegionMax = kRegionLimitMax;

struct Params {
  const double *X, *Y, *Z;       // canonical coordinates
  const uint32_t *gcount;
  const uint64_t *goff;
  const uint32_t *glist;
  double *radius;
  const double *cells;           // 8 doubles per cell
  const float *cellf;            // 8 floats per cell: the FP32 cell (see cell_f)
  const uint64_t *strips;        // kStrips x 8: cells a great circle can meet (k_strips)
  double blo[3], bhi[3];         // cloud AABB
  int s_max;
  uint32_t *region;              // region size of a probed anchor
  uint32_t *lists;               // kLists rows of list_cap entries
  uint32_t list_cap;
  EventRec *events;
  uint64_t event_cap;
  FallbackRec *fallbacks;
  uint64_t fallback_cap;
  uint32_t *fb_region;
  uint64_t fb_region_cap;
  struct Rescan *rescans;        // sides of faces left to k_rescan
  uint64_t rescan_cap;
  unsigned long long *counters;  // [0] events [1] fallbacks [2] region words [3] candidates [4] rescans
                                 // [5] FP64 [6] FP32 operations, then the lists' lengths and the open anchors
  const uint32_t *anchors;
  uint32_t anchor_count;
  int probe;                     // 1: stop once the region is in the slab
  uint32_t one_wave, two_waves;  // regions up to these sizes take workgroups of one and of two waves
  int ascending;                 // 1: the slabs' regions are in increasing distance
  double *scratch;
  uint64_t slab_doubles;
  uint32_t gcap;                 // gathered points a slab holds
  int count_flops;               // 1: count the FP64 (counters[5]) and FP32 (counters[6]) operations
  uint32_t region_limit;         // largest region the global-memory path enumerates
};

__device__ inline void list_add(const Params &P, int list, uint32_t v) {
  const unsigned long long at = atomicAdd(&P.counters[kListCount + list], 1ull);
  if (at < P.list_cap) P.lists[(size_t)list * P.list_cap + at] = v;
}

// The certificate needs a larger gather than radius Rg (one lane).
__device__ inline void widen(const Params &P, uint32_t u, double need, double Rg) {
  P.radius[u] = fmax(need * 1.02, Rg * 1.05);
  list_add(P, L_WIDEN, u);
}

// Anchor u's region of M points is in slab a (one lane): queued for the
// enumeration of its size, or left open beyond the region limit.
__device__ inline void probed(const Params &P, uint32_t u, uint32_t a, uint32_t M);

struct Work {
  double *gx, *gy, *gz;
  uint32_t *gid;
  float *rho;        // certificate radius per cell (FP32, rounded up)
  uint32_t *ridx;    // gathered index of each region slot (until the points are compacted)
  uint64_t *rmask;  // 6 words per member
  uint16_t *kidx;    // candidate vertices (region slots)
  float4 *fc;       // FP32 offset and distance per gathered point (certificate and masks)
  uint32_t *cand;   // candidate supports classified (LDS, flushed once per anchor)
  unsigned long long *flops;  // FP64 operations of the certified predicates (LDS, flushed once per anchor; null: not counted)
  float4 *f;                  // FP32 copies of the region's coordinates and distances from the anchor
  unsigned long long *flops32;  // FP32 operations of the tests (as flops; null: not counted)
  bool ascending;             // the region is in increasing distance: scans end at a sphere's diameter
  uint32_t slab;              // the anchor's index in its launch
  const float4 *cell;         // LDS: direction and cosine of the 64 cells of a cube face, in its frame
};

// FP64 operations (add, subtract, multiply; a fused multiply-add counts two)
// of one evaluation of each certified predicate, counted from predicates.hpp:
// the value, its magnitude bound and the certification test.
constexpr uint32_t kFlopPairSide = 18;   // PairSphere::side
constexpr uint32_t kFlopTetSide = 21;    // TetSphere::side
constexpr uint32_t kFlopFacePoint = 33;  // TriSphere::power + height, two certified signs
constexpr uint32_t kFlopSweepKey = 24;   // sweep_key
constexpr uint32_t kFlopTriInit = 66;    // TriSphere::init
constexpr uint32_t kFlopTetInit = 150;   // TetSphere::init

// Counting is off unless the launch asks for it (flops == nullptr): the
// timed path pays for one uniform branch per call.
__device__ inline void add_flops(const Work &w, uint64_t v) {
  if (w.flops && v) atomicAdd(w.flops, (unsigned long long)v);
}
// FP32 operations of the FP32 tests, counted the same way (the certificate
// and mask tests of a cell, the pencil tests, the face, pair and tetrahedron
// polynomials with their bounds, a key interval); reciprocals and square
// roots count one each.
constexpr uint32_t kF32Cover = 16;      // one point against one cell (certificate)
constexpr uint32_t kF32Mask = 16;       // one point against one cell (membership)
constexpr uint32_t kF32Pencil = 15;     // Pencil::outside, per slot
constexpr uint32_t kF32Cell = 28;       // one shared cell of a face (face_interval)
constexpr uint32_t kF32FacePoint = 24;  // TriSphereF::eval and two certified signs
constexpr uint32_t kF32Key = 16;        // key_bounds_32
constexpr uint32_t kF32PairSide = 13;   // SphereF::place of a pair
constexpr uint32_t kF32TetSide = 13;    // SphereF::place of a tetrahedron
__device__ inline void add_flops32(const Work &w, uint64_t v) {
  if (w.flops32 && v) atomicAdd(w.flops32, (unsigned long long)v);
}

__device__ inline V3 gpt(const Work &w, uint32_t i) { return {w.gx[i], w.gy[i], w.gz[i]}; }

// Interior id lists are sorted with static indices only, so they stay in
// registers: an odd-even transposition network (unused slots hold kInvalid and
// sort last).
__device__ inline void sort_static(uint32_t (&a)[kMaxInterior], int n) {
#pragma unroll
  for (int j = 0; j < kMaxInterior; ++j) a[j] = j < n ? a[j] : kInvalid;
#pragma unroll
  for (int pass = 0; pass < kMaxInterior; ++pass) {
#pragma unroll
    for (int j = pass & 1; j + 1 < kMaxInterior; j += 2) {
      const uint32_t x = a[j], y = a[j + 1];
      a[j] = min(x, y);
      a[j + 1] = max(x, y);
    }
  }
}

__device__ __attribute__((always_inline)) inline void emit_event(const Params &P, uint32_t u, const uint32_t *sup, int m, int nint,
                           const uint32_t *interior, double level, double lerr) {
  const unsigned long long slot = wave_append(true, &P.counters[0]);
  if (slot >= P.event_cap) return;
  EventRec &e = P.events[slot];
  e.ids[0] = u;
  for (int i = 1; i < 4; ++i) e.ids[i] = i < m ? sup[i - 1] : kInvalid;
  e.meta = (uint32_t)m | ((uint32_t)(nint + m) << 8) | ((uint32_t)nint << 16);
#pragma unroll
  for (int i = 0; i < kMaxInterior; ++i) e.interior[i] = i < nint ? interior[i] : kInvalid;
  e.level = level;
  // rounded up into float (an infinite bound only sends the record to the
  // exact host ordering)
  e.level_err = (float)lerr * (1.0f + 1e-6f);
}

// Queues undecided work and, once per anchor, its region for the host.
__device__ __attribute__((always_inline)) inline void emit_fallback(const Params &P, const Work &w, uint32_t u, uint32_t kind,
                              const uint32_t *ids, int m, uint32_t M, uint32_t *region_slot) {
  if (*region_slot == kInvalid) {
    uint32_t expected = kInvalid;
    // first fallback of this anchor publishes its region
    unsigned long long off = atomicAdd(&P.counters[2], (unsigned long long)M);
    if (off + M <= P.fb_region_cap) {
      for (uint32_t s = 0; s < M; ++s) P.fb_region[off + s] = w.gid[s];
      atomicCAS(region_slot, expected, (uint32_t)off);
    }
  }
  unsigned long long slot = atomicAdd(&P.counters[1], 1ull);
  if (slot >= P.fallback_cap) return;
  FallbackRec &f = P.fallbacks[slot];
  f.kind = kind;
  f.ids[0] = u;
  for (int i = 1; i < 4; ++i) f.ids[i] = i < m ? ids[i - 1] : kInvalid;
  f.region_off = *region_slot;
  f.region_len = M;
  f.pad = 0;
}

// FP32 certification of a sign: v against its magnitude bound a.  With
// the coordinates, the coefficients and the at most ~9 roundings of a chain
// in FP32 (the FP64 coefficients rounded to nearest), |v32 - v| < 1e-6 a
// for the polynomials below; a sign is certified when |v32| > 1e-5 a and
// a > 1e-30 (FP32 underflow then adds at most ~1e-37, far below the
// threshold).  0 leaves the point to the FP64 test.
__device__ inline int cert32(float v, float a) {
  const float e = 1e-5f * a;
  return !(a > 1e-30f) ? 0 : (v > e ? 1 : (v < -e ? -1 : 0));
}

// A candidate sphere through the anchor in FP32: the scaled power
// v = a |p|^2 - p.b of a point, and 1e-5 of its magnitude bound
// |p| (aA |p| + bA) (the norms bound the sums of magnitudes) plus 1e-35; a
// larger |v| certifies the sign (cert32).  reach: no point farther from the
// anchor is inside (the sphere passes through the anchor, so its diameter with
// a margin for the FP32 estimate; infinite when the region is not in
// increasing distance).
struct SphereF {
  float a, aE, b[3], bE, reach;
  __device__ void test(const float4 &p, float &v, float &e) const {
    const float pp = p.w * p.w;
    v = a * pp - (p.x * b[0] + p.y * b[1] + p.z * b[2]);
    e = aE * pp + (bE * p.w + 1e-35f);
  }
};
__device__ inline float norm_up(double x, double y, double z) {
  return (float)sqrt(x * x + y * y + z * z) * (1.0f + 1e-6f);
}
__device__ inline SphereF to_f32(const PairSphere &s, bool ascending) {
  const float l = norm_up(s.a.x, s.a.y, s.a.z);
  return {1.0f, 1e-5f, {(float)s.a.x, (float)s.a.y, (float)s.a.z}, 1e-5f * l, ascending ? l * (1.0f + 1e-4f) + 1e-30f : INFINITY};
}
__device__ inline SphereF to_f32(const TetSphere &t, bool ascending) {
  // diameter |N| / |V|; both hold 12 digits at worst below their magnitude
  // bounds (their signs are certified), hence the wide margin
  const double sg = t.V > 0 ? 1.0 : -1.0;
  const double d = sqrt(dot(t.N, t.N)) * __builtin_amdgcn_rcp(fabs(t.V));
  return {(float)(sg * t.V), (float)(1e-5 * t.VA), {(float)(sg * t.N.x), (float)(sg * t.N.y), (float)(sg * t.N.z)},
          1e-5f * norm_up(t.NA.x, t.NA.y, t.NA.z), ascending ? (float)d * 1.05f + 1e-30f : INFINITY};
}

// Bits of a test over n <= 32 slots, slot 0 first, shifted in from below (one
// add with carry each) and turned round.
__device__ inline uint32_t shift_in(uint32_t bits, bool b) { return bits + bits + (b ? 1u : 0u); }
__device__ inline uint32_t in_order(uint32_t bits, uint32_t n) { return __builtin_bitreverse32(bits) >> (32u - n); }

// Up to kMaxInterior region slots, 16 bits each, 2 per word; the newest lowest.
constexpr int kPacked = (kMaxInterior + 1) / 2;
__device__ inline void push_packed(uint32_t (&pk)[kPacked], uint32_t slot) {
#pragma unroll
  for (int k = kPacked - 1; k > 0; --k) pk[k] = __builtin_amdgcn_alignbit(pk[k], pk[k - 1], 16);
  pk[0] = pk[0] << 16 | slot;
}
__device__ inline void unpack_ids(const Work &w, const uint32_t (&pk)[kPacked], int n, uint32_t (&ids)[kMaxInterior]) {
#pragma unroll
  for (int j = 0; j < kMaxInterior; ++j) ids[j] = j < n ? w.gid[(pk[j / 2] >> ((j % 2) * 16)) & 0xFFFFu] : kInvalid;
}

// Certified classification of the region against a candidate sphere through
// the anchor and m - 1 region points (slots skip).  FP32 for 32 slots at a time
// into two bit masks (inside, undecided), FP64 for the undecided; the inside
// slots are packed.  Returns 1 event, 0 not critical, -1 undecided (host).
// Bound by VALU issue; collecting the ids point by point over the whole region
// took 24 of the enumeration's 73 ms for the 50 000-point lattice, this about 5.
template <class S>
__device__ __attribute__((always_inline)) inline int classify(const Params &P, const Work &w, uint32_t M, const S &sph,
                        const uint32_t *skip, int m, uint32_t (&interior)[kPacked], int &nint) {
  nint = 0;
#pragma unroll
  for (int k = 0; k < kPacked; ++k) interior[k] = 0;
  const int cap = P.s_max - m;
  int undecided = 0;
  constexpr uint32_t per = sizeof(S) == sizeof(PairSphere) ? kFlopPairSide : kFlopTetSide;
  constexpr uint32_t per32 = sizeof(S) == sizeof(PairSphere) ? kF32PairSide : kF32TetSide;
  uint32_t evals = 0, evals32 = 0;
  const SphereF f = to_f32(sph, w.ascending);
  bool over = false;
#pragma unroll 1
  for (uint32_t s0 = 0; s0 < M; s0 += 32) {
    if (w.f[s0].w > f.reach) break;
    const uint32_t cn = min(32u, M - s0);
    uint32_t in = 0, open = 0;
#pragma unroll 4
    for (uint32_t j = 0; j < cn; ++j) {
      float v, e;
      f.test(w.f[s0 + j], v, e);
      in = shift_in(in, v < -e);
      open = shift_in(open, !(fabsf(v) > e));
    }
    in = in_order(in, cn);
    open = in_order(open, cn);
    evals32 += cn;
    for (int k = 0; k < m - 1; ++k)
      if (skip[k] - s0 < cn) {
        in &= ~(1u << (skip[k] - s0));
        open &= ~(1u << (skip[k] - s0));
      }
    while (open) {
      const uint32_t j = (uint32_t)(__ffs((int)open) - 1);
      open &= open - 1;
      const int side = sph.side(gpt(w, s0 + j));
      evals++;
      in |= (uint32_t)(side < 0) << j;
      undecided += side == 0;
    }
    if (nint + __popc(in) > cap) {
      over = true;
      break;
    }
    while (in) {
      push_packed(interior, s0 + (uint32_t)(__ffs((int)in) - 1));
      in &= in - 1;
      nint++;
    }
  }
  add_flops(w, (uint64_t)evals * per);
  add_flops32(w, (uint64_t)evals32 * per32);
  return over ? 0 : undecided ? -1 : 1;
}


__device__ __attribute__((always_inline)) inline void process_pair(const Params &P, const Work &w, uint32_t u, uint32_t M, uint32_t vi,
                             uint32_t *region_slot) {
  PairSphere sph;
  sph.init(gpt(w, vi));
  uint32_t packed[kPacked];
  int nint;
  uint32_t skip[1] = {vi};
  int r = classify(P, w, M, sph, skip, 2, packed, nint);
  uint32_t vid = w.gid[vi];
  if (r == 0) return;
  atomicAdd(w.cand, 1u);
  if (r < 0) {
    emit_fallback(P, w, u, 2, &vid, 2, M, region_slot);
    return;
  }
  uint32_t interior[kMaxInterior];
  unpack_ids(w, packed, nint, interior);
  sort_static(interior, nint);
  emit_event(P, u, &vid, 2, nint, interior, sph.level(), 8 * kCert);
}

__device__ __attribute__((always_inline)) inline void process_tet(const Params &P, const Work &w, uint32_t u, uint32_t M, uint32_t vi, uint32_t wi,
                            uint32_t zi, uint32_t *region_slot) {
  TetSphere t;
  int wc = t.init(gpt(w, vi), gpt(w, wi), gpt(w, zi));
  add_flops(w, kFlopTetInit);
  uint32_t ids[3] = {w.gid[vi], w.gid[wi], w.gid[zi]};
  if (wc < 0) return;
  atomicAdd(w.cand, 1u);
  if (wc == 0) { emit_fallback(P, w, u, 4, ids, 4, M, region_slot); return; }
  uint32_t packed[kPacked];
  int nint;
  uint32_t skip[3] = {vi, wi, zi};
  int r = classify(P, w, M, t, skip, 4, packed, nint);
  if (r == 0) return;
  if (r < 0) { emit_fallback(P, w, u, 4, ids, 4, M, region_slot); return; }
  uint32_t interior[kMaxInterior];
  unpack_ids(w, packed, nint, interior);
  sort_static(interior, nint);
  emit_event(P, u, ids, 4, nint, interior, t.level(), t.level_err());
}

// Smallest upper bounds of the sweep keys of the outside points ahead of one
// side.  Insertion runs over static indices, so the list stays in registers.
struct SweepList {
  static constexpr int kCap = 8;  // >= s_max - 3 for s_max <= 11
  double hi[kCap];                // upper key bounds, ascending
  __device__ void init() {
#pragma unroll
    for (int j = 0; j < kCap; ++j) hi[j] = INFINITY;
  }
  __device__ void insert(double t, double e) {
    double h = t + e;
#pragma unroll
    for (int j = 0; j < kCap; ++j) {
      const double lo = fmin(hi[j], h);
      h = fmax(hi[j], h);
      hi[j] = lo;
    }
  }
  __device__ void pop() {
#pragma unroll
    for (int j = 0; j + 1 < kCap; ++j) hi[j] = hi[j + 1];
    hi[kCap - 1] = INFINITY;
  }
};

// Largest lower key bounds of the inside points behind one side (a subset
// of them only weakens the apex pruning bound, never invalidates it).
struct BehindList {
  static constexpr int kCap = 4;
  double v[kCap];
  __device__ void init() {
#pragma unroll
    for (int j = 0; j < kCap; ++j) v[j] = -INFINITY;
  }
  __device__ void insert(double x) {
#pragma unroll
    for (int j = kCap - 1; j > 0; --j) v[j] = x > v[j - 1] ? v[j - 1] : (x > v[j] ? x : v[j]);
    v[0] = fmax(v[0], x);
  }
  __device__ int count_above(double x) const {
    int c = 0;
#pragma unroll
    for (int j = 0; j < kCap; ++j) c += v[j] > x;
    return c;
  }
};

// The same two lists in FP32, filled for both sides during a face's pass
// without a branch: a point of the other side goes in as the weakest value.  An
// entry of the sweep list is a double whose high word is the key's FP32 upper
// bound (at least 0, so the word's order is the bound's, and no double that
// begins with it is infinite or NaN) and whose low word is the region slot: one
// minimum and one maximum per entry keep bound and slot in order.  A point whose
// key lies past the end of the face's pencil cannot be an apex, so bounds end
// there.  An entry's lower bound is the entry less the face's widest interval.
// All bounds err outwards: a wider interval only admits more apex candidates,
// which are classified exactly, or sends a side to k_rescan.  Against one word
// an entry (22 to 24 bits of fixed point above the slot, a median of three
// each) this costs nothing that the runs show (50 000 points K 10: 43.7 and
// 43.9 ms; the 2 003-point mixture 27.5 and 27.6), and a face whose pencil has
// no end keeps its keys apart.
// Minimum and maximum are the bare instructions: on values that a loop carries
// the compiler has fmin and fmax quiet a signalling NaN first, which no entry is
// (the mixture 29.7 ms with them).
__device__ inline double min_entry(double a, double b) {
  double r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ inline double max_entry(double a, double b) {
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
struct SweepListF {
  static constexpr int kCap = 8;  // >= s_max - 3 for s_max <= 11
  static constexpr int kNone = 0x7f900000;  // past every bound (infinity is 0x7f800000)
  double hi[kCap];  // entries, ascending
  double evicted;   // smallest entry that left or missed the list
  __device__ static double none() { return __hiloint2double(kNone, 0); }
  __device__ static bool used(double e) { return __double2hiint(e) != kNone; }
  __device__ static float bound(double e) { return __int_as_float(__double2hiint(e)); }
  __device__ static uint32_t slot(double e) { return (uint32_t)__double2loint(e); }
  __device__ void init() {
#pragma unroll
    for (int j = 0; j < kCap; ++j) hi[j] = none();
    evicted = none();
  }
  __device__ void insert(double e) {
    evicted = min_entry(evicted, max_entry(hi[kCap - 1], e));
#pragma unroll
    for (int j = kCap - 1; j > 0; --j) hi[j] = max_entry(hi[j - 1], min_entry(hi[j], e));
    hi[0] = min_entry(hi[0], e);
  }
  // upper bound of the need-th entry, infinite when there are fewer
  __device__ float threshold(int need) const {
    double r = none();
#pragma unroll
    for (int j = 0; j < kCap; ++j) r = (j == need - 1) ? hi[j] : r;
    return used(r) ? bound(r) : INFINITY;
  }
};
struct BehindListF {
  static constexpr int kCap = 4;
  float v[kCap];
  __device__ void init() {
#pragma unroll
    for (int j = 0; j < kCap; ++j) v[j] = 0.0f;
  }
  __device__ void insert(float x) {
    // descending: the median of the entry above, x and the entry
#pragma unroll
    for (int j = kCap - 1; j > 0; --j) v[j] = __builtin_amdgcn_fmed3f(v[j - 1], x, v[j]);
    v[0] = fmaxf(v[0], x);
  }
  __device__ int count_above(float x) const {
    int c = 0;
#pragma unroll
    for (int j = 0; j < kCap; ++j) c += v[j] > x;
    return c;
  }
};

// Sweep key of a point against the face (tau = P / |H|) and its error bound.
// The reciprocal of |H| is the hardware estimate refined by two Newton
// steps; the residual e = 1 - |H| r of the result bounds its relative error
// (up to the rounding of e), which joins the key's error bound.  Outside the
// range where the estimate is reliable the key is unknown: tau = 0 with an
// infinite bound, which meets every threshold and sends the side to its full
// scan.
__device__ inline void sweep_key(double Pw, double PA, double H, double HA, double &tau, double &terr) {
  const double h = fabs(H);
  double r = __builtin_amdgcn_rcp(h);
  double e = __builtin_fma(-h, r, 1.0);
  r = __builtin_fma(r, e, r);
  e = __builtin_fma(-h, r, 1.0);
  r = __builtin_fma(r, e, r);
  const double rerr = 2.0 * fabs(__builtin_fma(-h, r, 1.0));
  tau = Pw * r;
  terr = (kCert * PA + kCertAbs + (kCert * HA + kCertAbs) * fabs(tau)) * r * (1.0 + 1e-12) + (1e-15 + rerr) * fabs(tau);
  if (!(h > 1e-290 && h < 1e290)) {
    tau = 0.0;
    terr = INFINITY;
  }
}

// FP32 bounds of the key interval [tau - terr, tau + terr], rounded outwards.
__device__ inline void key_bounds_f(double tau, double terr, float &hf, float &lf) {
  const double hd = tau + terr, ld = tau - terr;
  hf = (float)hd;
  if (!((double)hf >= hd)) hf = nextafterf(hf, INFINITY);
  lf = (float)ld;
  if (!((double)lf <= ld)) lf = nextafterf(lf, -INFINITY);
}

// A face's power and height polynomials in FP32 (the FP64 coefficients
// rounded to nearest).  With the coordinates, the coefficients and the at
// most 8 roundings of a chain in FP32, |P32 - P| < 1e-6 Pabs and
// |H32 - H| < 1e-6 Habs (about 5e-7 each); a sign is certified when it
// exceeds 1e-5 of its magnitude bound and the bound exceeds 1e-30 (FP32
// underflow then adds at most ~1e-37, far below the threshold).  Undecided
// points take the FP64 path.
struct TriSphereF {
  float D, DA, g[3], gA, n[3], nA;  // gA, nA: norms, which bound the sums of magnitudes
  __device__ void init(const TriSphere &f) {
    D = (float)f.D;
    DA = (float)f.DA;
    g[0] = (float)f.g.x; g[1] = (float)f.g.y; g[2] = (float)f.g.z;
    gA = norm_up(f.gA.x, f.gA.y, f.gA.z);
    n[0] = (float)f.n.x; n[1] = (float)f.n.y; n[2] = (float)f.n.z;
    nA = norm_up(f.nA.x, f.nA.y, f.nA.z);
  }
  __device__ void eval(const float4 &p, float &P, float &PA, float &H, float &HA) const {
    P = D * (p.w * p.w) - (p.x * g[0] + p.y * g[1] + p.z * g[2]);
    PA = p.w * (DA * p.w + gA);
    H = p.x * n[0] + p.y * n[1] + p.z * n[2];
    HA = p.w * nA;
  }
};
// Key interval of a point whose FP32 signs are certified: the true P lies
// within 1e-6 PA of P32 and |H| within 1e-6 HA of |H32| (< |H32| / 10), so
// tau = P / |H| lies between the quotients of the extreme values; the
// roundings of the sums, the reciprocals (1 ulp) and the products stay
// inside the final 1e-6 widening.  lf is a lower bound for P > 0 only.
__device__ inline void key_bounds_32(float Pv, float PA, float H, float HA, float &hf, float &lf) {
  const float ah = fabsf(H), eP = 1e-6f * PA, eH = 1e-6f * HA;
  const float rlo = __builtin_amdgcn_rcpf(ah + eH), rhi = __builtin_amdgcn_rcpf(ah - eH);
  lf = (Pv - eP) * rlo;
  hf = (Pv + eP) * (Pv > 0.0f ? rhi : rlo);
  lf = lf - 1e-6f * fabsf(lf) - 1e-37f;
  hf = hf + 1e-6f * fabsf(hf) + 1e-37f;
}

// The part of a face's pencil that can be critical: spheres through u, v, w
// with centres c3 + t n, t in an interval [tl, tu] (face_interval).  A point's
// power against such a sphere is linear in t, so a point outside both end
// spheres is outside all of them.  FP32 with the anchor at the origin:
// outside when p.p > 2 p.c for both end centres c, by a margin of
// 1e-3 p.p + a, which exceeds the rounding of the products (below
// 1e-6 |p| |c|) for every |p|: 2 sqrt(1e-3 a) >= 1e-6 |c| for a = 1e-8 |c|^2.
struct Pencil {
  float l[3], u[3];  // twice the end centres
  float a;           // infinite: every point is kept
  float reach;       // no point farther from the anchor is in any of the spheres (as SphereF::reach)
  double end;        // sweep key of the farther end, a little past it (0: unrestricted)
  __device__ bool outside(const float4 &p) const {
    const float dl = p.x * l[0] + p.y * l[1] + p.z * l[2], du = p.x * u[0] + p.y * u[1] + p.z * u[2];
    return p.w * p.w * 0.999f - a > fmaxf(dl, du);
  }
};

// Ends of the pencil for t in [lo, hi] x r3 (r3: the face's circumradius);
// lo = -infinity: not restricted.
__device__ inline Pencil face_pencil(const TriSphere &f, float lo, float hi, bool ascending) {
  Pencil c{};
  c.a = INFINITY;
  c.reach = INFINITY;
  c.end = 0.0;
  if (!(lo > -INFINITY)) return c;
  const double s = 1.0 / f.D;
  const V3 k = {f.g.x * s, f.g.y * s, f.g.z * s};  // twice the circumcentre
  const double q = sqrt(dot(k, k) * s);            // 2 r3 / |n|
  const double l = lo * q, h = hi * q;
  c.end = fmax(fabs(l), fabs(h)) * f.D * (1.0 + 1e-3);
  const double cl[3] = {k.x + l * f.n.x, k.y + l * f.n.y, k.z + l * f.n.z};
  const double cu[3] = {k.x + h * f.n.x, k.y + h * f.n.y, k.z + h * f.n.z};
  double ll = 0, uu = 0;
  for (int i = 0; i < 3; ++i) {
    c.l[i] = (float)cl[i];
    c.u[i] = (float)cu[i];
    ll += cl[i] * cl[i];
    uu += cu[i] * cu[i];
  }
  const double m2 = fmax(ll, uu);  // the larger sphere's squared diameter
  c.a = (float)(1e-8 * m2) + 1e-34f;
  if (ascending) c.reach = (float)sqrt(m2) * (1.0f + 1e-4f) + 1e-30f;
  return c;
}

// The face passes scan the region in chunks of 64 slots: first the pencil
// test of every slot of the chunk (a bit mask), then the point work for the
// set bits only, in ascending slot order, exactly the order of a plain scan.
// The lanes of a wave run the point work as often as the busiest lane of the
// chunk needs it, instead of once for every slot that any lane needs.
// tests32 counts the slots tested (the face's own vertices excluded).
__device__ inline uint64_t pencil_chunk(const Work &w, const Pencil &c, uint32_t s0, uint32_t M, uint32_t vi,
                                        uint32_t wi, uint32_t &tests32) {
  const uint32_t cn = min(64u, M - s0), c0 = min(cn, 32u);
  uint32_t lo = 0, hi = 0;
#pragma unroll 4
  for (uint32_t j = 0; j < c0; ++j) lo = shift_in(lo, !c.outside(w.f[s0 + j]));
#pragma unroll 4
  for (uint32_t j = c0; j < cn; ++j) hi = shift_in(hi, !c.outside(w.f[s0 + j]));
  uint64_t in = in_order(lo, c0);
  if (cn > 32) in |= (uint64_t)in_order(hi, cn - 32) << 32;
  if (vi - s0 < cn) in &= ~(1ull << (vi - s0));
  if (wi - s0 < cn) in &= ~(1ull << (wi - s0));
  tests32 += cn;
  return in;
}

// Per-wave work queue of the face phase (LDS).  The pass of every face runs
// one face per lane; the tetrahedra it leads to are queued and then taken one
// per lane, so the lanes of a wave run scans of equal length instead of
// waiting for the face with the most apexes.  A full queue falls back to doing the work in place.
constexpr uint32_t kTetQ = 256;
struct WaveQueues {
  uint32_t *tet;     // vi | wi << 10 | zi << 20 (region slots, < 1024)
  uint32_t *ntet;
};

// A side of a face whose apexes its face's list does not decide (near-equal
// keys past its end, a few thousand in 25 million records): the face by its
// PointIds with its pencil interval, and the inside points ahead of the side.
// Settled by k_rescan from the anchor's slab; in the enumeration kernel the
// FP64 passes of these sides cost 160 spilled registers.
struct Rescan {
  uint32_t anchor;  // slab of the launch
  uint32_t v, w;
  uint32_t side;    // side | cin << 1
  float lo, hi;
};
static_assert(sizeof(Rescan) == kRescanBytes, "rescan layout");

// Apexes of one side among the FP32 list its face's pass filled: bit j for
// entry j.  rescan: a point left or missed the list with a lower bound within
// the threshold, so the side takes its own passes instead.
__device__ inline uint32_t apex_mask(int cin_side, int K, const SweepListF &top, const BehindListF &beh,
                                     float widest, bool &rescan) {
  rescan = false;
  if (cin_side >= K) return 0;
  const float thr = (top.threshold(K - cin_side) + widest) * (1.0f + 1e-6f);  // past both roundings
  if (SweepListF::used(top.evicted) && SweepListF::bound(top.evicted) <= thr) {
    rescan = true;
    return 0;
  }
  uint32_t cand = 0;
#pragma unroll
  for (int j = 0; j < SweepListF::kCap; ++j) {
    // inside points behind: counted while their key exceeds z's
    const float h = SweepListF::bound(top.hi[j]);
    const bool ok = SweepListF::used(top.hi[j]) && h <= thr && cin_side + beh.count_above(h) < K;
    cand |= ok ? (1u << j) : 0u;
  }
  return cand;
}

// Face (u, v, w): its triangle event, then the apexes of each side.  One
// pass certifies every side and insideness, builds the triangle's interior,
// counts the inside points ahead of each side and fills both sides' sweep
// lists, from which the apexes follow (apex_mask): the outside points ahead of
// the side whose sweep key is among the s_max - 3 smallest (fewer when inside
// points are already ahead), each checked against the inside points behind.
// QUEUED (LDS paths): tetrahedra go to the wave's queue; otherwise in place.
// The pass runs on the region's FP32 copies (FP64 only for the points whose FP32
// signs are not certified) and sees the points that some sphere of the face's
// pencil within [lo, hi] (face_interval; n oriented as v x w) can hold.
template <bool QUEUED>
__device__ __attribute__((always_inline)) inline void process_face(const Params &P, const Work &w, uint32_t u, uint32_t M, uint32_t vi,
                             uint32_t wi, float lo, float hi, uint32_t *region_slot, WaveQueues *q) {
  // the sphere is built from its points in PointId order, so its FP64 level
  // (and every later tetrahedron's) does not depend on the enumeration order
  uint32_t ids[2] = {w.gid[vi], w.gid[wi]};
  if (ids[0] > ids[1]) { uint32_t t = ids[0]; ids[0] = ids[1]; ids[1] = t; uint32_t q = vi; vi = wi; wi = q; float l = lo; lo = -hi; hi = -l; }
  TriSphere f;
  const int wc = f.init(gpt(w, vi), gpt(w, wi));
  add_flops(w, kFlopTriInit);
  if (!f.nondegenerate()) {
    // collinear or undecided: a triangle cannot be a support; an undecided
    // face goes to the host together with its apexes
    if (cert_sign(f.D, f.DA) == 0) emit_fallback(P, w, u, 3, ids, 3, M, region_slot);
    return;
  }
  const uint32_t wid = ids[1];
  const int smax = P.s_max;
  const int K = smax - 3;  // an apex must be among the first K points swept
  const Pencil pen = face_pencil(f, lo, hi, w.ascending);
  // the triangle's own sphere (t = 0) is critical only within the interval;
  // a side that the interval does not reach has no apexes
  const bool tri = lo <= 0.0f && hi >= 0.0f;
  // the triangle's level, before the pass (the vertices need not stay live)
  const double tri_level = f.level(), tri_level_err = f.level_err();
  // inside the triangle's sphere, ahead of side 0 / 1
  int cin0 = hi < 0.0f ? K : 0, cin1 = lo > 0.0f ? K : 0;
  int total_in = 0;
  // region slots of the first inside points (a triangle event has at most
  // s_max - 3 <= 8)
  uint32_t tri_pk[kPacked] = {};
  uint32_t evals = 0;
  SweepListF top0, top1;  // outside points ahead of side 0 / 1
  BehindListF beh0, beh1;  // inside points behind side 0 / 1
  top0.init();
  top1.init();
  beh0.init();
  beh1.init();
  constexpr uint32_t kFlopPoint = kFlopFacePoint + kFlopSweepKey;
  uint32_t tests32 = 0, evals32 = 0;  // FP32 work
  const float end = pen.end > 1e-30 ? (float)(pen.end * (1.0 + 1e-6)) : INFINITY;  // no apex past it
  float widest = 0.0f;                                                             // widest key interval
  const int tri_limit = tri ? smax - 2 : 0;  // inside points that exclude the triangle
  TriSphereF f32;
  f32.init(f);
#pragma unroll 1
  for (uint32_t s0 = 0; s0 < M; s0 += 64) {
    if (w.f[s0].w > pen.reach) break;
    uint64_t in = pencil_chunk(w, pen, s0, M, vi, wi, tests32);
#pragma unroll 1
    while (in) {
      const uint32_t gi = s0 + (uint32_t)(__ffsll((long long)in) - 1);
      in &= in - 1;
      float hf, lf, P32, PA32, H32, HA32;
      f32.eval(w.f[gi], P32, PA32, H32, HA32);
      bool outer = P32 > 0.0f, above = H32 > 0.0f;
      evals32++;
      key_bounds_32(P32, PA32, H32, HA32, hf, lf);
      if (cert32(P32, PA32) == 0 || cert32(H32, HA32) == 0) {
        const V3 p = gpt(w, gi);
        evals++;
        double Pw, PA, H, HA;
        // rare: the FP64 sphere is rebuilt (same arithmetic, same values)
        // rather than kept live through the pass
        TriSphere f64;
        f64.init(gpt(w, vi), gpt(w, wi));
        f64.power(p, Pw, PA);
        f64.height(p, H, HA);
        const int sp = cert_sign(Pw, PA), sh = cert_sign(H, HA);
        // every sign the side passes use is certified here, before anything is emitted
        if (sp == 0 || sh == 0) {
          add_flops(w, (uint64_t)evals * kFlopPoint);
          add_flops32(w, (uint64_t)tests32 * kF32Pencil + (uint64_t)evals32 * (kF32FacePoint + kF32Key));
          emit_fallback(P, w, u, 3, ids, 3, M, region_slot);
          return;
        }
        double tau, terr;
        sweep_key(Pw, PA, H, HA, tau, terr);
        key_bounds_f(tau, terr, hf, lf);
        outer = sp > 0;
        above = sh > 0;
        if (!(lf <= hf)) hf = INFINITY, lf = 0.0f;  // overflow: unknown
        lf = fmaxf(lf, 0.0f);                        // used of outside points, whose keys are positive
        if (!outer) hf = fminf(hf, 0.0f);  // a key interval that reaches past 0: weakest
      }
      // outside: ahead of side 0 when above, of side 1 otherwise
      const bool ahead = outer && !(lf >= end);
      hf = fminf(hf, end);
      widest = fmaxf(widest, ahead ? hf - lf : 0.0f);
      const int key = __float_as_int(hf);
      top0.insert(__hiloint2double(ahead && above ? key : SweepListF::kNone, (int)gi));
      top1.insert(__hiloint2double(ahead && !above ? key : SweepListF::kNone, (int)gi));
      // inside: behind side 1 when above, behind side 0 otherwise; -hf is a
      // lower bound of -tau - terr
      const float x = outer ? 0.0f : -hf;
      beh0.insert(above ? 0.0f : x);
      beh1.insert(above ? x : 0.0f);
      if (outer) continue;
      push_packed(tri_pk, gi);
      total_in++;
      cin0 += above;
      cin1 += !above;
      // both sides saturated and the triangle out of rank: nothing left here
      if (cin0 >= K && cin1 >= K && total_in >= tri_limit) {
        add_flops(w, (uint64_t)evals * kFlopPoint);
        add_flops32(w, (uint64_t)tests32 * kF32Pencil + (uint64_t)evals32 * (kF32FacePoint + kF32Key));
        return;
      }
    }
  }
  add_flops(w, (uint64_t)evals * kFlopPoint);
  add_flops32(w, (uint64_t)tests32 * kF32Pencil + (uint64_t)evals32 * (kF32FacePoint + kF32Key));
  // triangle event
  if (!tri) {
    // not critical by the certificate
  } else if (wc > 0 && total_in + 3 <= smax) {
    atomicAdd(w.cand, 1u);
    uint32_t tri_int[kMaxInterior];
    unpack_ids(w, tri_pk, total_in, tri_int);
    sort_static(tri_int, total_in);
    emit_event(P, u, ids, 3, total_in, tri_int, tri_level, tri_level_err);
  } else if (wc == 0 && total_in + 3 <= smax) {
    emit_fallback(P, w, u, 3, ids, 3, M, region_slot);
    return;
  }
  if (K <= 0) return;
  bool rescan[2];
  uint32_t cand = apex_mask(cin0, K, top0, beh0, widest, rescan[0]);
  cand |= apex_mask(cin1, K, top1, beh1, widest, rescan[1]) << SweepListF::kCap;
  // queued on the LDS paths, in place on the global-memory path
  while (cand) {
    const int j = __ffs(cand) - 1;
    cand &= cand - 1;
    uint32_t zi = 0;  // selected by static index, the lists stay in registers
#pragma unroll
    for (int e = 0; e < SweepListF::kCap; ++e) {
      zi = e == j ? SweepListF::slot(top0.hi[e]) : zi;
      zi = e + SweepListF::kCap == j ? SweepListF::slot(top1.hi[e]) : zi;
    }
    if (w.gid[zi] <= wid) continue;
    if (QUEUED) {
      const uint32_t at = atomicAdd(q->ntet, 1u);
      if (at < kTetQ) {
        q->tet[at] = vi | (wi << 10) | (zi << 20);
        continue;
      }
    }
    process_tet(P, w, u, M, vi, wi, zi, region_slot);
  }
#pragma unroll
  for (int side = 0; side < 2; ++side) {
    if (!rescan[side]) continue;
    const unsigned long long at = atomicAdd(&P.counters[4], 1ull);
    if (at < P.rescan_cap) P.rescans[at] = Rescan{w.slab, ids[0], ids[1], (uint32_t)side | ((uint32_t)(side ? cin1 : cin0) << 1), lo, hi};
  }
}

// Cell direction and angular radius in FP32, rounded so that the cell only
// grows (cos delta down, sin delta up): every FP32 test below errs towards a
// larger certificate radius and a larger region (the table is rounded on
// the host, see make_cells_f).  Reciprocals and square
// roots use the hardware approximations (1 ulp); their error, like the
// rounding of the products, stays far inside the slack of the tests (1e-5 on
// the mask cosines, 1e-4 on the certificate radius; cancellation is bounded
// by skipping covers with cos(theta + delta) < 0.01).  Lengths below kTinyLen
// (where the approximations flush) take the conservative branch.
constexpr float kTinyLen = 1e-30f;
struct CellF {
  float dx, dy, dz, cosd, sind;
};
__device__ inline CellF cell_f(const float *cf) {
  const float4 a = *reinterpret_cast<const float4 *>(cf);
  return {a.x, a.y, a.z, a.w, cf[4]};
}

// Cells whose union of closed tangent balls (radius rho'_C) contains gathered
// point i: cos of the smallest angle between its direction and the cell.
// FP32 with relative and absolute slack; a point may only be included too
// often, which costs work but never a support.
// rmax2 bounds 2 rho'_C over every cell from above: a point beyond it is in
// no cell's balls; wlim[wd] bounds it over the 64 cells of mask word wd.
__device__ bool member_mask(const Params &P, const Work &w, uint32_t i, float rmax2, const float *wlim,
                            uint64_t mask[6]) {
  const float4 q = w.fc[i];
  for (int k = 0; k < 6; ++k) mask[k] = 0;
  if (!(q.w > kTinyLen)) {  // distance lost to underflow: member everywhere
    for (int k = 0; k < 6; ++k) mask[k] = ~0ull;
    return true;
  }
  if (q.w > rmax2) return false;
  const float inv = __builtin_amdgcn_rcpf(q.w);
  bool any = false;
  // one mask word per 64 cells, each built in a register; a word whose
  // largest radius the point exceeds stays empty
#pragma unroll
  for (int wd = 0; wd < kCells / 64; ++wd) {
    if (q.w > wlim[wd]) continue;
    add_flops32(w, 64ull * kF32Mask);
    uint64_t bits = 0;
#pragma unroll 1
    for (int b = 0; b < 64; ++b) {
      const int c = 64 * wd + b;
      const CellF cf = cell_f(P.cellf + 8 * c);
      const float ct = (q.x * cf.dx + q.y * cf.dy + q.z * cf.dz) * inv;
      float cm;  // cos(max(theta - delta, 0))
      if (ct >= cf.cosd) cm = 1.0f;
      else cm = ct * cf.cosd + __builtin_amdgcn_sqrtf(fmaxf(0.0f, 1.0f - ct * ct)) * cf.sind;
      const float rho = w.rho[c];
      if (q.w <= 2.0f * rho * (cm + 1e-5f) * (1.0f + 1e-5f)) bits |= 1ull << b;
    }
    mask[wd] = bits;
    any |= bits != 0;
  }
  return any;
}

constexpr int kCoverCap = 10;  // s_max - 1 <= 10

// Certificate radius of cell c from its (s_max-1)-th cover radius bk: with the
// FP32 slack, at most the AABB exit distance of the cell, rounded up to a
// float (a larger radius only enlarges the region).
__device__ inline float cell_radius(const Params &P, int c, float bk, double ux, double uy, double uz) {
  const double *cd = P.cells + 8 * c;
  const double chord = cd[5];
  const double rc = (double)bk * (1.0 + 1e-4);
  double dir[3] = {cd[0], cd[1], cd[2]};
  double uu[3] = {ux, uy, uz};
  double e = INFINITY;
  for (int a = 0; a < 3; ++a) {
    double lo = dir[a] - chord, hi = dir[a] + chord;
    if (lo > 0) e = fmin(e, (P.bhi[a] - uu[a]) / lo);
    else if (hi < 0) e = fmin(e, (P.blo[a] - uu[a]) / hi);
  }
  e = fmax(e, 0.0) * (1.0 + 1e-9) + 1e-300;
  const double rd = fmin(rc, e);
  float rf = (float)rd;
  if (!((double)rf >= rd)) rf = rd <= (double)FLT_MIN ? FLT_MIN : nextafterf(rf, INFINITY);
  return rf;
}

// Axis cell of a great circle with normal m (or -m): kStripSide^2 cells on each
// of three cube faces.  Of the 15 cells that a pair of the 50 000-point lattice
// shares, its lanes' longest walks (4 to 6 times that) bound face_interval;
// dropping those that the pencil's circle misses by one 64-byte row halves
// them: K 10 53.1 -> 46.3 ms, K 4 13.6 -> 12.8 ms (the walk itself on a table
// of one cube face in LDS: 2.5 and 0.7 ms before that).
constexpr int kStripSide = 16;
constexpr int kStrips = 3 * kStripSide * kStripSide;
__device__ inline uint32_t strip_of(float mx, float my, float mz) {
  const float ax = fabsf(mx), ay = fabsf(my), az = fabsf(mz);
  const bool fy = ay > ax && ay >= az, fz = az > ax && az > ay;
  const float m = fz ? mz : fy ? my : mx, a = fz ? mx : fy ? mz : my, b = fz ? my : fy ? mx : mz;
  const float r = __builtin_amdgcn_rcpf(m) * (0.5f * kStripSide);
  const int i = min(max((int)(a * r + 0.5f * kStripSide), 0), kStripSide - 1);
  const int j = min(max((int)(b * r + 0.5f * kStripSide), 0), kStripSide - 1);
  return (uint32_t)(((fz ? 2 : fy ? 1 : 0) * kStripSide + i) * kStripSide + j);
}

// For every axis cell of strip_of (a workgroup) the direction cells (its
// threads) that a great circle with its normal there can meet, six words of
// eight: |angle(g, m) - 90 degrees| at most the two cells' radii and 2e-3, which
// covers the lowered cosines of face_interval and the rounding of the axis.
__global__ void k_strips(const double *__restrict__ cells, uint64_t *__restrict__ strips) {
  const int f = blockIdx.x / (kStripSide * kStripSide), i = blockIdx.x / kStripSide % kStripSide, j = blockIdx.x % kStripSide;
  auto axis = [&](double s, double t) {
    const double a = 2.0 * s / kStripSide - 1.0, b = 2.0 * t / kStripSide - 1.0, q = 1.0 / sqrt(1.0 + a * a + b * b);
    return f == 0 ? V3{q, a * q, b * q} : f == 1 ? V3{b * q, q, a * q} : V3{a * q, b * q, q};
  };
  const V3 m = axis(i + 0.5, j + 0.5);
  double least = 1.0;
  for (int c = 0; c < 4; ++c) least = fmin(least, dot(m, axis(i + c / 2, j + c % 2)));
  const double radius = acos(least) + 2e-3;
  const double *g = cells + 8 * threadIdx.x;
  // |g.m| <= sin(delta + radius), the sum below 90 degrees
  const bool met = fabs(dot(m, V3{g[0], g[1], g[2]})) <= g[4] * cos(radius) + g[3] * sin(radius);
  const uint64_t word = __ballot(met);
  if (threadIdx.x % 64 == 0) strips[8 * blockIdx.x + threadIdx.x / 64] = word;
}

// Face (u, v, w) of region slots si, sj: the part of its pencil of spheres
// that the certificate leaves.  A critical sphere through the three points has
// its centre at c3 + t n (n the unit normal along v x w, t = s r3), its
// direction in a cell shared by v and w and its radius r3 sqrt(1 + s^2) within
// that cell's rho.  The directions of the pencil inside a cell of centre g and
// angular radius delta are an interval of s, the roots of
// (g.c + s g.n)^2 = cos^2 delta (1 + s^2) (c the unit vector to c3); [lo, hi]
// spans the intervals of the shared cells.  Returns false when there is none.
//
// FP32 on unit vectors normalised in FP64: the products lose below 2e-6, which
// the cells' cosines lowered by 1e-4 cover (a cell only grows), and the radius
// bound carries 2e-5.  Where a cell holds (nearly) the normal itself the roots
// are unbounded and its interval is taken as that whole side.  An
// ill-conditioned face is not restricted (lo = -infinity).  The cells of the
// six cube faces are one table in the frame of their face (w.cell).
// key: the squared radius of the larger end sphere (it only orders the faces
// into waves of similar work).
__device__ inline bool face_interval(const Params &P, const Work &w, uint32_t si, uint32_t sj, float &lo, float &hi,
                                     float &key) {
  uint64_t sh[6];
  bool share = false;
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    sh[k] = w.rmask[6 * si + k] & w.rmask[6 * sj + k];
    share |= sh[k] != 0;
  }
  if (!share) return false;
  const V3 a = gpt(w, si), b = gpt(w, sj);
  const double aa = dot(a, a), bb = dot(b, b), ab = dot(a, b);
  const double D = aa * bb - ab * ab;
  lo = -INFINITY;
  hi = INFINITY;
  key = INFINITY;
  if (!(D > 1e-6 * (aa * bb + fabs(ab) * fabs(ab)))) return true;
  const V3 amb = sub(a, b);
  const double r2 = aa * bb * dot(amb, amb) / (4.0 * D);
  const double al = bb * (aa - ab), be = aa * (bb - ab);
  const V3 g = {al * a.x + be * b.x, al * a.y + be * b.y, al * a.z + be * b.z}, n = cross(a, b);
  const double ig = __builtin_amdgcn_rsq(dot(g, g)), in = __builtin_amdgcn_rsq(D);
  const float cx = (float)(g.x * ig), cy = (float)(g.y * ig), cz = (float)(g.z * ig);
  const float nx = (float)(n.x * in), ny = (float)(n.y * in), nz = (float)(n.z * in);
  const float ir3 = (float)__builtin_amdgcn_rsq(r2);
  if (!(fabsf(cx) <= 1.001f && fabsf(nx) <= 1.001f && ir3 > 1e-30f && ir3 < 1e30f)) return true;  // out of FP32's range
  float l = INFINITY, h = -INFINITY;
  uint32_t cells = 0;
  // only the cells that the pencil's great circle can meet (of the others, q < 0)
  const uint64_t *strip = P.strips + 8 * strip_of(cy * nz - cz * ny, cz * nx - cx * nz, cx * ny - cy * nx);
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    uint64_t mm = sh[k] & strip[k];
    // c and n in the frame of cube face k
    const float sg = k % 2 ? -1.0f : 1.0f;
    const float kc[3] = {sg * (k < 2 ? cx : k < 4 ? cy : cz), k < 2 ? cy : k < 4 ? cz : cx, k < 2 ? cz : k < 4 ? cx : cy};
    const float kn[3] = {sg * (k < 2 ? nx : k < 4 ? ny : nz), k < 2 ? ny : k < 4 ? nz : nx, k < 2 ? nz : k < 4 ? nx : ny};
    while (mm) {
      const int c = 64 * k + __ffsll((long long)mm) - 1;
      mm &= mm - 1;
      cells++;
      const float ratio = w.rho[c] * ir3;
      const float sc2 = ratio * ratio * (1.0f + 2e-5f) - (1.0f - 1e-5f);
      if (sc2 < 0.0f) continue;
      const float4 cf = w.cell[c & 63];
      const float ga = cf.x * kc[0] + cf.y * kc[1] + cf.z * kc[2], gn = cf.x * kn[0] + cf.y * kn[1] + cf.z * kn[2];
      const float cd = cf.w - 1e-4f, kk = cd * cd;
      const float q = ga * ga + gn * gn - kk, den = kk - gn * gn;
      if (q < 0.0f) continue;
      const float sc = __builtin_amdgcn_sqrtf(sc2);
      float s1, s2;
      if (den > 0.02f) {
        if (ga <= 0.0f) continue;  // the opposite direction
        const float root = cd * __builtin_amdgcn_sqrtf(q), inv = __builtin_amdgcn_rcpf(den);
        s1 = fmaxf((ga * gn - root) * inv, -sc);
        s2 = fminf((ga * gn + root) * inv, sc);
      } else {
        s1 = gn > 0.0f ? 0.0f : -sc;
        s2 = gn > 0.0f ? sc : 0.0f;
      }
      if (s1 > s2) continue;
      l = fminf(l, s1);
      h = fmaxf(h, s2);
    }
  }
  add_flops32(w, (uint64_t)cells * kF32Cell);
  lo = l;
  hi = h;
  const float e = fmaxf(fabsf(l), fabsf(h));
  key = (float)r2 * (1.0f + e * e);
  return l <= h;
}

// Pairs, faces and tetrahedra of anchor u over its compacted region (M
// points at the front of the point arrays, masks by region slot, cell radii
// in w.rho); *sK == 0 and *sregion == kInvalid on entry, visible to every
// lane.
//
// An anchor may be split over several workgroups (SPLIT: blockIdx.y of
// gridDim.y, each with its own copy of the region): the candidate vertices
// are listed in region order, so every workgroup sees the same numbering of
// the faces, and takes its share of them and of the pairs.  The workgroups
// beyond one per kSplitFaces candidate faces have nothing to do (2 048: the
// mixture's catalogue 3% slower; 512 below a wave's round).
constexpr uint64_t kSplitFaces = 1024;
template <bool BIG, bool SPLIT, int WAVES>
__device__ void anchor_faces(const Params &P, const Work &w, uint32_t u, uint32_t M, uint32_t *sK_,
                             uint32_t *sregion_) {
  uint32_t &sK = *sK_;
  uint32_t &sregion = *sregion_;
  const int t = threadIdx.x;
  // candidate vertices (ids above the anchor) in region order (a rank sort
  // by direction cell, to give neighbouring lanes overlapping pencil capsules,
  // measured slower); the FP32 copies of the region's coordinates for the
  // face passes
  if (t < 64) {
    uint32_t k = 0;
    for (uint32_t s0 = 0; s0 < M; s0 += 64) {
      const uint32_t s = s0 + t;
      const bool above = s < M && w.gid[min(s, M - 1)] > u;
      const uint64_t m = __ballot(above);
      if (above) w.kidx[k + (uint32_t)__popcll(m & ((1ull << t) - 1ull))] = (uint16_t)s;
      k += (uint32_t)__popcll(m);
    }
    if (t == 0) sK = k;
  }
  for (uint32_t s = t; s < M; s += blockDim.x) {
    const V3 p = gpt(w, s);
    w.f[s] = make_float4((float)p.x, (float)p.y, (float)p.z, (float)sqrt(dot(p, p)));
  }
  __syncthreads();
  const uint32_t Kc = sK;
  const uint64_t F = Kc ? (uint64_t)Kc * (Kc - 1) / 2 : 0;
  uint32_t part = 0, parts = 1;
  if (SPLIT) {
    part = blockIdx.y;
    parts = (uint32_t)min((uint64_t)gridDim.y, F / kSplitFaces + 1);
    if (part >= parts) return;
  }
  // 3. pairs (u, v), v > u
  for (uint32_t k = part * blockDim.x + t; k < Kc; k += parts * blockDim.x)
    process_pair(P, w, u, M, w.kidx[k], &sregion);
  // 4. faces (u, v, w), u < v < w, whose members share a cell.  Each wave
  // takes 64 candidate faces at a time: first passes one per lane, then the
  // queued sides and tetrahedra one per lane (LDS path; the global-memory
  // path works in place).
  __shared__ uint32_t q_pair[WAVES][128];
  __shared__ uint32_t q_face[WAVES][128];
  __shared__ uint32_t q_key[WAVES][128];  // key (a positive float) with its low 7 bits the position: no ties
  __shared__ float q_lo[WAVES][128], q_hi[WAVES][128];
  __shared__ uint32_t q_tet[WAVES][kTetQ];
  __shared__ uint32_t q_n[WAVES];
  const int wave = t >> 6, lane = t & 63, nwaves = (int)(blockDim.x >> 6);
  WaveQueues wq{q_tet[wave], &q_n[wave]};
  WaveQueues *q = BIG ? nullptr : &wq;
  if (lane == 0) q_n[wave] = 0;
  wave_sync();
  // candidate face fidx -> region slots of (v, w): the pair (i < j) of the
  // strictly lower triangle
  auto face_of = [&](uint64_t fidx, uint32_t &si, uint32_t &sj) {
    const uint32_t f = (uint32_t)fidx;  // at most 2048 x 2047 / 2
    uint32_t j = (uint32_t)((1.0f + __builtin_amdgcn_sqrtf(1.0f + 8.0f * (float)f)) * 0.5f);
    while (j * (j - 1) / 2 > f) j--;
    while ((j + 1) * j / 2 <= f) j++;
    const uint32_t i = f - j * (j - 1) / 2;
    si = w.kidx[i];
    sj = w.kidx[j];
  };
  if (BIG) {
    for (uint64_t base = ((uint64_t)part * nwaves + wave) * 64; base < F; base += (uint64_t)parts * nwaves * 64) {
      const uint64_t fidx = base + lane;
      if (fidx >= F) continue;
      uint32_t si, sj;
      face_of(fidx, si, sj);
      float lo, hi, key;
      if (face_interval(P, w, si, sj, lo, hi, key)) process_face<false>(P, w, u, M, si, sj, lo, hi, &sregion, q);
    }
  } else {
    // Each wave lists the candidate faces that share a cell (q_pair), takes 64
    // of them at a time through the interval test, so that its lanes are full
    // (about half of the candidates share none), and collects up to 128
    // feasible faces with their pencil intervals; it orders them by the extent of their pencils, then runs the first passes
    // of the 64 largest one per lane (lanes of similar work), then the queued
    // tetrahedra; the smaller ones wait for the next round.
    uint32_t nf = 0, np = 0;  // faces and candidates in the wave's lists (uniform)
    uint64_t cbase = ((uint64_t)part * nwaves + wave) * 64;
    const uint64_t cstride = (uint64_t)parts * nwaves * 64;
    for (;;) {
      while (nf <= 64 && (np || cbase < F)) {
        while (np < 64 && cbase < F) {
          const uint64_t fidx = cbase + lane;
          bool share = false;
          uint32_t si = 0, sj = 0;
          if (fidx < F) {
            face_of(fidx, si, sj);
            for (int k = 0; k < 6; ++k) share |= (w.rmask[6 * si + k] & w.rmask[6 * sj + k]) != 0;
          }
          const uint64_t m = __ballot(share);
          if (share) q_pair[wave][np + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = si | (sj << 10);
          np += (uint32_t)__popcll(m);
          cbase += cstride;
        }
        wave_sync();
        const uint32_t got = min(np, 64u);
        np -= got;
        bool ok = false;
        uint32_t fv = 0;
        float key = 0.0f, lo = 0.0f, hi = 0.0f;
        if ((uint32_t)lane < got) {
          fv = q_pair[wave][np + lane];
          ok = face_interval(P, w, fv & 1023u, fv >> 10, lo, hi, key);
        }
        const uint64_t m = __ballot(ok);
        if (ok) {
          const uint32_t at = nf + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
          q_face[wave][at] = fv;
          q_key[wave][at] = (__float_as_uint(key) & ~127u) | at;
          q_lo[wave][at] = lo;
          q_hi[wave][at] = hi;
        }
        nf += (uint32_t)__popcll(m);
        wave_sync();  // the list's words are read before the next ones take them
      }
      wave_sync();
      if (nf > 64) {
        // rank sort of the list by key, ascending
        uint32_t fv[2], kv[2], rk[2] = {0, 0};
        float lv[2], hv[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const uint32_t i = (uint32_t)lane + 64u * h;
          const bool has = i < nf;
          kv[h] = has ? q_key[wave][i] : ~0u;
          fv[h] = has ? q_face[wave][i] : 0;
          lv[h] = has ? q_lo[wave][i] : 0.0f;
          hv[h] = has ? q_hi[wave][i] : 0.0f;
        }
        for (uint32_t j = 0; j < nf; ++j) {
          const uint32_t kj = q_key[wave][j];
          rk[0] += kj < kv[0];
          rk[1] += kj < kv[1];
        }
        wave_sync();
#pragma unroll
        for (int h = 0; h < 2; ++h)
          if ((uint32_t)lane + 64u * h < nf) {
            q_face[wave][rk[h]] = fv[h];
            q_lo[wave][rk[h]] = lv[h];
            q_hi[wave][rk[h]] = hv[h];
            q_key[wave][rk[h]] = (kv[h] & ~127u) | rk[h];
          }
        wave_sync();
      }
      const uint32_t take = min(nf, 64u);
      nf -= take;
      if ((uint32_t)lane < take) {
        const uint32_t fv = q_face[wave][nf + lane];
        const uint32_t si = fv & 1023u, sj = fv >> 10;
        process_face<true>(P, w, u, M, si, sj, q_lo[wave][nf + lane], q_hi[wave][nf + lane], &sregion, q);
      }
      wave_sync();
      // whole rounds of 64 tetrahedra (the top of the queue); the rest waits
      // for the next round's, so that the lanes stay busy, or ends the anchor
      const bool last = nf == 0 && np == 0 && cbase >= F;
      const uint32_t nt = min(q_n[wave], kTetQ);
      const uint32_t full = last ? nt : nt & ~63u;
#pragma unroll 1
      for (uint32_t it = nt - full + lane; it < nt; it += 64) {
        const uint32_t item = q_tet[wave][it];
        process_tet(P, w, u, M, item & 1023u, (item >> 10) & 1023u, item >> 20, &sregion);
      }
      if (last) break;
      wave_sync();
      if (lane == 0) q_n[wave] = nt - full;
      wave_sync();
    }
  }
  __syncthreads();
  if (t == 0) {
    if (*w.cand) atomicAdd(&P.counters[3], (unsigned long long)*w.cand);
    if (w.flops && *w.flops) atomicAdd(&P.counters[5], *w.flops);
    if (w.flops32 && *w.flops32) atomicAdd(&P.counters[6], *w.flops32);
  }
}

// The whole work of one anchor on a global slab: certificate, region, and
// (unless P.probe) the enumeration in place.
__device__ void anchor_work(const Params &P, const Work &w, uint32_t u, uint32_t a) {
  __shared__ uint32_t sM, sK, sflag, sregion;
  const int t = threadIdx.x;
  const uint32_t G = P.gcount[u];
  const uint64_t off = P.goff[u];
  const double ux = P.X[u], uy = P.Y[u], uz = P.Z[u];
  const double Rg = P.radius[u];
  __shared__ uint32_t scan_buf[kBlock];
  if (t == 0) { sM = 0; sK = 0; sflag = 0; sregion = kInvalid; }
  if (G <= 4 * blockDim.x) {
    // load in increasing distance from the anchor (rank sort in LDS), so that
    // every scan below meets the points most likely to be inside first
    for (uint32_t i = t; i < G; i += blockDim.x) {
      uint32_t id = P.glist[off + i];
      double dx = P.X[id] - ux, dy = P.Y[id] - uy, dz = P.Z[id] - uz;
      w.gx[i] = dx * dx + dy * dy + dz * dz;
    }
    __syncthreads();
    uint32_t rank[4];
    for (int r = 0; r < 4; ++r) {
      uint32_t i = t + r * blockDim.x;
      rank[r] = 0;
      if (i >= G) continue;
      const double di = w.gx[i];
      uint32_t cnt = 0;
      for (uint32_t j = 0; j < G; ++j) {
        const double dj = w.gx[j];
        cnt += (dj < di) || (dj == di && j < i);
      }
      rank[r] = cnt;
    }
    __syncthreads();
    for (int r = 0; r < 4; ++r) {
      uint32_t i = t + r * blockDim.x;
      if (i >= G) continue;
      uint32_t id = P.glist[off + i];
      w.gid[rank[r]] = id;
      w.gx[rank[r]] = P.X[id] - ux;
      w.gy[rank[r]] = P.Y[id] - uy;
      w.gz[rank[r]] = P.Z[id] - uz;
    }
  } else {
    for (uint32_t i = t; i < G; i += blockDim.x) {
      uint32_t id = P.glist[off + i];
      w.gid[i] = id;
      w.gx[i] = P.X[id] - ux;
      w.gy[i] = P.Y[id] - uy;
      w.gz[i] = P.Z[id] - uz;
    }
  }
  __syncthreads();
  // FP32 copy of the offsets with their lengths (rounded up), for the
  // certificate and the masks
  for (uint32_t i = t; i < G; i += blockDim.x) {
    const double x = w.gx[i], y = w.gy[i], z = w.gz[i];
    w.fc[i] = make_float4((float)x, (float)y, (float)z, (float)sqrt(x * x + y * y + z * z) * (1.0f + 1e-6f));
  }
  __syncthreads();
  // 1. direction-cell certificate (FP32; every rounding errs towards larger radii)
  const int need_cover = P.s_max - 1;
  // the points come in increasing distance when the rank sort ran: a point at
  // distance l covers at radius >= l / 2 (up to the FP32 rounding, inside the
  // factor below), so once l / 2 exceeds the list's last entry no later point
  // can enter it (and dropping points only enlarges the radius anyway)
  const bool by_distance = G <= 4 * blockDim.x;
  uint32_t covers = 0;  // point-cell tests (FP32 count)
  for (int c = t; c < kCells; c += blockDim.x) {
    const CellF cf = cell_f(P.cellf + 8 * c);
    float best[kCoverCap];  // the last need_cover of them; the others stay below
#pragma unroll
    for (int j = 0; j < kCoverCap; ++j) best[j] = j < kCoverCap - need_cover ? -INFINITY : INFINITY;
    for (uint32_t i = 0; i < G; ++i) {
      const float4 q = w.fc[i];
      if (!(q.w > kTinyLen)) continue;  // skipping a point only enlarges the radius
      if (by_distance && q.w * 0.49999f > best[kCoverCap - 1]) break;
      covers++;
      const float ct = (q.x * cf.dx + q.y * cf.dy + q.z * cf.dz) * __builtin_amdgcn_rcpf(q.w);
      if (ct <= 0.0f) continue;
      const float st = __builtin_amdgcn_sqrtf(fmaxf(0.0f, 1.0f - ct * ct));
      const float cs = ct * cf.cosd - st * cf.sind;  // cos(theta + delta)
      if (cs < 0.01f) continue;  // ill-conditioned cover: skipped
      const float r = q.w * __builtin_amdgcn_rcpf(2.0f * cs);
      if (!(r < best[kCoverCap - 1])) continue;
#pragma unroll
      for (int j = kCoverCap - 1; j > 0; --j) best[j] = __builtin_amdgcn_fmed3f(best[j - 1], r, best[j]);
      best[0] = fminf(best[0], r);
    }
    w.rho[c] = cell_radius(P, c, best[kCoverCap - 1], ux, uy, uz);
  }
  add_flops32(w, (uint64_t)covers * kF32Cover);
  __syncthreads();
  __shared__ float s_rmax2, s_wlim[kCells / 64];
  if (t == 0) {
    double m = 0, wm[kCells / 64] = {};
    for (int c = 0; c < kCells; ++c) {
      m = fmax(m, w.rho[c]);
      wm[c >> 6] = fmax(wm[c >> 6], w.rho[c]);
    }
    // 2 max rho in FP32, rounded up past the slack of the membership test
    // (over all cells and over each mask word's 64)
    s_rmax2 = (float)(2.0 * m) * 1.0001f;
    for (int wd = 0; wd < kCells / 64; ++wd) s_wlim[wd] = (float)(2.0 * wm[wd]) * 1.0001f;
    if (2.0 * m > Rg) {
      widen(P, u, 2.0 * m, Rg);
      sflag = 1;
    }
  }
  __syncthreads();
  if (sflag) return;
  const float rmax2 = s_rmax2;
  // 2. region membership masks, compacted in gathered order (chunks of four
  // points per lane)
  uint32_t members = 0;
  for (uint32_t c0 = 0; c0 < G; c0 += 4 * blockDim.x) {
    const uint32_t g = min(G - c0, 4 * blockDim.x);
    const uint32_t chunk = (g + blockDim.x - 1) / blockDim.x;
    const uint32_t b0 = c0 + t * chunk;
    uint64_t mk[4][6];  // static indices only: the masks stay in registers
    bool mem[4];
    uint32_t cnt = 0;
#pragma unroll
    for (uint32_t r = 0; r < 4; ++r) {
      mem[r] = false;
      if (r < chunk && t * chunk + r < g) {
        mem[r] = member_mask(P, w, b0 + r, rmax2, s_wlim, mk[r]);
        cnt += mem[r];
      }
    }
    scan_buf[t] = cnt;
    __syncthreads();
    for (int o = 1; o < (int)blockDim.x; o <<= 1) {
      uint32_t v = t >= o ? scan_buf[t - o] : 0;
      __syncthreads();
      scan_buf[t] += v;
      __syncthreads();
    }
    uint32_t slot = members + scan_buf[t] - cnt;
#pragma unroll
    for (uint32_t r = 0; r < 4; ++r) {
      if (!mem[r]) continue;
      w.ridx[slot] = b0 + r;
#pragma unroll
      for (int k = 0; k < 6; ++k) w.rmask[6 * slot + k] = mk[r][k];
      slot++;
    }
    members += scan_buf[blockDim.x - 1];
    __syncthreads();
  }
  if (t == 0) sM = members;
  __syncthreads();
  const uint32_t M = sM;
  // the region's points move to the front of the point arrays, in region
  // order: from here on a region slot indexes them directly.  ridx ascends,
  // so every source lies at or after its destination and after the
  // destinations of earlier chunks; each chunk reads before it writes.
  for (uint32_t c0 = 0; c0 < M; c0 += blockDim.x) {
    const uint32_t s = c0 + t;
    double x = 0, y = 0, z = 0;
    uint32_t id = 0;
    if (s < M) {
      const uint32_t gi = w.ridx[s];
      x = w.gx[gi];
      y = w.gy[gi];
      z = w.gz[gi];
      id = w.gid[gi];
    }
    __syncthreads();
    if (s < M) {
      w.gx[s] = x;
      w.gy[s] = y;
      w.gz[s] = z;
      w.gid[s] = id;
    }
    __syncthreads();
  }
  if (P.probe) {
    // the region is known and compacted in the slab; one that fits LDS is
    // enumerated there (k_anchor_region)
    if (t == 0) probed(P, u, a, M);
    return;
  }
  anchor_faces<true, false, kBlock / 64>(P, w, u, M, &sK, &sregion);
}

__device__ inline void probed(const Params &P, uint32_t u, uint32_t a, uint32_t M) {
  if (M > P.region_limit) {
    // budget stop: the anchor stays open, the catalogue is conditional
    atomicAdd(&P.counters[kOpenCount], 1ull);
    atomicMax(&P.counters[kOpenLargest], (unsigned long long)M);
    return;
  }
  P.region[u] = M;
  if (M) list_add(P, M <= P.one_wave ? L_TINY : M <= P.two_waves ? L_LITTLE : M <= kRegionCap ? L_SMALL : M <= kRegionCapWide ? L_MID : M <= kRegionCapHuge ? L_LARGE : L_SLAB, a);
}

// Certificate and region of one anchor per workgroup, gathers of up to GCAP
// points in LDS: six waves, one direction cell per lane.  A cell's radius
// takes a scan of the points in increasing distance; the membership masks come
// from the transposed loop, a wave per mask word and a ballot per point, so
// that the cell stays in registers, the point is a broadcast and a word's scan
// ends at the first point beyond the word's largest ball.  The region goes to
// the anchor's slab, and its enumeration is another launch (k_anchor_region):
// this kernel needs few registers and no enumeration queues, so more waves
// share a CU than when one kernel did both, and the enumeration is split over
// as many workgroups as its size asks for.  VALU bound.  Against one kernel per
// anchor (two LDS sizes): catalogue of a 2 003-point mixture 332 -> 116 ms,
// pipeline of 17 117 points K 4 19.3 -> 17.0 ms.  A scan that ends with the
// certificate's own radius (the (s_max - 1)-th) instead of the tenth: K 4 12.65
// -> 10.6 ms for 50 000 points' enumeration; four points at a time without
// branches: 10.65 -> 9.1 ms, K 10 38.3 -> 35.2 ms, catalogue of 256 points K 3
// 1.10 -> 1.03 ms.
//
// SLAB: the masks are built in the slab instead of LDS (98 KB for 2 048 points;
// 48 KB then remain, three workgroups a CU).  Such gathers took the
// global-memory kernel, whose 256 lanes scan all points for 384 cells and whose
// regions are not in increasing distance: 2 003-point mixture, 1 531 such
// anchors, catalogue 29.8 -> 26.0 ms.  Up to 4 096 points (98 KB, one workgroup a
// CU) it is no better: mixtures of 2 003, 3 000 and 4 000 points, K 10, 21.3,
// 130.5 and 459 ms with 2 048, 25.1, 126.8 and 486 with 4 096.
constexpr int kProbeBlock = kCells;
template <int GCAP, bool SLAB>
__global__ void __launch_bounds__(kProbeBlock) k_anchor_probe(Params P) {
  constexpr int kPer = (GCAP + kProbeBlock - 1) / kProbeBlock;
  constexpr int kWaves = kProbeBlock / 64;
  __shared__ __align__(16) float4 fc[GCAP];   // FP32 offset and distance (rounded up), ascending
  __shared__ uint32_t gid[GCAP];
  __shared__ __align__(16) uint64_t lmask[SLAB ? GCAP / 2 : 6 * GCAP];
  __shared__ float wmax[kWaves];
  __shared__ uint32_t wcount[kPer][kWaves];
  __shared__ unsigned long long flops32;
  const uint32_t a = blockIdx.x;
  if (a >= P.anchor_count) return;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const uint32_t u = P.anchors[a];
  const uint32_t G = P.gcount[u];
  if (G > (uint32_t)GCAP) {
    if (t == 0) list_add(P, G <= (uint32_t)kGatherCapWide ? L_WIDE : G <= (uint32_t)kGatherCapSlab ? L_WIDER : L_BIG, u);
    return;
  }
  if (t == 0) flops32 = 0;
  double *slab = P.scratch + (uint64_t)a * P.slab_doubles;
  const uint64_t S = P.gcap;
  float *srho = reinterpret_cast<float *>(slab + 3 * S);
  uint64_t *smask = reinterpret_cast<uint64_t *>(slab + slab_masks(S));
  uint32_t *sgid = reinterpret_cast<uint32_t *>(slab + slab_ids(S));
  uint64_t *rmask = SLAB ? smask : lmask;
  const uint64_t off = P.goff[u];
  const double ux = P.X[u], uy = P.Y[u], uz = P.Z[u];
  const double Rg = P.radius[u];  // before the first barrier: one lane may widen it below
  // load, ranked by distance (the keys sit in the mask area until the masks come)
  float *key = reinterpret_cast<float *>(lmask);
  float4 mine[kPer];
  uint32_t id[kPer];
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const uint32_t i = t + r * kProbeBlock;
    mine[r] = make_float4(0.f, 0.f, 0.f, INFINITY);
    id[r] = 0;
    if (i < G) {
      id[r] = P.glist[off + i];
      const double x = P.X[id[r]] - ux, y = P.Y[id[r]] - uy, z = P.Z[id[r]] - uz;
      mine[r] = make_float4((float)x, (float)y, (float)z, (float)sqrt(x * x + y * y + z * z) * (1.0f + 1e-6f));
      key[i] = mine[r].w;
    }
  }
  const uint32_t G4 = (G + 3) & ~3u;
  if (t < 4 && G + t < G4) key[G + t] = INFINITY;
  __syncthreads();
  uint32_t rank[kPer] = {};
  for (uint32_t j = 0; j < G4; j += 4) {
    const float4 k4 = *reinterpret_cast<const float4 *>(key + j);
    const float kv[4] = {k4.x, k4.y, k4.z, k4.w};
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
      const uint32_t i = t + r * kProbeBlock;
#pragma unroll
      for (int q = 0; q < 4; ++q) rank[r] += kv[q] < mine[r].w || (kv[q] == mine[r].w && j + q < i);
    }
  }
#pragma unroll
  for (int r = 0; r < kPer; ++r)
    if (t + r * kProbeBlock < G) {
      fc[rank[r]] = mine[r];
      gid[rank[r]] = id[r];
    }
  if (t < 4 && G + t < G4) fc[G + t] = make_float4(0.f, 0.f, 0.f, INFINITY);
  __syncthreads();
  // 1. direction-cell certificate (FP32; every rounding errs towards larger
  // radii): a point at distance l covers at radius >= l / 2 (up to the FP32
  // rounding, inside the factor below), so once l / 2 exceeds the list's last
  // entry no later point can enter it (and dropping points only enlarges the
  // radius anyway)
  const int c = t;
  const CellF cf = cell_f(P.cellf + 8 * c);
  float rho;
  {
    // the last s_max - 1 entries are the least radii, the others stay below:
    // the scan ends with the certificate's own radius
    float best[kCoverCap];
#pragma unroll
    for (int j = 0; j < kCoverCap; ++j) best[j] = j < kCoverCap - (P.s_max - 1) ? -INFINITY : INFINITY;
    uint32_t covers = 0;
    // four points at a time, for the latency of a launch of few anchors
    for (uint32_t i = 0; i < G; i += 4) {
      if (fc[i].w * 0.49999f > best[kCoverCap - 1]) break;
      covers += 4;
      float r[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float4 q = fc[i + k];
        const float ct = (q.x * cf.dx + q.y * cf.dy + q.z * cf.dz) * __builtin_amdgcn_rcpf(q.w);
        const float st = __builtin_amdgcn_sqrtf(fmaxf(0.0f, 1.0f - ct * ct));
        const float cs = ct * cf.cosd - st * cf.sind;  // cos(theta + delta)
        // skipping a point (lost to underflow, ill-conditioned) only enlarges the radius
        const bool covering = q.w > kTinyLen && ct > 0.0f && cs >= 0.01f;
        r[k] = covering ? q.w * __builtin_amdgcn_rcpf(2.0f * cs) : INFINITY;
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (!(r[k] < best[kCoverCap - 1])) continue;
#pragma unroll
        for (int j = kCoverCap - 1; j > 0; --j) best[j] = __builtin_amdgcn_fmed3f(best[j - 1], r[k], best[j]);
        best[0] = fminf(best[0], r[k]);
      }
    }
    if (P.count_flops) atomicAdd(&flops32, (unsigned long long)covers * kF32Cover);
    rho = cell_radius(P, c, best[kCoverCap - 1], ux, uy, uz);
  }
  float m = rho;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
  // 2 max rho over the word's cells in FP32, past the slack of the test
  const float wlim = (float)(2.0 * (double)m) * 1.0001f;
  if (lane == 0) wmax[wave] = m;
  __syncthreads();
  double need = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) need = fmax(need, 2.0 * (double)wmax[w]);
  if (need > Rg) {  // uniform
    if (t == 0) widen(P, u, need, Rg);
    return;
  }
  // 2. region membership masks, word `wave`: FP32 with slack, a point may
  // only be included too often
  {
    uint32_t tests = 0;
    const float reach = 2.0f * rho * (1.0f + 1e-5f);
    bool open = true;  // points up to the word's limit
    for (uint32_t i0 = 0; i0 < G; i0 += 64) {
      uint64_t word = 0;
      const uint32_t n = min(64u, G - i0);
      for (uint32_t j = 0; open && j < n; j += 4) {
        if (fc[i0 + j].w > wlim) {
          open = false;
          break;
        }
        tests += 4;
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
          const float4 q = fc[i0 + j + k];
          const float ct = (q.x * cf.dx + q.y * cf.dy + q.z * cf.dz) * __builtin_amdgcn_rcpf(q.w);
          const float cm = ct >= cf.cosd ? 1.0f  // cos(max(theta - delta, 0))
                                         : ct * cf.cosd + __builtin_amdgcn_sqrtf(fmaxf(0.0f, 1.0f - ct * ct)) * cf.sind;
          // distance lost to underflow: member everywhere
          const uint64_t b = __ballot(q.w <= reach * (cm + 1e-5f) || !(q.w > kTinyLen));
          word = (uint32_t)lane == j + k ? b : word;
        }
      }
      if (i0 + lane < G) rmask[6 * (i0 + lane) + wave] = word;
    }
    if (P.count_flops && lane == 0) atomicAdd(&flops32, (unsigned long long)tests * 64 * kF32Mask);
  }
  __syncthreads();
  // members, compacted in order of distance into the slab
  uint64_t bits[kPer];
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const uint32_t i = t + r * kProbeBlock;
    uint64_t any = 0;
    if (i < G)
      for (int k = 0; k < 6; ++k) any |= rmask[6 * i + k];
    bits[r] = __ballot(any != 0);
    if (lane == 0) wcount[r][wave] = (uint32_t)__popcll(bits[r]);
  }
  __syncthreads();
  srho[c] = rho;
  uint32_t M = 0;
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    uint32_t slot = M;
    for (int w = 0; w < kWaves; ++w) {
      if (w < wave) slot += wcount[r][w];
      M += wcount[r][w];
    }
    const bool member = (bits[r] >> lane) & 1;
    slot += (uint32_t)__popcll(bits[r] & ((1ull << lane) - 1ull));
    const uint32_t i = t + r * kProbeBlock;
    uint64_t row[6];
    if (member)
      for (int k = 0; k < 6; ++k) row[k] = rmask[6 * i + k];
    // in the slab the rows move to the front of where they are: every row of
    // the chunk is read before one is written
    if (SLAB) __syncthreads();
    if (member) {
      const uint32_t v = gid[i];
      slab[slot] = P.X[v] - ux;
      slab[S + slot] = P.Y[v] - uy;
      slab[2 * S + slot] = P.Z[v] - uz;
      sgid[slot] = v;
      for (int k = 0; k < 6; ++k) smask[6 * (uint64_t)slot + k] = row[k];
    }
  }
  if (t == 0) {
    // a region beyond the LDS enumerations is probed again on its own slab
    if (M > (uint32_t)kRegionCapHuge) list_add(P, L_BIG, u);
    else probed(P, u, a, M);
    if (P.count_flops) atomicAdd(&P.counters[6], flops32);
  }
}

// Offset (in doubles, even) of the FP32 offsets in a global slab of gather
// capacity G; the slab holds big_fc_offset(G) + 2G doubles.
__host__ __device__ inline uint64_t big_fc_offset(uint64_t G) {
  return (slab_ids(G) + (3 * G + 1) / 2 + 1 + 1) & ~1ull;
}

// Anchors whose gather or region exceeds LDS: the same work on global slabs.
__global__ void __launch_bounds__(kBlock) k_anchor_big(Params P) {
  const uint32_t a = blockIdx.x;
  if (a >= P.anchor_count) return;
  const uint32_t u = P.anchors[a];
  double *slab = P.scratch + (uint64_t)a * P.slab_doubles;
  const uint32_t G = P.gcap;
  Work w{};
  w.gx = slab;
  w.gy = slab + G;
  w.gz = slab + 2 * G;
  w.rho = reinterpret_cast<float *>(slab + 3 * G);
  w.rmask = (uint64_t *)(slab + slab_masks(G));
  w.gid = (uint32_t *)(slab + slab_ids(G));
  w.ridx = w.gid + G;
  w.kidx = reinterpret_cast<uint16_t *>(w.ridx + G);
  w.fc = reinterpret_cast<float4 *>(slab + big_fc_offset(G));
  // the FP32 region copies take the FP32 offsets' area once the region is
  // compacted (4G floats)
  w.f = w.fc;
  __shared__ uint32_t cand;
  __shared__ unsigned long long flops;
  if (threadIdx.x == 0) { cand = 0; flops = 0; }
  __syncthreads();
  w.cand = &cand;
  w.flops = P.count_flops ? &flops : nullptr;
  w.slab = a;
  __shared__ float4 cell[64];
  if (threadIdx.x < 64) cell[threadIdx.x] = *reinterpret_cast<const float4 *>(P.cellf + 8 * threadIdx.x);
  w.cell = cell;
  anchor_work(P, w, u, a);
}

// Enumeration of probed regions that fit LDS: the region (coordinates,
// PointIds, masks) and cell radii are loaded from the anchor's slab, and the
// face phase runs on them with the wave queues.  Sizes: up to 384 points
// (three workgroups of four waves per CU at 168 VGPRs), up to 640 (two) and up
// to 1 023 (one of eight waves; region slots stay below 1 024, as the packed
// queue items need).  list: the launch's slabs with such a region.
//
// In launches of many anchors small regions take one wave (up to 96 points) or
// two (up to 180, the most of which six workgroups share a CU): a wave's 64
// lanes fill from its own share of an anchor's faces, of which a K 4 lattice
// has 89 in all, and the last rounds of fewer waves are less often part empty.
// 50 000-point lattice: K 10 57.7 -> 53.6 ms, K 4 18.3 -> 14.3 ms.  With fewer
// anchors than the CUs hold waves of one launch after another loses more (1 000
// points 2.05 -> 3.2 ms), hence the rule by the launch's anchors.
//
// One workgroup per anchor left the chip idle wherever tens of anchors held
// large regions (43 anchors: 313 ms, each workgroup alone on its CU): a launch
// asks for about kRegionParts workgroups in all, a few per CU slot so that
// the longest ones do not end it alone.  A 2 003-point mixture's catalogue:
// 885 -> 332 ms.
//
// Bound by VALU issue: 14 G wave instructions for the 50 000-point lattice K 10
// (25 million records), 23 of the launches' 28 ms; about 4.5 G in the points of
// the faces' passes (39 million wave steps), 2.8 G in the interval walks (55
// million), 1.8 G in the pencil tests (143 million slots), 1.3 G in the
// tetrahedra.  FP64 state of rare passes spilled 160 registers (k_rescan has
// them now).  Scans that end at a sphere's diameter and id lists read from bit
// masks: 73 -> 58 ms for the whole enumeration with its probes; sweep lists of
// one word per entry, filled without branches, bits shifted in by add with
// carry and a rank sort without ties: 46 -> 39 ms, 1 000 points 1.75 -> 1.55 ms,
// uniform 8 000 points K 8 8.5 -> 6.5 ms.
constexpr uint32_t kRegionParts = 4096;
constexpr uint32_t kSmallRegionLaunch = 8192;  // anchors of a launch that splits off the small regions
template <int RCAP, int WAVES, int PER_SIMD>
__global__ void __launch_bounds__(64 * WAVES, PER_SIMD) k_anchor_region(Params P, const uint32_t *__restrict__ list) {
  const uint32_t a = list[blockIdx.x];
  const uint32_t u = P.anchors[a];
  const uint32_t M = P.region[u];
  if (M > (uint32_t)RCAP) return;
  const uint64_t G = P.gcap;
  const double *slab = P.scratch + (uint64_t)a * P.slab_doubles;
  const uint64_t *smask = (const uint64_t *)(slab + slab_masks(G));
  const uint32_t *sgid = (const uint32_t *)(slab + slab_ids(G));
  __shared__ double gx[RCAP], gy[RCAP], gz[RCAP];
  __shared__ uint32_t gid[RCAP];
  __shared__ float rho[kCells];
  __shared__ uint64_t rmask[6 * RCAP];
  __shared__ uint16_t kidx[RCAP];
  __shared__ float4 f[RCAP];
  __shared__ float4 cell[64];
  __shared__ uint32_t cand, sK, sregion;
  __shared__ unsigned long long flops, flops32;
  const int t = threadIdx.x;
  if (t < 64) cell[t] = *reinterpret_cast<const float4 *>(P.cellf + 8 * t);
  if (P.ascending) {
    for (uint32_t i = t; i < M; i += blockDim.x) {
      gx[i] = slab[i];
      gy[i] = slab[G + i];
      gz[i] = slab[2 * G + i];
      gid[i] = sgid[i];
    }
    for (uint32_t i = t; i < 6 * M; i += blockDim.x) rmask[i] = smask[i];
  } else {
    // into increasing distance from the anchor (the same in every workgroup)
    constexpr int kPer = (RCAP + 64 * WAVES - 1) / (64 * WAVES);
    for (uint32_t i = t; i < M; i += blockDim.x) {
      const double x = slab[i], y = slab[G + i], z = slab[2 * G + i];
      gx[i] = x * x + y * y + z * z;
    }
    __syncthreads();
    uint32_t rank[kPer];
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
      const uint32_t i = t + r * 64 * WAVES;
      const double d = i < M ? gx[i] : 0.0;
      rank[r] = 0;
      for (uint32_t j = 0; j < M; ++j) rank[r] += gx[j] < d || (gx[j] == d && j < i);
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
      const uint32_t i = t + r * 64 * WAVES, q = rank[r];
      if (i >= M) continue;
      gx[q] = slab[i];
      gy[q] = slab[G + i];
      gz[q] = slab[2 * G + i];
      gid[q] = sgid[i];
      for (int k = 0; k < 6; ++k) rmask[6 * q + k] = smask[6 * (uint64_t)i + k];
    }
  }
  for (int c = t; c < kCells; c += blockDim.x) rho[c] = reinterpret_cast<const float *>(slab + 3 * G)[c];
  if (t == 0) { cand = 0; sK = 0; sregion = kInvalid; flops = 0; flops32 = 0; }
  __syncthreads();
  Work w{gx, gy, gz, gid, rho, nullptr, rmask, kidx, nullptr, &cand, P.count_flops ? &flops : nullptr, f,
         P.count_flops ? &flops32 : nullptr, true, a, cell};
  anchor_faces<false, true, WAVES>(P, w, u, M, &sK, &sregion);
}

// Sides of faces left by the enumeration of one launch, one per wave, in FP64
// over the anchor's slab (lanes over the points that the pencil can hold): a
// first scan finds the side's key threshold and the inside points behind it, a
// second one the apexes, each classified against the whole region.  The face
// pass has certified every sign with the same arithmetic.  Few sides come here
// (0 to a few hundred of a catalogue), so their latency counts: M / 64 steps
// a scan.  The grid is fixed; the number of sides is read on the device.
constexpr int kRescanBlocks = 4096;
__global__ void __launch_bounds__(64) k_rescan(Params P) {
  const unsigned long long count = min(P.counters[4], (unsigned long long)P.rescan_cap);
  const uint64_t G = P.gcap;
  const int K = P.s_max - 3, lane = threadIdx.x;
  unsigned long long evals = 0, cands = 0;
  for (unsigned long long it = blockIdx.x; it < count; it += kRescanBlocks) {
    const Rescan r = P.rescans[it];
    const uint32_t u = P.anchors[r.anchor], M = P.region[u], side = r.side & 1u;
    const int cin = (int)(r.side >> 1), need = K - cin;
    if (need <= 0) continue;
    double *slab = P.scratch + (uint64_t)r.anchor * P.slab_doubles;
    Work w{};
    w.gx = slab;
    w.gy = slab + G;
    w.gz = slab + 2 * G;
    w.gid = (uint32_t *)(slab + slab_ids(G));
    const V3 o = {P.X[u], P.Y[u], P.Z[u]};
    const V3 pv = sub({P.X[r.v], P.Y[r.v], P.Z[r.v]}, o), pw = sub({P.X[r.w], P.Y[r.w], P.Z[r.w]}, o);
    TriSphere f;
    f.init(pv, pw);
    const Pencil pen = face_pencil(f, r.lo, r.hi, false);
    uint32_t region_slot = kInvalid;
    // sign of the power and whether ahead of the side; false: not in the pencil
    auto key = [&](uint32_t s, int &sp, bool &ahead, double &tau, double &terr) {
      const uint32_t id = w.gid[s];
      if (id == r.v || id == r.w) return false;
      const V3 p = gpt(w, s);
      if (pen.outside(make_float4((float)p.x, (float)p.y, (float)p.z, (float)sqrt(dot(p, p))))) return false;
      evals++;
      double Pw, PA, H, HA;
      f.power(p, Pw, PA);
      f.height(p, H, HA);
      sp = cert_sign(Pw, PA);
      const int sh = cert_sign(H, HA);
      ahead = side == 0 ? sh > 0 : sh < 0;
      sweep_key(Pw, PA, H, HA, tau, terr);
      return true;
    };
    SweepList top;
    BehindList beh;
    top.init();
    beh.init();
    for (uint32_t s = lane; s < M; s += 64) {
      int sp;
      bool ahead;
      double tau, terr;
      if (!key(s, sp, ahead, tau, terr)) continue;
      // inside the triangle's sphere and behind this side: inside the
      // pencil's spheres until the sweep key reaches -tau
      if (sp < 0 && !ahead) beh.insert(-tau - terr);
      else if (sp > 0 && ahead) top.insert(tau, terr);
    }
    // the need-th smallest upper bound over the lanes' lists
    double thr = INFINITY;
    for (int k = 0; k < need; ++k) {
      thr = top.hi[0];
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) thr = fmin(thr, __shfl_xor(thr, d));
      const uint64_t who = __ballot(top.hi[0] == thr);
      if (lane == __ffsll((long long)who) - 1) top.pop();
    }
    for (uint32_t s0 = 0; s0 < M; s0 += 64) {
      const uint32_t s = s0 + lane;
      int sp = 0;
      bool ahead = false;
      double tau = 0, terr = 0;
      const bool apex = s < M && key(s, sp, ahead, tau, terr) && sp > 0 && ahead && w.gid[min(s, M - 1)] > r.w &&
                        !(tau - terr > thr);
      for (uint64_t todo = __ballot(apex); todo; todo &= todo - 1) {
        const int j = __ffsll((long long)todo) - 1;
        // inside points behind: counted while their key exceeds z's
        int ahead_of = beh.count_above(__shfl(tau + terr, j));
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) ahead_of += __shfl_xor(ahead_of, d);
        if (cin + ahead_of >= K) continue;
        const uint32_t id = w.gid[s0 + j];
        TetSphere t;
        const int wc = t.init(pv, pw, gpt(w, s0 + j));
        if (wc < 0) continue;
        cands++;
        const uint32_t ids[3] = {r.v, r.w, id};
        uint32_t interior[kMaxInterior];
#pragma unroll
        for (int k = 0; k < kMaxInterior; ++k) interior[k] = kInvalid;
        int nint = 0;
        bool open = wc == 0;
        for (uint32_t q0 = 0; wc > 0 && q0 < M && nint + 4 <= P.s_max; q0 += 64) {
          const uint32_t q = min(q0 + lane, M - 1), x = w.gid[q];
          int sd = 1;
          if (q0 + lane < M && x != r.v && x != r.w && x != id) sd = t.side(gpt(w, q));
          open |= __ballot(sd == 0) != 0;
          for (uint64_t in = __ballot(sd < 0); in; in &= in - 1) {
            const uint32_t y = __shfl(x, __ffsll((long long)in) - 1);
#pragma unroll
            for (int k = 0; k < kMaxInterior; ++k) interior[k] = k == nint ? y : interior[k];
            nint++;
          }
        }
        if (nint + 4 > P.s_max) continue;
        sort_static(interior, nint);
        if (lane == 0) {
          if (open) emit_fallback(P, w, u, 4, ids, 4, M, &region_slot);
          else emit_event(P, u, ids, 4, nint, interior, t.level(), t.level_err());
        }
      }
    }
  }
  if (lane == 0 && cands) atomicAdd(&P.counters[3], cands);
  if (P.count_flops && evals) atomicAdd(&P.counters[5], evals * (kFlopFacePoint + kFlopSweepKey));
}

// The list starts again; its longest length is kept for the host.
__global__ void k_rescans_done(Params P) {
  P.counters[kRescanMost] = max(P.counters[kRescanMost], P.counters[4]);
  P.counters[4] = 0;
}

// Ball count / emit around every anchor of the list: one wave per anchor over
// the wave tree, hits appended with ballot prefix counts.  The traversal
// order is fixed, so the count and emit passes visit the same points.  Bound
// by VALU issue of the group tests and distances.  With one thread per anchor
// walking the binary tree a pass took 230 us at 256 points and 0.7-0.9 ms at
// 17 117; the catalogue of 256 points went from 2.92 to 2.27 ms with this and
// the radius kernel below, the 17 117-point pipeline from 23.5 to 22.1 ms.
constexpr int kGatherBlock = 256;  // four waves, four anchors
template <bool EMIT>
__global__ void __launch_bounds__(kGatherBlock) k_gather(WaveTree T, const uint32_t *__restrict__ leaf_pos,
                                                         const uint32_t *__restrict__ anchors, uint32_t count,
                                                         const double *__restrict__ radius, uint32_t *gcount,
                                                         const uint64_t *__restrict__ goff, uint32_t *glist) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t a = blockIdx.x * (kGatherBlock / 64) + (threadIdx.x >> 6);
  if (a >= count) return;  // uniform over the wave
  const uint64_t below = (1ull << lane) - 1ull;
  const uint32_t u = anchors[a];
  const uint32_t p = leaf_pos[u];
  const double q[3] = {T.LX[p], T.LY[p], T.LZ[p]};
  const double R = radius[u];
  const double R2 = R * R * (1.0 + 1e-9);
  const WaveQuery Q(q[0], q[1], q[2]);
  double most = wave_bound(R2);
  const uint64_t base = EMIT ? goff[u] : 0;
  uint32_t cnt = 0;
  wave_tree_visit(T, Q, most, [&](uint32_t g) {
    const uint32_t lp = g * 64 + lane, at = min(lp, T.n - 1);
    const double dx = T.LX[at] - q[0], dy = T.LY[at] - q[1], dz = T.LZ[at] - q[2];
    const bool hit = lp < T.n && lp != p && dx * dx + dy * dy + dz * dz <= R2;
    const uint64_t m = __ballot(hit);
    if (EMIT && hit) glist[base + cnt + (uint32_t)__popcll(m & below)] = T.leaf_id[at];
    cnt += (uint32_t)__popcll(m);
  });
  if (!EMIT && lane == 0) gcount[u] = cnt;
}

// Initial gather radius of every point: factor x the distance to its kq-th
// nearest neighbour (kq <= 32), from outward-rounded FP32 differences.  The
// radius only sizes the first gather; the certificate widens any anchor it
// does not cover.  One wave per point over the wave tree, lane l holding the
// l-th smallest squared distance so far; bound by VALU issue (182 us at 256
// points with one thread per point).
constexpr int kRadiusBlock = 256;  // four waves, four points
__global__ void __launch_bounds__(kRadiusBlock) k_knn_radius(WaveTree T, int kq, float factor, double *radius) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t p = blockIdx.x * (kRadiusBlock / 64) + (threadIdx.x >> 6);
  if (p >= T.n) return;
  const double x = T.LX[p], y = T.LY[p], z = T.LZ[p];
  const float q[3] = {(float)x, (float)y, (float)z};
  const WaveQuery Q(x, y, z);
  // the differences are taken in the input's frame, whose FP32 rounding
  // (query half an ulp, box one ulp per axis) can bring a point nearer by up
  // to this much
  const float off = 3.5e-7f * fmaxf(fmaxf(fabsf(q[0]), fabsf(q[1])), fabsf(q[2]));
  float best = INFINITY, cut = INFINITY;
  double most = INFINITY;
  auto group = [&](uint32_t g) {
    const uint32_t lp = g * 64 + lane, at = min(lp, T.n - 1);
    const double v[3] = {T.LX[at], T.LY[at], T.LZ[at]};
    float d2 = 0.f;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const float d = fmaxf(fmaxf(__double2float_rd(v[a]) - q[a], q[a] - __double2float_ru(v[a])), 0.f);
      d2 += d * d;
    }
    const bool valid = lp < T.n && lp != p;
    uint64_t cand = __ballot(valid && d2 < cut);
    if (!cand) return;
    while (cand) {
      const int i = __builtin_amdgcn_readfirstlane(__ffsll((long long)cand) - 1);
      cand &= cand - 1;
      const float cd = __uint_as_float(lane_u32(__float_as_uint(d2), i));
      const uint32_t pos = (uint32_t)__popcll(__ballot(best <= cd));
      const float up = __shfl_up(best, 1u);
      best = lane < pos ? best : (lane == pos ? cd : up);
      cut = __uint_as_float(lane_u32(__float_as_uint(best), kq - 1));
      cand &= __ballot(d2 < cut);
    }
    const double r = sqrt((double)cut) * (1.0 + 1e-6) + (double)off;
    most = cut > 0.f ? wave_bound(r * r) : -1.0;  // nothing enters below a zero distance
  };
  const uint32_t own = p >> 6;
  group(own);
  wave_tree_visit(T, Q, most, [&](uint32_t g) {
    if (g != own) group(g);
  });
  if (lane == 0) radius[T.leaf_id[p]] = (double)factor * (sqrt((double)cut) * (1.0 + 1e-6));
}

// exclusive scan of gcount over the anchor list into goff (single workgroup)
__global__ void k_scan_offsets(const uint32_t *__restrict__ anchors, uint32_t count,
                               const uint32_t *__restrict__ gcount, uint64_t *goff, uint64_t *total) {
  __shared__ uint64_t part[1024];
  const int t = threadIdx.x;
  const uint32_t per = (count + blockDim.x - 1) / blockDim.x;
  const uint32_t b = t * per, e = min(b + per, count);
  uint64_t s = 0;
  for (uint32_t i = b; i < e; ++i) s += gcount[anchors[i]];
  part[t] = s;
  __syncthreads();
  for (int o = 1; o < (int)blockDim.x; o <<= 1) {
    uint64_t v = t >= o ? part[t - o] : 0;
    __syncthreads();
    part[t] += v;
    __syncthreads();
  }
  uint64_t run = part[t] - s;
  for (uint32_t i = b; i < e; ++i) {
    goff[anchors[i]] = run;
    run += gcount[anchors[i]];
  }
  if (t == (int)blockDim.x - 1) *total = part[t];
}

}  // namespace

// Direction cells: centre, cos/sin of the angular radius, chord bound.
static std::vector<double> make_cells() {
  std::vector<double> out(8 * kCells);
  const int G = 8;
  int q = 0;
  for (int f = 0; f < 6; ++f)
    for (int i = 0; i < G; ++i)
      for (int j = 0; j < G; ++j) {
        auto dir = [&](double s, double t, double v[3]) {
          double a = 2 * s - 1, b = 2 * t - 1, w[3];
          int ax = f / 2;
          double sg = (f % 2) ? -1 : 1;
          w[ax] = sg;
          w[(ax + 1) % 3] = a;
          w[(ax + 2) % 3] = b;
          double nn = std::sqrt(w[0] * w[0] + w[1] * w[1] + w[2] * w[2]);
          for (int k = 0; k < 3; ++k) v[k] = w[k] / nn;
        };
        double c[3];
        dir((i + 0.5) / G, (j + 0.5) / G, c);
        double delta = 0;
        for (int ci = 0; ci < 2; ++ci)
          for (int cj = 0; cj < 2; ++cj) {
            double v[3];
            dir((double)(i + ci) / G, (double)(j + cj) / G, v);
            double dt = c[0] * v[0] + c[1] * v[1] + c[2] * v[2];
            delta = std::max(delta, std::acos(std::min(1.0, dt)));
          }
        delta = delta * 1.01 + 1e-9;
        double *o = out.data() + 8 * q++;
        o[0] = c[0]; o[1] = c[1]; o[2] = c[2];
        o[3] = std::cos(delta);
        o[4] = std::sin(delta);
        o[5] = 2.0 * std::sin(delta / 2.0) * 1.001;
        o[6] = delta;
        o[7] = 0;
      }
  return out;
}

// The FP32 cells of the certificate and the membership masks (8 floats per
// cell: direction xyz, cos delta rounded down, sin delta rounded up, padding),
// so that every FP32 test errs towards a larger cell.
static std::vector<float> make_cells_f(const std::vector<double> &cells) {
  std::vector<float> out(8 * kCells, 0.0f);
  for (int c = 0; c < kCells; ++c) {
    const double *cd = cells.data() + 8 * c;
    float *o = out.data() + 8 * c;
    o[0] = (float)cd[0];
    o[1] = (float)cd[1];
    o[2] = (float)cd[2];
    o[3] = (float)cd[3] * (1.0f - 1e-6f);
    o[4] = (float)cd[4] * (1.0f + 1e-6f) + 1e-7f;
  }
  return out;
}

void supports_device(Context &c, int k_max, std::vector<EventRec> &events,
                     std::vector<FallbackRec> &fbs, std::vector<uint32_t> &fb_region,
                     mhgp_catalog_info *info);

void launch_radius(hipStream_t s, Context &c, int kq, CatalogBuffers &Bf) {
  hipLaunchKernelGGL(k_knn_radius, dim3(blocks_for(c.n, kRadiusBlock / 64)), dim3(kRadiusBlock), 0, s, wave_tree(c),
                     kq, 2.2f, Bf.radius.p);
}

template <bool EMIT>
void launch_gather(hipStream_t s, Context &c, CatalogBuffers &Bf, uint32_t cnt) {
  hipLaunchKernelGGL((k_gather<EMIT>), dim3(blocks_for(cnt, kGatherBlock / 64)), dim3(kGatherBlock), 0, s,
                     wave_tree(c), c.leaf_pos.p, Bf.anchors.p, cnt, Bf.radius.p, Bf.gcount.p, Bf.goff.p, Bf.glist.p);
}

void supports_device(Context &c, int k_max, std::vector<EventRec> &events,
                     std::vector<FallbackRec> &fbs, std::vector<uint32_t> &fb_region,
                     mhgp_catalog_info *info) {
  const int64_t n = c.n;
  if (!c.catalog) c.catalog = std::make_unique<CatalogBuffers>();
  CatalogBuffers &B = *c.catalog;
  hipStream_t s = c.stream;
  const int64_t keff = std::min<int64_t>(k_max, n);
  const int smax = (int)std::min<int64_t>(keff + 1, n);
  B.k_max = k_max;
  B.s_max = smax;
  info->s_max = smax;
  if (n < 2 || smax < 2) {
    B.count = 0;  // no support of two or more points: an empty catalogue
    return;
  }
  if (smax > 11) throw std::invalid_argument("k_max must lie in 1..10");
  B.radius.ensure(n);
  B.gcount.ensure(n);
  B.goff.ensure(n);
  B.region.ensure(n);
  B.lists.ensure((size_t)kLists * n);
  B.counters.ensure(kCounters);
  B.anchors.ensure(n);
  if (B.cells.cap < 8 * kCells) {
    auto cells = make_cells();
    B.cells.ensure(8 * kCells);
    copy_wait(B.cells.p, cells.data(), cells.size() * 8, hipMemcpyHostToDevice, s);
    const std::vector<float> cf = make_cells_f(cells);
    B.cellf.ensure(8 * kCells);
    copy_wait(B.cellf.p, cf.data(), cf.size() * 4, hipMemcpyHostToDevice, s);
    B.strips.ensure(8 * kStrips);
    hipLaunchKernelGGL(k_strips, dim3(kStrips), dim3(kCells), 0, s, B.cells.p, B.strips.p);
    MHGP_LAUNCH_CHECK();
  }
  // Test hook (MHGP_TEST_ANCHOR_PATH): "region" sends every anchor through
  // the big path's probe and LDS region kernels, "slabs" through the
  // global-memory kernel, so that small clouds check those paths against the
  // exhaustive oracle.  Unset, the anchors take their normal tiers.
  int force_path = 0;
  if (const char *tp = std::getenv("MHGP_TEST_ANCHOR_PATH")) {
    if (std::strcmp(tp, "region") == 0) force_path = 1;
    else if (std::strcmp(tp, "slabs") == 0) force_path = 2;
  }
  // initial gather radius: twice the distance to the min(32, n-1)-th neighbour
  const int kq = (int)std::min<int64_t>(32, n - 1);
  StageTimer tm(s);
  DevBuf<uint64_t> &total = B.total;
  total.ensure(1);
  B.glist.ensure(1);
  launch_radius(s, c, kq, B);
  MHGP_LAUNCH_CHECK();
  double bounds[6];
  copy_wait(bounds, c.bounds.p, sizeof(bounds), hipMemcpyDeviceToHost, s);
  // under a capacity the slabs and rescans are given back when the call ends:
  // what they took is the next stage's room
  const bool bounded = c.capacity_bytes > 0;
  auto give_back = [&] {
    if (!bounded) return;
    B.scratch.release();
    B.rescans.release();
  };
  give_back();  // of a call that failed
  CatalogueQueues cap = bounded ? first_queues_bounded(n, smax) : first_queues(n, smax);
  // bytes that queues of these capacities take beyond those that are held
  auto more = [&](const CatalogueQueues &q) {
    auto grown = [](uint64_t want, uint64_t have, uint64_t bytes) { return want > have ? want * bytes - have * bytes : 0; };
    return (int64_t)(grown(q.events, B.events.cap, sizeof(EventRec)) + grown(q.fallbacks, B.fallbacks.cap, sizeof(FallbackRec)) +
                     grown(q.region_words, B.fb_region.cap, 4) + grown(q.rescans, B.rescans.cap / sizeof(Rescan), sizeof(Rescan)));
  };
  uint64_t ctr[kCounters];
  int64_t widened = 0;
  // The record queues have a fixed capacity per launch; records past it are
  // dropped on the device and counted.  A catalogue that outgrows them runs
  // again with queues sized from the counts (the widened gather radii are
  // kept), unless the device cannot hold them.
  for (int attempt = 0;; ++attempt) {
  if (bounded) {
    // the record queues are the catalogue's large, data-sized allocation
    if (device_bytes(c) + more(cap) > c.capacity_bytes)
      throw CapacityError("the catalogue's record queues (" + std::to_string(cap.events) + " records) exceed the " +
                          "context's device capacity of " + std::to_string(c.capacity_bytes) + " bytes");
  }
  B.events.ensure(cap.events);
  B.fallbacks.ensure(cap.fallbacks);
  B.fb_region.ensure(cap.region_words);
  B.rescans.ensure(cap.rescans * sizeof(Rescan));
  MHGP_HIP(hipMemsetAsync(B.counters.p, 0, kCounters * 8, s));
  widened = 0;
  Params P{};
  P.X = c.X.p; P.Y = c.Y.p; P.Z = c.Z.p;
  P.gcount = B.gcount.p; P.goff = B.goff.p; P.radius = B.radius.p;
  P.cells = B.cells.p;
  P.cellf = B.cellf.p;
  P.strips = B.strips.p;
  for (int a = 0; a < 3; ++a) { P.blo[a] = bounds[a]; P.bhi[a] = bounds[3 + a]; }
  P.s_max = smax;
  P.region = B.region.p;
  P.lists = B.lists.p;
  P.list_cap = (uint32_t)n;
  P.events = B.events.p; P.event_cap = cap.events;
  P.fallbacks = B.fallbacks.p; P.fallback_cap = cap.fallbacks;
  P.fb_region = B.fb_region.p; P.fb_region_cap = cap.region_words;
  P.rescans = reinterpret_cast<Rescan *>(B.rescans.p); P.rescan_cap = cap.rescans;
  P.counters = (unsigned long long *)B.counters.p;
  P.count_flops = c.count_flops ? 1 : 0;
  P.region_limit = std::min<uint32_t>(c.region_limit, kBigRegionMax);
  auto list = [&](int l) { return B.lists.p + (size_t)l * n; };
  auto read_counters = [&] { copy_wait(ctr, B.counters.p, sizeof ctr, hipMemcpyDeviceToHost, s); };
  // clears the lengths of lists [first, last)
  auto clear_lists = [&](int first, int last) {
    MHGP_HIP(hipMemsetAsync(B.counters.p + kListCount + first, 0, (last - first) * 8, s));
  };
  // enumerates the regions of one probe launch (ctr holds its list lengths),
  // the largest first and each size on a stream of its own: one after the
  // other each size left the chip to its last workgroups before the next
  // began (2 003-point mixture, 13 launches of 3 to 1 214 anchors: catalogue
  // 39.1 -> 33.7 ms; 50 000-point lattice's pipeline 103.4 -> 101.5 ms)
  auto enumerate = [&](const Params &Q) {
    int sizes[kLists], count = 0;
    for (int l = L_LARGE; l >= L_TINY; --l)
      if (ctr[kListCount + l]) sizes[count++] = l;
    const int sides = std::min(count - 1, SideStreams::kCount);
    if (sides > 0) B.sides.fork(s, sides);
    for (int i = 0; i < count; ++i) {
      const int l = sizes[i];
      const uint32_t m = (uint32_t)ctr[kListCount + l];
      const dim3 grid(m, std::clamp<uint32_t>(kRegionParts / m, 1, 64));
      hipStream_t t = i == 0 ? s : B.sides.stream[(i - 1) % SideStreams::kCount];
      if (l == L_LARGE)
        hipLaunchKernelGGL((k_anchor_region<kRegionCapHuge, 8, 2>), grid, dim3(512), 0, t, Q, list(l));
      else if (l == L_MID)
        hipLaunchKernelGGL((k_anchor_region<kRegionCapWide, 4, 2>), grid, dim3(256), 0, t, Q, list(l));
      else if (l == L_TINY)
        hipLaunchKernelGGL((k_anchor_region<kRegionCapTiny, 1, 3>), grid, dim3(64), 0, t, Q, list(l));
      else if (l == L_LITTLE)
        hipLaunchKernelGGL((k_anchor_region<kRegionCapLittle, 2, 3>), grid, dim3(128), 0, t, Q, list(l));
      else
        hipLaunchKernelGGL((k_anchor_region<kRegionCap, 4, 3>), grid, dim3(256), 0, t, Q, list(l));
      MHGP_LAUNCH_CHECK();
    }
    if (sides > 0) B.sides.join(s, sides);
  };
  // the sides that a launch's enumeration left, before its slabs are reused
  auto settle = [&](const Params &Q) {
    hipLaunchKernelGGL(k_rescan, dim3(kRescanBlocks), dim3(64), 0, s, Q);
    hipLaunchKernelGGL(k_rescans_done, dim3(1), dim3(1), 0, s, Q);
    MHGP_LAUNCH_CHECK();
  };
  // scratch for slabs: 8 GiB, 1 GiB in a context with a device capacity; and
  // at most a quarter of the device memory still free (other contexts on the
  // device keep theirs), but never below 1 GiB
  auto slab_budget = [&]() -> uint64_t {
    if (c.capacity_bytes > 0) return 1ull << 30;
    size_t free_b = 0, total_b = 0;
    MHGP_HIP(hipMemGetInfo(&free_b, &total_b));
    return std::max<uint64_t>(1ull << 30, std::min<uint64_t>(8ull << 30, free_b / 4));
  };
  // Probes `count` anchors of the device list in chunks whose slabs fit 2 GiB,
  // each chunk enumerated before the next one takes its slabs.  Slabs beyond
  // those held grow into at most a quarter of the device memory still free
  // (other contexts on the device keep theirs), under a capacity a quarter of
  // what that leaves; at least probe_slabs_least.
  auto probe_lds = [&](const uint32_t *anchors, uint32_t count, uint32_t g) {
    const uint64_t slab = probe_slab_doubles(g), held = B.scratch.bytes();
    uint32_t per = 0;
    auto chunks_of = [&](uint64_t budget) {
      const uint32_t most = (uint32_t)std::clamp<uint64_t>(budget / (slab * 8), 1, count);
      const uint32_t chunks = (count + most - 1) / most;
      per = (count + chunks - 1) / chunks;
    };
    chunks_of(kProbeSlabs);
    if (per * slab * 8 > held) {
      size_t free_b = 0, total_b = 0;
      if (!bounded) MHGP_HIP(hipMemGetInfo(&free_b, &total_b));
      chunks_of(bounded ? probe_slab_budget(c.capacity_bytes - device_bytes(c), held, probe_slabs_least(n), kProbeSlabs / 2)
                        : probe_slab_budget((int64_t)free_b, held, probe_slabs_least(n), kProbeSlabs));
    }
    B.scratch.ensure(slab * per);
    for (uint32_t a0 = 0; a0 < count; a0 += per) {
      Params Q = P;
      Q.anchors = anchors + a0;
      Q.anchor_count = std::min(per, count - a0);
      Q.gcap = g;
      Q.scratch = B.scratch.p;
      Q.slab_doubles = slab;
      Q.ascending = 1;
      if (Q.anchor_count >= kSmallRegionLaunch) {
        Q.one_wave = kRegionCapTiny;
        Q.two_waves = kRegionCapLittle;
      }
      clear_lists(L_TINY, kLists);
      const dim3 grid(Q.anchor_count), block(kProbeBlock);
      if (g == kGatherCap)
        hipLaunchKernelGGL((k_anchor_probe<kGatherCap, false>), grid, block, 0, s, Q);
      else if (g == kGatherCapWide)
        hipLaunchKernelGGL((k_anchor_probe<kGatherCapWide, false>), grid, block, 0, s, Q);
      else
        hipLaunchKernelGGL((k_anchor_probe<kGatherCapSlab, true>), grid, block, 0, s, Q);
      MHGP_LAUNCH_CHECK();
      read_counters();
      enumerate(Q);
      settle(Q);
    }
  };
  // anchors in Morton order: neighbouring workgroups share cache lines
  MHGP_HIP(hipMemcpyAsync(B.anchors.p, c.leaf_id.p, n * 4, hipMemcpyDeviceToDevice, s));
  uint32_t cnt = (uint32_t)n;
  for (int iter = 0; cnt > 0; ++iter) {
    if (iter > 24) throw CapacityError("anchor gather radii did not converge");
    launch_gather<false>(s, c, B, cnt);
    hipLaunchKernelGGL(k_scan_offsets, dim3(1), dim3(1024), 0, s, B.anchors.p, cnt, B.gcount.p,
                       B.goff.p, total.p);
    uint64_t tot = 0;
    copy_wait(&tot, total.p, 8, hipMemcpyDeviceToHost, s);
    B.glist.ensure(tot + 1);
    launch_gather<true>(s, c, B, cnt);
    P.glist = B.glist.p;
    if (bounded && iter == 0) {
      // an eighth of what is left for rescans, up to an unbounded context's;
      // the list is still empty
      const uint64_t left = (uint64_t)std::max<int64_t>(0, c.capacity_bytes - device_bytes(c));
      const uint64_t held = B.rescans.cap / sizeof(Rescan), full = first_queues(n, smax).rescans;
      if (held < full && left / 8 >= sizeof(Rescan)) B.rescans.ensure(std::min<uint64_t>(full, held + left / 8 / sizeof(Rescan)) * sizeof(Rescan));
      cap.rescans = std::max(cap.rescans, B.rescans.cap / sizeof(Rescan));
      P.rescans = reinterpret_cast<Rescan *>(B.rescans.p);
      P.rescan_cap = cap.rescans;
    }
    tm.mark("catalogue gather");
    uint64_t before[kCounters];
    copy_wait(before, B.counters.p, sizeof before, hipMemcpyDeviceToHost, s);
    clear_lists(0, kLists);
    c.anchor_clock.start(s);
    if (!force_path) {
      probe_lds(B.anchors.p, cnt, kGatherCap);
      const uint32_t wide = (uint32_t)ctr[kListCount + L_WIDE], wider = (uint32_t)ctr[kListCount + L_WIDER];
      if (wide) probe_lds(list(L_WIDE), wide, kGatherCapWide);
      if (wider) probe_lds(list(L_WIDER), wider, kGatherCapSlab);
      if (tm.on && (wide || wider)) std::fprintf(stderr, "[mhgp] wide anchors: %u, wider: %u\n", wide, wider);
    }
    c.anchor_clock.stop(s);
    tm.mark("catalogue anchors");
    // gathers beyond LDS: probed on slabs in chunks of anchors of similar
    // gather size (ascending), each chunk's slabs sized by its own largest
    // gather within the scratch budget, so that a few anchors that gather most
    // of the cloud do not shrink every launch to a handful of workgroups
    std::vector<uint32_t> big(force_path ? cnt : (uint32_t)ctr[kListCount + L_BIG]);
    if (!big.empty()) {
      copy_wait(big.data(), force_path ? B.anchors.p : list(L_BIG), big.size() * 4, hipMemcpyDeviceToHost, s);
      std::vector<uint32_t> gc(n);
      copy_wait(gc.data(), B.gcount.p, n * 4, hipMemcpyDeviceToHost, s);
      const uint64_t kScratchBudget = slab_budget();
      auto slab_of = [](uint32_t g) { return big_fc_offset(g) + 2ull * g; };
      // the probed regions beyond LDS come back in `slabs`
      auto launch_big = [&](std::vector<uint32_t> todo, int probe, std::vector<uint32_t> &slabs) {
        std::sort(todo.begin(), todo.end(),
                  [&](uint32_t x, uint32_t y) { return gc[x] < gc[y] || (gc[x] == gc[y] && x < y); });
        const size_t lc = todo.size();
        std::vector<std::pair<size_t, uint32_t>> chunks;  // (end, gather cap)
        uint64_t scratch = 0;
        for (size_t b0 = 0; b0 < lc;) {
          size_t b1 = b0;
          uint32_t g = 64;
          while (b1 < lc) {
            const uint32_t gn = std::max<uint32_t>(64, gc[todo[b1]]);
            if (b1 > b0 && slab_of(gn) * 8 * (b1 - b0 + 1) > kScratchBudget) break;
            g = gn;
            ++b1;
          }
          chunks.push_back({b1, g});
          scratch = std::max<uint64_t>(scratch, slab_of(g) * (b1 - b0));
          b0 = b1;
        }
        B.scratch.ensure(scratch);
        B.big.ensure(lc);
        MHGP_HIP(hipMemcpyAsync(B.big.p, todo.data(), lc * 4, hipMemcpyHostToDevice, s));
        size_t b0 = 0;
        for (const auto &ch : chunks) {
          const uint32_t bn = (uint32_t)(ch.first - b0), g = ch.second;
          Params Q = P;
          Q.anchors = B.big.p + b0; Q.anchor_count = bn; Q.probe = probe;
          Q.scratch = B.scratch.p; Q.slab_doubles = slab_of(g); Q.gcap = g;
          if (probe) clear_lists(L_TINY, kLists);
          hipLaunchKernelGGL(k_anchor_big, dim3(bn), dim3(kBlock), 0, s, Q);
          MHGP_LAUNCH_CHECK();
          if (!probe) settle(Q);
          if (probe) {
            read_counters();
            // test hook: every region through the slab enumeration
            if (force_path != 2) {
              enumerate(Q);
              settle(Q);
            }
            for (int l = force_path == 2 ? L_TINY : L_SLAB; l <= L_SLAB; ++l) {
              std::vector<uint32_t> at(ctr[kListCount + l]);
              if (!at.empty()) copy_wait(at.data(), list(l), at.size() * 4, hipMemcpyDeviceToHost, s);
              for (uint32_t i : at) {
                if (i >= bn) throw std::runtime_error("malformed region list from the device");
                slabs.push_back(todo[b0 + i]);
              }
            }
          }
          b0 = ch.first;
        }
      };
      // first the regions only, so that one the path cannot take is refused
      // before any long launch
      std::vector<uint32_t> slabs, none;
      launch_big(big, 1, slabs);
      tm.mark("catalogue big probe (+ LDS regions)");
      if (!slabs.empty()) launch_big(slabs, 0, none);
      tm.mark("catalogue big on slabs");
      if (tm.on)
        std::fprintf(stderr, "[mhgp] big anchors: %zu, %zu on slabs\n", big.size(), slabs.size());
    }
    read_counters();
    if (!force_path) {
      const uint64_t ev = ctr[0] - before[0];
      c.stats.anchor_ms += c.anchor_clock.ms();
      c.stats.anchor_launches++;
      c.stats.gathered_points += (int64_t)tot;
      c.stats.events += (int64_t)ev;
      // algorithmic bytes: every gathered neighbour read once (id + FP64 xyz),
      // every record written once
      c.stats.anchor_bytes += (int64_t)tot * 28 + (int64_t)ev * (int64_t)sizeof(EventRec);
      // FP64 and FP32 operations of the certified predicates the launches evaluated
      c.stats.anchor_flops += (int64_t)(ctr[5] - before[5]);
      c.stats.anchor_flops32 += (int64_t)(ctr[6] - before[6]);
    }
    // the widened gathers are the next pass
    cnt = (uint32_t)ctr[kListCount + L_WIDEN];
    widened += cnt;
    if (cnt) MHGP_HIP(hipMemcpyAsync(B.anchors.p, list(L_WIDEN), cnt * 4, hipMemcpyDeviceToDevice, s));
  }
  tm.mark("catalogue big anchors");
  read_counters();
  if (tm.on) std::fprintf(stderr, "[mhgp] sides left to the rescans, most in a launch: %llu\n", (unsigned long long)ctr[kRescanMost]);
  if (ctr[0] <= cap.events && ctr[1] <= cap.fallbacks && ctr[2] <= cap.region_words && ctr[kRescanMost] <= cap.rescans) break;
  // a launch that ran out of rescans has also counted too few records
  if (attempt >= 3) throw CapacityError("catalogue record queues did not settle after regrowth");
  auto needed = [&](int at) { return ctr[at] + ctr[at] / 8; };
  const CatalogueQueues need{needed(0), needed(1), needed(2), needed(kRescanMost)};
  cap = {std::max(cap.events, need.events), std::max(cap.fallbacks, need.fallbacks),
         std::max(cap.region_words, need.region_words), std::max(cap.rescans, need.rescans)};
  if (bounded && device_bytes(c) + more(cap) > c.capacity_bytes) {
    // no room for the first capacities beside the grown ones: what was counted
    cap = {std::max<uint64_t>(need.events, 1024), std::max<uint64_t>(need.fallbacks, 1024),
           std::max<uint64_t>(need.region_words, 1024), std::max<uint64_t>(need.rescans, 1024)};
    B.events.release();
    B.fallbacks.release();
    B.fb_region.release();
    B.rescans.release();
  }
  size_t free_b = 0, total_b = 0;
  MHGP_HIP(hipMemGetInfo(&free_b, &total_b));
  if ((uint64_t)more(cap) > free_b / 10 * 9)
    throw CapacityError("the catalogue needs " + std::to_string(ctr[0]) + " record slots, more than the device can hold");
  // grown buffers start empty: release before the larger allocation
  if (B.events.cap < cap.events) B.events.release();
  if (B.fallbacks.cap < cap.fallbacks) B.fallbacks.release();
  if (B.fb_region.cap < cap.region_words) B.fb_region.release();
  if (B.rescans.cap < cap.rescans * sizeof(Rescan)) B.rescans.release();
  }
  // records stay on the device; only the host's share of the work moves
  (void)events;
  B.count = (int64_t)ctr[0];
  fbs.resize(ctr[1]);
  fb_region.resize(ctr[2]);
  if (ctr[1]) copy_wait(fbs.data(), B.fallbacks.p, ctr[1] * sizeof(FallbackRec), hipMemcpyDeviceToHost, s);
  if (ctr[2]) copy_wait(fb_region.data(), B.fb_region.p, ctr[2] * 4, hipMemcpyDeviceToHost, s);
  give_back();
  tm.mark("catalogue download");
  info->candidate_count = (int64_t)ctr[3];
  info->anchors_widened = widened;
  info->anchors_open = (int64_t)ctr[kOpenCount];
  info->largest_open_region = (int64_t)ctr[kOpenLargest];
  info->status = ctr[kOpenCount] ? 1 : 0;
}

}  // namespace mhgp
