// Exact Euclidean minimum spanning tree by LBVH Borůvka on gfx950.
//
// Reference: morsehgp3d/src/cpu/hierarchy/boruvka.cpp:893 (build_exact_lbvh_boruvka):
// frozen component labels per round, subtrees uniform in the source's own
// component are skipped, and every component takes its lightest outgoing edge
// under kappa = (d^2, min id, max id).  Under kappa the minimum spanning tree
// is unique, so the output equals the complete-graph Kruskal anchor
// (emst.cpp:326).
//
// Points and components are numbered by Morton position (a component by one
// of its points).  A round: labels of the wave tree's groups -> per-point
// search, one wave per point -> per-component minima -> hooking with 2-cycle
// breaking -> roots.  A point's nearest external point stays its nearest
// while it is external (the external set only shrinks), so a search is run
// again only for points whose last result was absorbed or tied (what tied with
// it may have been absorbed), and not at all when that result's distance, a
// lower bound ever after, exceeds what another point of the component already
// offers.  FP64 distances that are not provably
// ordered (near ties that are not both exact) are flagged and settled on the
// host with exact integer arithmetic.
#include <algorithm>

#include "pipeline.hpp"
#include "stages.hpp"
#include "timing.hpp"
#include "traverse.hpp"
#include "wave_tree.hpp"

namespace mhgp {

namespace {

__device__ inline uint64_t edge_key(uint32_t a, uint32_t b) {
  uint32_t lo = a < b ? a : b, hi = a < b ? b : a;
  return ((uint64_t)lo << 32) | hi;
}

// counters: [0] edges, [1] components, [2] ambiguous components
struct Rounds {
  uint32_t *label;                  // component of each position
  uint32_t *glabel;                 // uniform component of each wave-tree group (levels 0, 1, 2), or kInvalid
  uint32_t *best_p;                 // nearest external position, kInvalid: none that counts
  double *best_d;                   // its squared distance; without one, a lower bound of it
  uint8_t *best_flag;               // 1: near tie, 4: the distance is not exact
  uint64_t *comp_d, *comp_e;        // per component: least distance (bits), least edge key at it
  uint32_t *comp_amb, *comp_cw, *comp_ce;  // tie flag; entries in the rounding window, exact equal ones
  uint32_t *hook, *root;
  uint32_t *edges, *counters;
};

__device__ inline double as_double(uint64_t b) { return __longlong_as_double((long long)b); }

__device__ inline void reset_component(const Rounds &R, int64_t p) {
  R.comp_d[p] = 0x7ff0000000000000ull;  // +infinity
  R.comp_e[p] = ~0ull;
  R.comp_amb[p] = 0;
  R.comp_cw[p] = 0;
  R.comp_ce[p] = 0;
}

__global__ void k_start(int64_t n, Rounds R) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p < 3) R.counters[p] = 0;
  if (p >= n) return;
  R.label[p] = (uint32_t)p;
  R.best_p[p] = kInvalid;
  R.best_d[p] = 0.0;
  R.best_flag[p] = 0;
  reset_component(R, p);
}

__device__ inline uint32_t wave_uniform(uint32_t v, bool valid) {
  const uint64_t m = __ballot(valid);
  if (!m) return kInvalid;
  const uint32_t f = lane_u32(v, __builtin_amdgcn_readfirstlane(__ffsll((long long)m) - 1));
  return __ballot(valid && v != f) ? kInvalid : f;
}

// Component shared by all leaves of each wave-tree group, one workgroup per
// level-1 group (as the boxes are made); thread per position: the results of
// the last round that still hold offer their distance to their component.
constexpr int kLabelBlock = 1024;
__global__ void __launch_bounds__(kLabelBlock) k_group_labels(WaveTree T, Rounds R) {
  __shared__ uint32_t lab[64];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  for (uint32_t j = wave; j < 64; j += kLabelBlock / 64) {
    const uint32_t g = blockIdx.x * 64 + j, p = g * 64 + lane;
    const bool valid = g < T.c0 && p < T.n;
    const uint32_t l = valid ? R.label[p] : kInvalid;
    const uint32_t f = wave_uniform(l, valid);
    if (lane == 0) {
      lab[j] = f;
      if (g < T.c0) R.glabel[g] = f;
    }
    if (!valid) continue;
    const uint32_t b = R.best_p[p];
    if (b == kInvalid) continue;
    const bool external = R.label[b] != l;
    if (external) {
      const uint64_t d = dbits(R.best_d[p]);
      if (d < R.comp_d[l]) atomicMin((unsigned long long *)&R.comp_d[l], (unsigned long long)d);
    }
    // absorbed, or tied in its round: searched again; its distance stays a lower bound
    if (!external || (R.best_flag[p] & 1)) R.best_p[p] = kInvalid;
  }
  __syncthreads();
  if (wave == 0) {
    const uint32_t f = wave_uniform(lab[lane], blockIdx.x * 64 + lane < T.c0);
    if (lane == 0) R.glabel[T.c0 + blockIdx.x] = f;
  }
}

__global__ void __launch_bounds__(64) k_top_labels(WaveTree T, Rounds R) {
  const uint32_t i = blockIdx.x * 64 + threadIdx.x;
  const uint32_t f = wave_uniform(i < T.c1 ? R.glabel[T.c0 + i] : kInvalid, i < T.c1);
  if (threadIdx.x == 0) R.glabel[T.c0 + T.c1 + blockIdx.x] = f;
}

// Lightest external edge under kappa of every point whose last one is gone:
// each lane keeps its own best over the groups, the wave combines them at the
// end.  The component's best offer bounds the search from the start: a result
// counts within the offer's rounding window (limit).  The search itself sees
// points up to the window of any result that counts, because a result may be
// kept for later rounds, where that offer is gone and nothing else shows that
// another point is as near.
constexpr int kSearchBlock = 256;  // four waves, four points
__global__ void __launch_bounds__(kSearchBlock) k_search(WaveTree T, Rounds R) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t p = blockIdx.x * (kSearchBlock / 64) + (threadIdx.x >> 6);
  if (p >= T.n || R.best_p[p] != kInvalid) return;
  const uint32_t lu = R.label[p];
  const double offer = as_double(R.comp_d[lu]);
  const double limit = offer * (1.0 + kSlack) + kSlackAbs;
  if (R.best_d[p] > limit) return;
  const uint32_t u = T.leaf_id[p];
  const double q[3] = {T.LX[p], T.LY[p], T.LZ[p]};
  const WaveQuery Q(q[0], q[1], q[2]);
  double bd = INFINITY;
  uint32_t bp = kInvalid, bv = kInvalid;
  bool bx = true, near_tie = false;
  double bound = offer * (1.0 + 4.0 * kSlack) + 4.0 * kSlackAbs;  // >= limit * (1 + kSlack) + kSlackAbs
  double most = wave_bound(bound);
  auto group = [&](uint32_t g) {
    const uint32_t lp = g * 64 + lane, at = min(lp, T.n - 1);
    const bool valid = lp < T.n && R.label[at] != lu;
    if (!__ballot(valid)) return;
    bool ex;
    const double d = d2_flag(q, T.LX[at], T.LY[at], T.LZ[at], ex);
    const bool in = valid && d <= bound;
    if (!__ballot(in)) return;
    if (in && d <= bd * (1.0 + kSlack) + kSlackAbs) {
      const uint32_t v = T.leaf_id[at];
      const bool both = ex && bx;
      if (!both && bd < INFINITY && fabs(d - bd) <= kSlack * bd + kSlackAbs) near_tie = true;  // order not provable
      if (d < bd || (d == bd && edge_key(u, v) < edge_key(u, bv))) {
        if (bd < INFINITY && !(fabs(d - bd) <= kSlack * bd + kSlackAbs)) near_tie = false;
        bd = d;
        bp = lp;
        bv = v;
        bx = ex;
      }
    }
    double m = bd;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmin(m, __shfl_xor(m, o));
    bound = fmin(bound, m * (1.0 + kSlack) + kSlackAbs);
    most = wave_bound(bound);
  };
  const uint32_t own = p >> 6;
  if (R.glabel[own] == kInvalid) group(own);
  const uint32_t *gl = R.glabel;
  wave_tree_visit(
      T, Q, most,
      [&](int level, uint32_t i) { return gl[(level == 0 ? 0u : level == 1 ? T.c0 : T.c0 + T.c1) + i] != lu; },
      [&](uint32_t g) {
        if (g != own) group(g);
      });
  double m = bd;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = fmin(m, __shfl_xor(m, o));
  if (!(m <= limit) || m == INFINITY) {
    // nothing the component can use: every external point lies beyond the offer
    if (lane == 0) R.best_d[p] = fmax(R.best_d[p], offer);
    return;
  }
  // lanes within rounding of the least distance: proven when alone or all exact
  const bool win = bd <= m * (1.0 + kSlack) + kSlackAbs;
  const uint64_t w = __ballot(win);
  const bool exact = !__ballot(win && !bx);
  const bool tie = __ballot(win && near_tie) != 0 || (!exact && __popcll(w) > 1);
  uint64_t key = win && bd == m ? edge_key(u, bv) : ~0ull;
  uint64_t least = key;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) least = min(least, (uint64_t)__shfl_xor((unsigned long long)least, o));
  if (key == least && key != ~0ull) {  // one lane: edge keys are distinct
    R.best_p[p] = bp;
    R.best_d[p] = m;
    R.best_flag[p] = (tie ? 1 : 0) | (bx ? 0 : 4);
    const uint64_t b = dbits(m);
    if (b < R.comp_d[lu]) atomicMin((unsigned long long *)&R.comp_d[lu], (unsigned long long)b);
  }
}

// Entries within rounding of a component's FP64 minimum decide whether the
// winner is proven: a single entry in the window is the exact minimum; several
// entries are settled on the device only when all are exact and equal (ties
// then break on the edge key).  Otherwise the component goes to the host.
__global__ void k_comp_tie(WaveTree T, Rounds R) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= T.n || R.best_p[p] == kInvalid) return;
  const uint32_t l = R.label[p];
  const uint64_t mb = R.comp_d[l];
  const double m = as_double(mb), d = R.best_d[p];
  if (d - m > kSlack * m + kSlackAbs) return;
  atomicAdd(&R.comp_cw[l], 1u);
  if (R.best_flag[p] & 1) atomicOr(&R.comp_amb[l], 1u);
  if (dbits(d) == mb) {
    atomicMin((unsigned long long *)&R.comp_e[l],
              (unsigned long long)edge_key(T.leaf_id[p], T.leaf_id[R.best_p[p]]));
    if (!(R.best_flag[p] & 4)) atomicAdd(&R.comp_ce[l], 1u);
  }
}

__global__ void k_comp_decide(int64_t n, Rounds R) {
  const int64_t l = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (l == 0) R.counters[1] = 0;
  if (l >= n || R.label[l] != (uint32_t)l) return;
  if (R.comp_cw[l] >= 2 && R.comp_cw[l] != R.comp_ce[l]) R.comp_amb[l] |= 8u;
  if (R.comp_amb[l]) atomicAdd(&R.counters[2], 1u);
}

// Every component hooks to the one across its winning edge and emits that
// edge; of two that chose the same edge (keys are unique) the smaller stays a
// root and emits it.  Nothing happens while ambiguous components wait for
// the host (counters[2]).
__global__ void k_hook(int64_t n, const uint32_t *__restrict__ leaf_pos, Rounds R) {
  const int64_t l = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (l >= n || R.counters[2] || R.label[l] != (uint32_t)l) return;
  const uint64_t e = R.comp_e[l];
  if (e == ~0ull) {
    R.hook[l] = (uint32_t)l;
    return;
  }
  const uint32_t a = R.label[leaf_pos[(uint32_t)(e >> 32)]], b = R.label[leaf_pos[(uint32_t)e]];
  const uint32_t other = a == (uint32_t)l ? b : a;
  const bool mutual = R.comp_e[other] == e;
  R.hook[l] = mutual && (uint32_t)l < other ? (uint32_t)l : other;
  if (mutual && (uint32_t)l > other) return;
  const uint32_t slot = atomicAdd(&R.counters[0], 1u);
  if (slot >= (uint32_t)n) return;
  R.edges[2 * slot] = (uint32_t)(e >> 32);
  R.edges[2 * slot + 1] = (uint32_t)e;
}

// Root of every component in the hook forest, by path halving: concurrent
// threads only ever store an ancestor of a component as its hook.
__global__ void k_roots(int64_t n, Rounds R) {
  const int64_t l = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (l >= n || R.counters[2] || R.label[l] != (uint32_t)l) return;
  volatile uint32_t *hook = R.hook;
  uint32_t x = (uint32_t)l;
  for (int64_t step = 0; step < n; ++step) {
    const uint32_t h = hook[x];
    if (h == x) break;
    const uint32_t g = hook[h];
    if (g == h) {
      x = h;
      break;
    }
    hook[x] = g;
    x = g;
  }
  R.root[l] = x;
  if (x == (uint32_t)l) atomicAdd(&R.counters[1], 1u);
}

// New labels, and the component arrays cleared for the next round.
__global__ void k_relabel(int64_t n, Rounds R) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n || R.counters[2]) return;
  R.label[p] = R.root[R.label[p]];
  reset_component(R, p);
}

}  // namespace

// Host exact settlement of the lightest external edge of one point.
static uint64_t exact_best_edge(Context &c, const std::vector<uint32_t> &label, int64_t u,
                                const ExactCloud &ex, const std::vector<double> &xyz) {
  const int64_t n = c.n;
  double bd = INFINITY;
  for (int64_t v = 0; v < n; ++v) {
    if (label[v] == label[u]) continue;
    double s = 0;
    for (int a = 0; a < 3; ++a) { double t = xyz[3 * v + a] - xyz[3 * u + a]; s += t * t; }
    bd = std::min(bd, s);
  }
  int64_t best = -1;
  for (int64_t v = 0; v < n; ++v) {
    if (label[v] == label[u]) continue;
    double s = 0;
    for (int a = 0; a < 3; ++a) { double t = xyz[3 * v + a] - xyz[3 * u + a]; s += t * t; }
    if (s > bd * (1.0 + 1e-9)) continue;
    if (best < 0) { best = v; continue; }
    int cmp = ex.cmp_dist(u, v, best);
    uint64_t kv = ((uint64_t)std::min<int64_t>(u, v) << 32) | (uint64_t)std::max<int64_t>(u, v);
    uint64_t kb = ((uint64_t)std::min<int64_t>(u, best) << 32) | (uint64_t)std::max<int64_t>(u, best);
    if (cmp < 0 || (cmp == 0 && kv < kb)) best = v;
  }
  return ((uint64_t)std::min<int64_t>(u, best) << 32) | (uint64_t)std::max<int64_t>(u, best);
}

// Sort keys of the forest's edges: the bits of the FP64 squared length (a
// non-negative double orders like its bit pattern) with the edge index.
__global__ void k_kappa_keys(int64_t m, const uint32_t *__restrict__ edges, const double *__restrict__ X,
                             const double *__restrict__ Y, const double *__restrict__ Z, uint64_t *key,
                             uint32_t *idx) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m) return;
  const uint32_t a = edges[2 * i], b = edges[2 * i + 1];
  const double dx = X[a] - X[b], dy = Y[a] - Y[b], dz = Z[a] - Z[b];
  key[i] = (uint64_t)__double_as_longlong(dx * dx + dy * dy + dz * dz);
  idx[i] = (uint32_t)i;
}

void emst_host(Context &c, uint32_t *edges_out) {
  const int64_t n = c.n;
  if (n <= 1) return;
  if (!c.emst) c.emst = std::make_unique<EmstBuffers>();
  EmstBuffers &B = *c.emst;
  hipStream_t s = c.stream;
  const int T = 256;
  const dim3 G(blocks_for(n, T)), B256(T);
  const WaveTree W = wave_tree(c);
  B.label.ensure(n);
  B.node_label.ensure((size_t)W.c0 + W.c1 + W.c2);
  B.best_v.ensure(n);
  B.best_d.ensure(n);
  B.best_flag.ensure(n);
  B.comp_d.ensure(n);
  B.comp_e.ensure(n);
  B.comp_amb.ensure(n);
  B.comp_cw.ensure(n);
  B.comp_ce.ensure(n);
  B.edges.ensure(2 * n);
  B.counters.ensure(4);
  B.hook.ensure(n);
  B.next_label.ensure(n);
  const Rounds R{B.label.p,  B.node_label.p, B.best_v.p,  B.best_d.p,  B.best_flag.p,  B.comp_d.p, B.comp_e.p,
                 B.comp_amb.p, B.comp_cw.p,    B.comp_ce.p, B.hook.p,    B.next_label.p, B.edges.p,  B.counters.p};
  hipLaunchKernelGGL(k_start, G, B256, 0, s, n, R);
  int64_t components = n, settled = 0;
  for (int round = 0; components > 1; ++round) {
    if (round > 64) throw std::runtime_error("Borůvka did not converge");
    hipLaunchKernelGGL(k_group_labels, dim3(W.c1), dim3(kLabelBlock), 0, s, W, R);
    if (W.c2 > 1) hipLaunchKernelGGL(k_top_labels, dim3(W.c2), dim3(64), 0, s, W, R);
    hipLaunchKernelGGL(k_search, dim3(blocks_for(n, kSearchBlock / 64)), dim3(kSearchBlock), 0, s, W, R);
    hipLaunchKernelGGL(k_comp_tie, G, B256, 0, s, W, R);
    hipLaunchKernelGGL(k_comp_decide, G, B256, 0, s, n, R);
    for (;;) {
      hipLaunchKernelGGL(k_hook, G, B256, 0, s, n, c.leaf_pos.p, R);
      hipLaunchKernelGGL(k_roots, G, B256, 0, s, n, R);
      hipLaunchKernelGGL(k_relabel, G, B256, 0, s, n, R);
      MHGP_LAUNCH_CHECK();
      uint32_t cnt[3];
      copy_wait(cnt, B.counters.p, sizeof cnt, hipMemcpyDeviceToHost, s);
      if (cnt[2] == 0) {
        components = cnt[1];
        if (cnt[0] + components != (uint64_t)n) throw std::runtime_error("Borůvka edge count mismatch");
        break;
      }
      // host exact settlement of ambiguous components (rare); the kernels
      // above left the round as it was
      std::vector<uint32_t> at(n), ids(n), amb(n), label(n);
      std::vector<uint64_t> ce(n);
      MHGP_HIP(hipMemcpyAsync(at.data(), B.label.p, n * 4, hipMemcpyDeviceToHost, s));
      MHGP_HIP(hipMemcpyAsync(ids.data(), c.leaf_id.p, n * 4, hipMemcpyDeviceToHost, s));
      MHGP_HIP(hipMemcpyAsync(amb.data(), B.comp_amb.p, n * 4, hipMemcpyDeviceToHost, s));
      copy_wait(ce.data(), B.comp_e.p, n * 8, hipMemcpyDeviceToHost, s);
      for (int64_t p = 0; p < n; ++p) label[ids[p]] = at[p];  // component by PointId
      const ExactCloud &ex = exact_cloud(c);
      const std::vector<double> &xyz = c.host->xyz;
      for (int64_t l = 0; l < n; ++l) {
        if (!amb[l]) continue;
        settled++;
        uint64_t best = ~0ull;
        for (int64_t u = 0; u < n; ++u) {
          if (label[u] != (uint32_t)l) continue;
          uint64_t e = exact_best_edge(c, label, u, ex, xyz);
          if (best == ~0ull) { best = e; continue; }
          int cmp = compare(ex.sq_dist(e >> 32, (uint32_t)e), ex.sq_dist(best >> 32, (uint32_t)best));
          if (cmp < 0 || (cmp == 0 && e < best)) best = e;
        }
        ce[l] = best;
      }
      copy_wait(B.comp_e.p, ce.data(), n * 8, hipMemcpyHostToDevice, s);
      MHGP_HIP(hipMemsetAsync(B.counters.p + 2, 0, sizeof(uint32_t), s));
    }
  }
  StageTimer tm(s);
  if (tm.on) std::fprintf(stderr, "[mhgp] emst components settled on the host: %lld\n", (long long)settled);
  // kappa order: FP64 squared lengths sorted on the device; runs of values
  // within rounding of their neighbours are ordered exactly on the host
  const int64_t m = n - 1;
  B.kappa_key.ensure(m);
  B.kappa_idx.ensure(m);
  hipLaunchKernelGGL(k_kappa_keys, dim3(blocks_for(m, T)), dim3(T), 0, s, m, B.edges.p, c.X.p, c.Y.p, c.Z.p,
                     B.kappa_key.p, B.kappa_idx.p);
  MHGP_LAUNCH_CHECK();
  c.sorter.sort(B.kappa_key.p, B.kappa_idx.p, m, 0, 64, s);
  std::vector<uint32_t> e(2 * m), idx(m);
  std::vector<double> len(m);
  MHGP_HIP(hipMemcpyAsync(e.data(), B.edges.p, e.size() * 4, hipMemcpyDeviceToHost, s));
  MHGP_HIP(hipMemcpyAsync(idx.data(), B.kappa_idx.p, m * 4, hipMemcpyDeviceToHost, s));
  copy_wait(len.data(), B.kappa_key.p, m * 8, hipMemcpyDeviceToHost, s);
  std::vector<std::pair<double, uint64_t>> ord(m);
  for (int64_t i = 0; i < m; ++i) {
    const uint32_t x = e[2 * (size_t)idx[i]], y = e[2 * (size_t)idx[i] + 1];
    ord[i] = {len[i], ((uint64_t)std::min(x, y) << 32) | std::max(x, y)};
  }
  // a run continues while each value is within 1e-12 (relative) of the one
  // before it, so values in different runs differ by far more than the
  // rounding of the FP64 lengths and their FP64 order is the exact one
  for (int64_t i = 0; i + 1 < m; ++i) {
    int64_t j = i;
    while (j + 1 < m && ord[j + 1].first - ord[j].first <= 1e-12 * ord[j + 1].first) j++;
    if (j > i) {
      const ExactCloud &ex = exact_cloud(c);
      std::sort(ord.begin() + i, ord.begin() + j + 1, [&](const auto &x, const auto &y) {
        int cmp = compare(ex.sq_dist(x.second >> 32, (uint32_t)x.second),
                          ex.sq_dist(y.second >> 32, (uint32_t)y.second));
        return cmp != 0 ? cmp < 0 : x.second < y.second;
      });
      i = j;
    }
  }
  tm.mark("emst kappa sort");
  for (int64_t i = 0; i < m; ++i) {
    edges_out[2 * i] = (uint32_t)(ord[i].second >> 32);
    edges_out[2 * i + 1] = (uint32_t)ord[i].second;
  }
}

}  // namespace mhgp
