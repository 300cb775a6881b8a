// k nearest neighbours (up to 63; the public call up to 32) of every data point
// over the wave tree, and top-k partitions of rational points.
//
// Semantics follow the reference's exact top-k (morsehgp3d/src/cpu/spatial/
// lbvh.cpp:1098-1198 lbvh_top_k): neighbours ordered by exact squared distance,
// ties ordered by PointId; the query point itself is excluded.  One wave
// per query, queries taken in Morton order so that neighbouring waves read
// the same groups.  Distances are FP64; a pair of candidates whose values
// are within rounding of each other and not both exact is reported in
// `flags` so that the host can settle the order exactly.
#include <algorithm>
#include <cmath>

#include "../host/exact.hpp"
#include "context.hpp"
#include "pipeline.hpp"
#include "traverse.hpp"
#include "wave_tree.hpp"

namespace mhgp {

namespace {

constexpr int kKnnBlock = 256;  // four waves, four queries

// One wave per query over the wave tree.  Lane l holds the l-th best
// neighbour so far, by (FP64 distance, PointId): a candidate's position is the
// number of lanes below it (one ballot), and the lanes above move up by one.
// The query's own group goes first, so the bound is tight before any other
// group is tested.  Bound by VALU issue of the insertions and the distance
// evaluations.  mhgp_knn over 50 000 points, k = 32: 10.4 ms with one thread
// per query (its list in scratch memory), 1.27 ms here, copies included.
__global__ void __launch_bounds__(kKnnBlock) k_knn(WaveTree T, int k, uint32_t *out, int stride,
                                                   uint8_t *flags) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t p = blockIdx.x * (kKnnBlock / 64) + (threadIdx.x >> 6);
  if (p >= T.n) return;
  const int kk = min(k + 1, (int)T.n - 1);  // slots that decide (k, plus one tie probe)
  const uint32_t self = T.leaf_id[p];
  const double q[3] = {T.LX[p], T.LY[p], T.LZ[p]};
  const WaveQuery Q(q[0], q[1], q[2]);
  double bd = INFINITY;
  uint32_t bi = kInvalid;
  uint32_t bx = 0;         // 1: the distance is exact
  double cut = INFINITY;   // squared distance of the kk-th best so far
  double most = INFINITY;
  auto group = [&](uint32_t g) {
    const uint32_t lp = g * 64 + lane, at = min(lp, T.n - 1);
    const uint32_t id = T.leaf_id[at];
    bool ex;
    const double d = d2_flag(q, T.LX[at], T.LY[at], T.LZ[at], ex);
    const bool valid = lp < T.n && lp != p;
    uint64_t cand = __ballot(valid && d <= cut);
    if (!cand) return;
    const uint64_t exact = __ballot(ex);
    while (cand) {
      const int i = __builtin_amdgcn_readfirstlane(__ffsll((long long)cand) - 1);
      cand &= cand - 1;
      const double cd = lane_f64(d, i);
      const uint32_t ci = lane_u32(id, i), cx = (uint32_t)(exact >> i) & 1u;
      const uint32_t pos = (uint32_t)__popcll(__ballot(bd < cd || (bd == cd && bi < ci)));
      const double ud = __shfl_up(bd, 1u);
      const uint32_t ui = __shfl_up(bi, 1u), ux = __shfl_up(bx, 1u);
      bd = lane < pos ? bd : (lane == pos ? cd : ud);
      bi = lane < pos ? bi : (lane == pos ? ci : ui);
      bx = lane < pos ? bx : (lane == pos ? cx : ux);
      cut = lane_f64(bd, kk - 1);
      cand &= __ballot(d <= cut);
    }
    most = wave_bound(cut);
  };
  const uint32_t own = p >> 6;
  group(own);
  wave_tree_visit(T, Q, most, [&](uint32_t g) {
    if (g != own) group(g);
  });
  const double nd = __shfl_down(bd, 1u);
  const uint32_t nx = __shfl_down(bx, 1u);
  const bool tie = (int)lane + 1 < kk && !(bx && nx) && (nd - bd) <= kSlack * nd + kSlackAbs;
  const uint64_t any = __ballot(tie);
  if ((int)lane < stride) out[(int64_t)self * stride + lane] = (int)lane < min(k, kk) ? bi : kInvalid;
  if (lane == 0) flags[self] = any ? 1 : 0;
}

// Exact top-k partition of rational query points (reference lbvh_top_k,
// morsehgp3d/include/morsehgp3d/spatial/lbvh.hpp:424 with the TopKPartition
// of spatial/query.hpp:109-169).  The device proposes: per query, the FP64
// k-th smallest distance r_k over the eligible points from the rounded query
// (pass 1), then every eligible point within r_k widened by the query's
// rounding and the distance roundings (pass 2).  Every point whose exact
// distance is at most the exact k-th lies in that set, so the host's exact
// replay over it decides the cutoff, the strict-below list and the complete
// cutoff shell.  Queries whose set overflows, or whose exclusion list does not
// fit, are settled by an exact host scan.
constexpr int kPartCand = 64;   // candidate slots per query
constexpr int kPartExcl = 64;   // exclusions checked on the device per query
constexpr uint32_t kPartHost = 1u;

struct PartParams {
  const double *q;        // 3 per query, device units
  const double *slack;    // per query: absolute distance slack (device units)
  const uint32_t *excl;   // exclusion ids, CSR
  const int64_t *eoff;
  int64_t queries;
  int k;
  WaveTree tree;
  uint32_t *cand;         // kPartCand per query
  uint32_t *ncand;
  uint32_t *flags;
};

// One wave per query over the wave tree.  Pass 1 keeps the k smallest eligible
// distances, lane l the l-th; pass 2 appends the candidates with ballots.  The
// exclusions sit one per lane.  With one thread per query the few hundred
// queries of a call were as many lanes of a handful of waves (509 queries of
// 20 011 points: 6.95 ms); bound by the latency of one traversal.
constexpr int kPartBlock = 256;  // four waves, four queries
__global__ void __launch_bounds__(kPartBlock) k_knn_partition(PartParams P) {
  const uint32_t lane = threadIdx.x & 63u;
  const int64_t q = (int64_t)blockIdx.x * (kPartBlock / 64) + (threadIdx.x >> 6);
  if (q >= P.queries) return;
  const WaveTree &T = P.tree;
  const int64_t e0 = P.eoff[q];
  const int ne = (int)min(P.eoff[q + 1] - e0, (int64_t)kPartExcl + 1);
  if (ne > kPartExcl) {
    if (lane == 0) {
      P.ncand[q] = 0;
      P.flags[q] = kPartHost;
    }
    return;
  }
  const uint32_t mine = (int)lane < ne ? P.excl[e0 + lane] : kInvalid;
  auto excluded = [&](uint32_t id) {
    bool x = false;
    for (int j = 0; j < ne; ++j) x |= lane_u32(mine, j) == id;
    return x;
  };
  const double qq[3] = {P.q[3 * q], P.q[3 * q + 1], P.q[3 * q + 2]};
  const WaveQuery Q(qq[0], qq[1], qq[2]);
  const int k = P.k;
  auto distance = [&](uint32_t at) {
    const double dx = T.LX[at] - qq[0], dy = T.LY[at] - qq[1], dz = T.LZ[at] - qq[2];
    return dx * dx + dy * dy + dz * dz;
  };
  // pass 1: the FP64 k-th smallest squared distance over eligible points
  double bd = INFINITY, cut = INFINITY;
  double most = INFINITY;
  auto group = [&](uint32_t g) {
    const uint32_t lp = g * 64 + lane, at = min(lp, T.n - 1);
    const double d = distance(at);
    bool in = lp < T.n && d < cut;
    if (!__ballot(in)) return;
    in = in && !excluded(T.leaf_id[at]);
    uint64_t cand = __ballot(in);
    while (cand) {
      const int i = __builtin_amdgcn_readfirstlane(__ffsll((long long)cand) - 1);
      cand &= cand - 1;
      const double cd = lane_f64(d, i);
      const uint32_t pos = (uint32_t)__popcll(__ballot(bd <= cd));
      const double ud = __shfl_up(bd, 1u);
      bd = lane < pos ? bd : (lane == pos ? cd : ud);
      cut = lane_f64(bd, k - 1);
      cand &= __ballot(d < cut);
    }
    most = wave_bound(cut);
  };
  const uint32_t first = wave_near_group(T, Q);
  group(first);
  wave_tree_visit(T, Q, most, [&](uint32_t g) {
    if (g != first) group(g);
  });
  if (!(cut < INFINITY)) {
    if (lane == 0) {
      P.ncand[q] = 0;
      P.flags[q] = kPartHost;
    }
    return;
  }
  // pass 2: every eligible point that can be at or below the exact k-th
  const double rk = sqrt(cut);
  const double R = (rk * (1.0 + 1e-12) + 2.0 * P.slack[q]) * (1.0 + 1e-12) + 1e-300;
  const double R2 = R * R * (1.0 + 1e-12);
  uint32_t nc = 0;
  most = wave_bound(R2);
  wave_tree_visit(T, Q, most, [&](uint32_t g) {
    const uint32_t lp = g * 64 + lane, at = min(lp, T.n - 1);
    bool in = lp < T.n && !(distance(at) > R2);
    if (!__ballot(in)) return;
    const uint32_t id = T.leaf_id[at];
    in = in && !excluded(id);
    const uint64_t m = __ballot(in);
    const uint32_t slot = nc + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
    if (in && slot < (uint32_t)kPartCand) P.cand[q * kPartCand + slot] = id;
    nc += (uint32_t)__popcll(m);
  });
  if (lane == 0) {
    P.ncand[q] = nc;
    P.flags[q] = nc > (uint32_t)kPartCand ? kPartHost : 0;
  }
}

}  // namespace

void knn_partition(Context &c, const int64_t *num, const int64_t *den, int64_t Q, int k, const uint32_t *excl,
                   const int64_t *eoff, uint32_t shell_cap, uint32_t *choice, uint32_t *strict,
                   uint32_t *strict_count, uint32_t *shell, uint32_t *shell_count, uint32_t *cutoff_id,
                   double *cutoff_sq) {
  require_cloud(c);
  const int64_t n = c.n;
  if (k < 1 || k > 32) throw std::invalid_argument("requested rank must lie in 1..32");
  if (Q < 0 || (Q > 0 && (!num || !den || !choice || !strict || !strict_count || !shell_count || !cutoff_id ||
                          !cutoff_sq || (shell_cap && !shell))))
    throw std::invalid_argument("invalid top-k partition arrays");
  if (Q == 0) return;
  std::vector<int64_t> off(Q + 1, 0);
  if (eoff) {
    if (eoff[0] != 0) throw std::invalid_argument("exclusion offsets must start at zero");
    for (int64_t q = 0; q < Q; ++q) {
      if (eoff[q + 1] < eoff[q]) throw std::invalid_argument("exclusion offsets must not decrease");
      off[q + 1] = eoff[q + 1];
    }
  }
  const int64_t E = off[Q];
  if (E && !excl) throw std::invalid_argument("null exclusion ids");
  std::vector<double> qf(3 * (size_t)Q), slack(Q);
  for (int64_t q = 0; q < Q; ++q) {
    if (den[q] <= 0) throw std::invalid_argument("query denominators must be positive");
    // eligible points: distinct, in range, not excluded
    std::vector<uint32_t> ex(excl + off[q], excl + off[q + 1]);
    std::sort(ex.begin(), ex.end());
    ex.erase(std::unique(ex.begin(), ex.end()), ex.end());
    for (uint32_t id : ex)
      if (id >= (uint64_t)n) throw std::invalid_argument("excluded PointId out of range");
    if ((int64_t)ex.size() + k > n) throw std::invalid_argument("the requested rank exceeds the eligible point count");
    double m = 0;
    for (int a = 0; a < 3; ++a) {
      // num / den rounded (each conversion and the division lose at most half
      // an ulp), in the device's unit
      const double v = (double)num[3 * q + a] / (double)den[q];
      qf[3 * q + a] = std::ldexp(v, c.scale_exp);
      m = std::max(m, std::fabs(v));
    }
    slack[q] = std::ldexp(m * 8.0 * 0x1p-53 * 1.7320508075688772 + 1e-300, c.scale_exp) + 1e-300;
  }
  hipStream_t s = c.stream;
  DevBuf<double> d_q, d_slack;
  DevBuf<uint32_t> d_ex, d_cand, d_nc, d_fl;
  DevBuf<int64_t> d_off;
  d_q.ensure(3 * Q);
  d_slack.ensure(Q);
  d_ex.ensure(std::max<int64_t>(E, 1));
  d_off.ensure(Q + 1);
  d_cand.ensure((size_t)Q * kPartCand);
  d_nc.ensure(Q);
  d_fl.ensure(Q);
  MHGP_HIP(hipMemcpyAsync(d_q.p, qf.data(), 3 * Q * 8, hipMemcpyHostToDevice, s));
  MHGP_HIP(hipMemcpyAsync(d_slack.p, slack.data(), Q * 8, hipMemcpyHostToDevice, s));
  if (E) MHGP_HIP(hipMemcpyAsync(d_ex.p, excl, E * 4, hipMemcpyHostToDevice, s));
  MHGP_HIP(hipMemcpyAsync(d_off.p, off.data(), (Q + 1) * 8, hipMemcpyHostToDevice, s));
  std::vector<uint32_t> cand((size_t)Q * kPartCand), nc(Q), fl(Q, kPartHost);
  if (n > 1) {
    PartParams P{d_q.p, d_slack.p, d_ex.p, d_off.p, Q, k, wave_tree(c), d_cand.p, d_nc.p, d_fl.p};
    hipLaunchKernelGGL(k_knn_partition, dim3(blocks_for(Q, kPartBlock / 64)), dim3(kPartBlock), 0, s, P);
    MHGP_LAUNCH_CHECK();
    MHGP_HIP(hipMemcpyAsync(cand.data(), d_cand.p, cand.size() * 4, hipMemcpyDeviceToHost, s));
    MHGP_HIP(hipMemcpyAsync(nc.data(), d_nc.p, Q * 4, hipMemcpyDeviceToHost, s));
    copy_wait(fl.data(), d_fl.p, Q * 4, hipMemcpyDeviceToHost, s);
  }
  // exact replay: squared distances times den^2 (and a power of two common to
  // the whole cloud) as integers, X_a = P_a * den - num_a scaled to integers
  const ExactCloud &ex = exact_cloud(c);
  const int e0 = ex.e0();
  std::vector<std::pair<BigInt, uint32_t>> ev;
  for (int64_t q = 0; q < Q; ++q) {
    BigInt bden(den[q]), bnum[3];
    for (int a = 0; a < 3; ++a) bnum[a] = BigInt(num[3 * q + a]);
    // value = P 2^e0: with e0 < 0 the numerators take the power instead
    BigInt pden = e0 >= 0 ? BigInt::from_dyadic(den[q], e0) : bden;
    if (e0 < 0)
      for (int a = 0; a < 3; ++a) bnum[a] = bnum[a] * BigInt::from_dyadic(1, -e0);
    std::vector<uint32_t> exq(excl + off[q], excl + off[q + 1]);
    std::sort(exq.begin(), exq.end());
    auto excluded = [&](uint32_t id) { return std::binary_search(exq.begin(), exq.end(), id); };
    auto dist = [&](uint32_t id) {
      BigInt sum(0);
      for (int a = 0; a < 3; ++a) {
        BigInt x = ex.coord(id, a) * pden - bnum[a];
        sum = sum + x * x;
      }
      return sum;
    };
    ev.clear();
    if (fl[q] & kPartHost) {
      for (int64_t id = 0; id < n; ++id)
        if (!excluded((uint32_t)id)) ev.emplace_back(dist((uint32_t)id), (uint32_t)id);
    } else {
      for (uint32_t i = 0; i < nc[q]; ++i) {
        const uint32_t id = cand[(size_t)q * kPartCand + i];
        ev.emplace_back(dist(id), id);
      }
    }
    if ((int64_t)ev.size() < k) throw std::logic_error("top-k partition: fewer candidates than the requested rank");
    std::sort(ev.begin(), ev.end(), [](const auto &a, const auto &b) {
      const int s2 = compare(a.first, b.first);
      return s2 != 0 ? s2 < 0 : a.second < b.second;
    });
    const BigInt &cutv = ev[k - 1].first;
    uint32_t ns = 0, nsh = 0;
    std::vector<uint32_t> sh;
    for (const auto &e : ev) {
      const int s2 = compare(e.first, cutv);
      if (s2 < 0) strict[(size_t)q * k + ns++] = e.second;
      else if (s2 == 0) sh.push_back(e.second);
    }
    std::sort(sh.begin(), sh.end());
    nsh = (uint32_t)sh.size();
    for (uint32_t i = ns; i < (uint32_t)k; ++i) strict[(size_t)q * k + i] = kInvalid;
    strict_count[q] = ns;
    shell_count[q] = nsh;
    for (uint32_t i = 0; i < shell_cap; ++i) shell[(size_t)q * shell_cap + i] = i < nsh ? sh[i] : kInvalid;
    cutoff_id[q] = sh[0];
    std::vector<uint32_t> ch(strict + (size_t)q * k, strict + (size_t)q * k + ns);
    for (uint32_t i = 0; ns + i < (uint32_t)k; ++i) ch.push_back(sh[i]);
    std::sort(ch.begin(), ch.end());
    std::copy(ch.begin(), ch.end(), choice + (size_t)q * k);
    // cutoff = sum / den^2 in input units (times 2^(2 e0) when e0 < 0)
    cutoff_sq[q] = cutv.sign() == 0 ? 0.0 : ratio_to_double(cutv, bden * bden, e0 < 0 ? 2 * e0 : 0);
  }
}

void knn_all(Context &c, int k, uint32_t *d_out, uint8_t *d_flags, hipStream_t stream, int stride) {
  if (k < 1 || k > 63) throw std::invalid_argument("k must lie in 1..63");
  if (k >= c.n) throw std::invalid_argument("k must be smaller than the point count");
  hipStream_t s = stream ? stream : c.stream;
  hipLaunchKernelGGL(k_knn, dim3(blocks_for(c.n, kKnnBlock / 64)), dim3(kKnnBlock), 0, s, wave_tree(c), k, d_out,
                     stride ? stride : k, d_flags);
  MHGP_LAUNCH_CHECK();
}

}  // namespace mhgp
