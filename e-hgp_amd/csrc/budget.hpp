// Sizes of the catalogue's buffers and of a request, as plain host arithmetic
// (no HIP), so that the server's admission counts what the catalogue allocates.
#pragma once

#include <algorithm>
#include <cstdint>

namespace mhgp {

constexpr int kCells = 384;      // 6 cube faces x 8 x 8 direction cells
constexpr int kGatherCap = 600;  // gathered neighbours the probe holds in LDS
constexpr int64_t kRecordBytes = 72;  // EventRec
constexpr int64_t kRescanBytes = 24;  // a side of a face left to the rescan kernel

// Slab of one probed anchor (in doubles), for G gathered points:
// [0, 3G) coordinates x, y, z relative to the anchor; [3G, 3G + kCells) cell
// radii (float); [3G + kCells, 9G + kCells) masks, six words per point; then
// PointIds.  The global-memory kernel adds its own arrays behind them.
constexpr uint64_t slab_masks(uint64_t G) { return 3 * G + kCells; }
constexpr uint64_t slab_ids(uint64_t G) { return 9 * G + kCells; }
constexpr uint64_t probe_slab_doubles(uint64_t G) { return (slab_ids(G) + (G + 1) / 2 + 1) & ~1ull; }

// Most memory that the slabs of one probe launch take, and the least that a
// context with a device capacity keeps for them.
constexpr int64_t kProbeSlabs = int64_t(2) << 30;
constexpr int64_t probe_slabs_least(int64_t n) { return std::max<int64_t>(1 << 20, 64 * n); }

// Bytes for a launch's slabs: those held and a quarter of what is left, within
// [least, most].
constexpr uint64_t probe_slab_budget(int64_t left, uint64_t held, int64_t least, int64_t most) {
  const uint64_t b = (uint64_t)std::max<int64_t>(left, 0) / 4 + held;
  return std::min<uint64_t>(std::max<uint64_t>(b, (uint64_t)least), (uint64_t)most);
}

// First capacities of the catalogue's queues (a catalogue that outgrows them
// runs again with larger ones).
struct CatalogueQueues {
  uint64_t events, fallbacks, region_words, rescans;
};
inline CatalogueQueues first_queues(int64_t n, int s_max) {
  const uint64_t m = (uint64_t)n;
  // a longer rescan list costs the enumeration again (lattices displaced by 1%
  // of their spacing leave several sides a point)
  return {std::max<uint64_t>(1024, m * (s_max >= 11 ? 640 : 64 * (uint64_t)s_max)), std::max<uint64_t>(4096, m / 4),
          std::max<uint64_t>(1 << 20, m * 64), std::max<uint64_t>(1 << 14, m * 16)};
}
// The same in a context with a device capacity: one rescan a point (more where
// the capacity leaves room).  The queues give up what the slabs' least, the
// rescans, the tables and the anchor lists and neighbour rows take: the
// fallback regions the fixed part, the records 234 bytes a point (3.25 of at
// least 128 records), so that a capacity for the whole queues holds it all.
inline CatalogueQueues first_queues_bounded(int64_t n, int s_max) {
  CatalogueQueues q = first_queues(n, s_max);
  q.rescans = std::max<uint64_t>(1 << 14, (uint64_t)n);
  q.region_words -= ((1 << 20) + (1 << 14) * kRescanBytes + 53248) / 4;
  q.events -= (uint64_t)n * 13 / 4;
  return q;
}

// Predicted device bytes of one request (upload, EMST, catalogue, tower on one
// lane): the record queues, the slabs of a probe launch, and what grows with
// the records themselves (their order, 44 bytes; a tower lane's workspaces,
// about 120 bytes measured over 1 000 to 120 000 points, K 1 to 10), of which
// a generic cloud has about k^3 / 2 + 6 k per point.  Per point the LBVH, EMST
// and neighbour rows take 700 bytes, the gathers about 1 800.  Gathers beyond
// 2 048 points (anisotropic mixtures) take slabs of their own beyond this.
inline int64_t predict_bytes(int64_t n, int k_max) {
  const CatalogueQueues q = first_queues(n, std::min(k_max, 10) + 1);
  const int64_t k = k_max, records = n * (k * k * k + 12 * k) / 2;
  return (64ll << 20) + n * 2560 + (int64_t)q.events * kRecordBytes + (int64_t)q.fallbacks * 32 +
         (int64_t)q.region_words * 4 + (int64_t)q.rescans * kRescanBytes +
         std::min<int64_t>(kProbeSlabs, n * (int64_t)probe_slab_doubles(kGatherCap) * 8) + records * 170;
}

}  // namespace mhgp
