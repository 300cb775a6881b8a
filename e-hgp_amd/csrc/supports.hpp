// Device buffers and host records of the critical-sphere catalogue.
#pragma once

#include <vector>

#include "budget.hpp"
#include "stages.hpp"

namespace mhgp {

constexpr uint32_t kRegionCapTiny = 96, kRegionCapLittle = 180;  // members that one and two waves hold in LDS
constexpr int kRegionCap = 384;  // region members the smallest enumeration holds in LDS
constexpr uint32_t kRegionLimitMax = 2048;  // largest candidate region any path enumerates
constexpr int kGatherCapWide = 1024;  // the same for the wide probe and the next enumeration
constexpr int kGatherCapSlab = 2048;  // the same with the masks in the slab
constexpr int kRegionCapWide = 640;
constexpr int kMaxInterior = 10; // s_max - 2 for s_max <= 11 (K_max <= 10)

// One catalogue record: support ids (unused = kInvalid), meta
// (size | rank << 8 | interior count << 16 | degenerate << 24), interior ids,
// FP64 squared radius and a bound on its relative error.
struct EventRec {
  uint32_t ids[4];
  uint32_t meta;
  uint32_t interior[kMaxInterior];
  float level_err;
  double level;
};
static_assert(sizeof(EventRec) == kRecordBytes, "event layout");

// Work the device could not certify: the host settles it exactly.
// kind 2: pair (u, v); 3: face (u, v, w) incl. its triangle and apexes;
// 4: tetrahedron (u, v, w, z).  region_off/len locate the anchor's region.
struct FallbackRec {
  uint32_t kind;
  uint32_t ids[4];
  uint32_t region_off;
  uint32_t region_len;
  uint32_t pad;
};

// Streams beside a context's own, for launches between a fork and a join.
struct SideStreams {
  static constexpr int kCount = 2;
  hipStream_t stream[kCount] = {};
  hipEvent_t forked = nullptr, done[kCount] = {};
  SideStreams() = default;
  SideStreams(const SideStreams &) = delete;
  SideStreams &operator=(const SideStreams &) = delete;
  ~SideStreams() {
    for (int i = 0; i < kCount; ++i) {
      if (stream[i]) (void)hipStreamDestroy(stream[i]);
      if (done[i]) (void)hipEventDestroy(done[i]);
    }
    if (forked) (void)hipEventDestroy(forked);
  }
  // the first `count` streams go on from what s holds now
  void fork(hipStream_t s, int count) {
    if (!forked) MHGP_HIP(hipEventCreateWithFlags(&forked, hipEventDisableTiming));
    MHGP_HIP(hipEventRecord(forked, s));
    for (int i = 0; i < count; ++i) {
      if (!stream[i]) MHGP_HIP(hipStreamCreateWithFlags(&stream[i], hipStreamNonBlocking));
      if (!done[i]) MHGP_HIP(hipEventCreateWithFlags(&done[i], hipEventDisableTiming));
      MHGP_HIP(hipStreamWaitEvent(stream[i], forked, 0));
    }
  }
  // s waits for them
  void join(hipStream_t s, int count) {
    for (int i = 0; i < count; ++i) {
      MHGP_HIP(hipEventRecord(done[i], stream[i]));
      MHGP_HIP(hipStreamWaitEvent(s, done[i], 0));
    }
  }
};

struct CatalogBuffers {
  bool valid = false;
  int k_max = 0;
  int s_max = 0;
  DevBuf<double> radius;          // gather radius per anchor
  DevBuf<uint32_t> gcount;        // gathered count per anchor
  DevBuf<uint64_t> goff;          // CSR offsets
  DevBuf<uint32_t> glist;         // gathered ids
  DevBuf<uint32_t> region;        // region size of a probed anchor
  DevBuf<uint32_t> lists;         // anchors by what comes next for them (supports.hip)
  DevBuf<uint8_t> rescans;        // sides of faces left to the rescan kernel
  DevBuf<uint32_t> big;           // anchors of a global-memory launch
  DevBuf<EventRec> events;
  DevBuf<FallbackRec> fallbacks;
  DevBuf<uint32_t> fb_region;     // region member ids of anchors with fallbacks
  DevBuf<uint64_t> counters;      // events, fallbacks, region words, candidates, operations, list lengths
  DevBuf<double> cells;           // per cell: dir xyz, cos d, sin d, chord
  DevBuf<float> cellf;            // per cell: the FP32 cell of the certificate and the masks
  DevBuf<uint64_t> strips;        // cells that a great circle can meet, by its axis
  DevBuf<double> scratch;         // slabs: the regions of probed anchors
  DevBuf<uint32_t> anchors;       // anchor list of the current launch
  // canonical order on the device: records (device emitted + host settled),
  // their order by (exact level, rank, support) and dense exact level classes
  int64_t count = 0;
  DevBuf<uint64_t> sort_keys;
  DevBuf<uint32_t> order;
  DevBuf<uint32_t> cls;
  DevBuf<uint32_t> ambiguous;     // open-run starts, and the runs left to the host (start, length)
  // small per-call device scratch, kept so that no call frees device memory
  // (a free waits for the whole device, side streams included)
  DevBuf<uint64_t> total;         // gathered entries of a pass
  DevBuf<uint64_t> run_count;     // open runs, runs left to the host
  DevBuf<uint32_t> run_pos, run_gidx, run_new, run_link;
  PinnedBuf pinned;               // small results on their way to the caller
  DevBuf<EventRec> run_rec;       // records of the runs ordered on the host
  int64_t open_runs = 0;          // runs the FP64 intervals left open
  int64_t host_runs = 0;          // of those, runs ordered exactly on the host
  mhgp_catalog_info info{};
  SideStreams sides;              // declared last: gone before the buffers they use
};

int64_t catalog_device_bytes(const CatalogBuffers &b);
// order.hip: canonical order and level classes of B.events[0, B.count)
void order_catalogue(Context &c, CatalogBuffers &B);

}  // namespace mhgp
