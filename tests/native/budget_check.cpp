// C entry points to the sizes of csrc/budget.hpp for test_memory_prediction.py.
#include "budget.hpp"

extern "C" {
int64_t budget_predict(int64_t n, int k_max) { return mhgp::predict_bytes(n, k_max); }
// queues, rescan list and slabs that the catalogue allocates first
int64_t budget_catalogue(int64_t n, int k_max) {
  const mhgp::CatalogueQueues q = mhgp::first_queues(n, k_max + 1);
  return (int64_t)(q.events * mhgp::kRecordBytes + q.fallbacks * 32 + q.region_words * 4 + q.rescans * mhgp::kRescanBytes) +
         std::min<int64_t>(mhgp::kProbeSlabs, n * (int64_t)mhgp::probe_slab_doubles(mhgp::kGatherCap) * 8);
}
}
