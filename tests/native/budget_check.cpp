// C entry points to the sizes of csrc/budget.hpp for test_memory_prediction.py.
#include "budget.hpp"

extern "C" {
static int64_t queue_bytes(const mhgp::CatalogueQueues &q) {
  return (int64_t)(q.events * mhgp::kRecordBytes + q.fallbacks * 32 + q.region_words * 4);
}
int64_t budget_predict(int64_t n, int k_max) { return mhgp::predict_bytes(n, k_max); }
// queues, rescan list and slabs that the catalogue allocates first
int64_t budget_catalogue(int64_t n, int k_max) {
  const mhgp::CatalogueQueues q = mhgp::first_queues(n, k_max + 1);
  return queue_bytes(q) + (int64_t)q.rescans * mhgp::kRescanBytes +
         std::min<int64_t>(mhgp::kProbeSlabs, n * (int64_t)mhgp::probe_slab_doubles(mhgp::kGatherCap) * 8);
}
// record queues of an unbounded context, and of one with a device capacity
// with its rescans and the slabs' least
int64_t budget_queues(int64_t n, int k_max) { return queue_bytes(mhgp::first_queues(n, k_max + 1)); }
int64_t budget_bounded(int64_t n, int k_max) {
  const mhgp::CatalogueQueues q = mhgp::first_queues_bounded(n, k_max + 1);
  return queue_bytes(q) + (int64_t)q.rescans * mhgp::kRescanBytes + mhgp::probe_slabs_least(n);
}
uint64_t budget_slabs(int64_t left, uint64_t held, int64_t least, int64_t most) {
  return mhgp::probe_slab_budget(left, held, least, most);
}
}
