// Levels of supports by predicates.hpp on the host, for test_gpu_levels.py:
// per support `size` offsets from its first point, in PointId order.
#include "predicates.hpp"

extern "C" void levels(const double *rel, const int *size, long n, double *out) {
  using namespace mhgp;
  for (long i = 0; i < n; ++i) {
    const double *r = rel + 9 * i;
    const V3 a = {r[0], r[1], r[2]}, b = {r[3], r[4], r[5]}, d = {r[6], r[7], r[8]};
    if (size[i] == 2) {
      PairSphere s;
      s.init(a);
      out[i] = s.level();
    } else if (size[i] == 3) {
      TriSphere s;
      s.init(a, b);
      out[i] = s.level();
    } else {
      TetSphere s;
      s.init(a, b, d);
      out[i] = s.level();
    }
  }
}
