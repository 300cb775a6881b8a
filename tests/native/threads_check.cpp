// A tower's copies when the system gives only some of the threads they ask for
// (pthread_create below refuses all after the first `allowed`): the arrays are
// complete all the same.  Prints "ok".
#include <dlfcn.h>
#include <errno.h>
#include <pthread.h>

#include <cstdio>
#include <cstdlib>

#include "tower_state.hpp"

static int allowed, asked;
extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *x) {
  static auto real = (int (*)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *))dlsym(RTLD_NEXT, "pthread_create");
  return asked++ < allowed ? real(t, a, f, x) : EAGAIN;
}

int main(int, char **argv) {
  allowed = std::atoi(argv[1]);
  mhgp::TowerState T;
  const int orders = 5, per = 20000;
  for (int o = 1; o <= orders; ++o) {
    mhgp::Forest F;
    for (int64_t i = 0; i < per; ++i) {
      const int64_t kid = i - 1;
      F.add(o, 1, i, 0.5 * (double)i, &kid, i ? 1 : 0);
      F.vtarget.push_back(o > 1 ? i / 2 : -1);
    }
    T.forests.push_back(std::move(F));
    T.node_count += per;
    T.child_count += per - 1;
  }
  std::vector<int32_t> order(T.node_count), kind(T.node_count);
  std::vector<int64_t> cls(T.node_count), off(T.node_count + 1), kids(T.child_count), target(T.node_count);
  std::vector<double> level(T.node_count);
  T.copy_out(order.data(), kind.data(), cls.data(), level.data(), off.data(), kids.data());
  asked = 0;
  T.copy_vertical(target.data());
  for (int64_t x = 0; x < T.node_count; ++x) {
    const int64_t o = x / per, i = x % per, first = o * (per - 1) + i;
    const bool good = order[x] == o + 1 && kind[x] == 1 && cls[x] == i && level[x] == 0.5 * (double)i &&
                      off[x + 1] == first && (i == 0 || kids[first - 1] == x - 1) &&
                      target[x] == (o ? (o - 1) * per + i / 2 : -1);
    if (!good) return std::printf("wrong at node %lld\n", (long long)x), 1;
  }
  std::puts("ok");
}
