// Host threads of one call.
#pragma once

#include <system_error>
#include <thread>
#include <utility>
#include <vector>

namespace mhgp {

// Threads that are joined when the group ends, also by an exception (the end of
// a joinable std::thread ends the process).  start() returns false when the
// system has no thread to give: the caller does the work itself or without it.
class Threads {
 public:
  Threads() = default;
  Threads(const Threads &) = delete;
  Threads &operator=(const Threads &) = delete;
  ~Threads() { join(); }
  template <class F>
  bool start(F f) {
    try {
      t_.emplace_back(std::move(f));
      return true;
    } catch (const std::system_error &) {
      return false;
    }
  }
  void join() {
    for (auto &t : t_) t.join();
    t_.clear();
  }

 private:
  std::vector<std::thread> t_;
};

}  // namespace mhgp
