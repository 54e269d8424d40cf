// Results that kernels write into pinned host memory, and the wait for them.
// Host code without HIP: the caller passes the stream synchronisation in.
#pragma once
#include <algorithm>
#include <chrono>
#include <cstdint>
#include <thread>
#include <vector>

namespace lmm {

// A signalling NaN, which no arithmetic returns: an entry that holds it has
// not been written yet.
constexpr uint64_t RESULT_UNWRITTEN = 0x7ff4a5a5c3c3f00dull;

class HostResults {
 public:
  // Marks the n entries from h on that the kernel launched next will write.
  double *arm(double *h, int n) {
    for (int q = 0; q < n; q++) {
      if (std::find(armed_.begin(), armed_.end(), h + q) != armed_.end()) twice_ = true;
      else armed_.push_back(h + q);
      __atomic_store_n(reinterpret_cast<uint64_t *>(h + q), RESULT_UNWRITTEN, __ATOMIC_RELAXED);
    }
    return h;
  }

  // Waits until every armed entry is written; false when they do not arrive.
  // Each entry is written whole and tells by itself that it is there, so no
  // order between them is needed.  A wait that finds nothing armed or an entry
  // armed twice (the first write would pass for the second), or that limit_us
  // do not end, calls sync (true when it succeeded), after which every entry
  // must have been written.  The poll spins for its first few microseconds and
  // then yields its core between looks, so that waiting threads outnumbering
  // the cores do not keep one another from launching.
  template <typename Sync>
  bool wait(long limit_us, Sync &&sync) {
    bool ok = !armed_.empty() && !twice_ && limit_us > 0 && poll(limit_us);
    if (!ok) ok = sync() && written();
    armed_.clear();
    twice_ = false;
    return ok;
  }

 private:
  static bool is_written(const double *e) {
    return __atomic_load_n(reinterpret_cast<const uint64_t *>(e), __ATOMIC_ACQUIRE) != RESULT_UNWRITTEN;
  }
  bool written() const { return std::all_of(armed_.begin(), armed_.end(), is_written); }
  bool poll(long limit_us) const {
    const auto t0 = std::chrono::steady_clock::now();
    size_t n = 0;
    for (unsigned spin = 1;; spin++) {
      while (n < armed_.size() && is_written(armed_[n])) n++;
      if (n == armed_.size()) return true;
      if (spin < SPINS) __builtin_ia32_pause();
      else std::this_thread::yield();
      if (spin % 64 == 0 && std::chrono::steady_clock::now() - t0 > std::chrono::microseconds(limit_us)) return false;
    }
  }
  static constexpr unsigned SPINS = 256;
  std::vector<double *> armed_;
  bool twice_ = false;
};

}  // namespace lmm
