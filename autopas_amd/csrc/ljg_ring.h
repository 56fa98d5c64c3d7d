// ljg_ring.h -- the host's side of a download's ring of chunks, and the threads that help with it (no HIP needed).
#pragma once

#include <atomic>
#include <cstddef>
#include <cstring>
#include <memory>
#include <thread>
#include <utility>
#include <vector>

namespace ljg {

// The copy out of a download: `total` doubles on the device, nine arrays of `count` back to back (null outputs
// are left out), as chunks through the ring.  Chunk k occupies ring slot k mod slots; it is queued once chunk
// k - slots has been copied out, and is complete when the progress word passes it.  The calling thread queues the
// chunks; all threads take chunks in order and copy them out.  The call does not wait for the helpers, which share
// this object: one that the scheduler lets start late (the caller's own worker threads may be spinning on every core:
// 2 to 3 ms were seen) finds no chunk left and ends without touching the buffers, and only chunks that were
// taken are waited for.
struct Download {
  const double *ring;
  size_t count, chunk, total;
  int nchunks, slots;
  double *outs[9];
  volatile unsigned long long *progress;
  unsigned long long base;  // progress holds base + the number of complete chunks
  std::unique_ptr<std::atomic<char>[]> done;  // 1: copied out, 2: given up
  std::atomic<int> next{0};
  std::atomic<bool> abort{false};

  bool ready(int k) const {
    const unsigned long long p = *progress;
    return p > base + (unsigned long long)k && p <= base + (unsigned long long)nchunks;
  }
  void copy_out(int k) {
    std::atomic_thread_fence(std::memory_order_acquire);
    const size_t b = (size_t)k * chunk, e = b + chunk < total ? b + chunk : total;
    const double *src = ring + (size_t)(k % slots) * chunk;
    for (size_t i = b; i < e;) {
      const size_t a = i / count, stop = (a + 1) * count < e ? (a + 1) * count : e;
      if (outs[a]) std::memcpy(outs[a] + (i - a * count), src + (i - b), (stop - i) * sizeof(double));
      i = stop;
    }
    done[k].store(1, std::memory_order_release);
  }
  void help() {
    for (;;) {
      const int k = next.fetch_add(1);
      if (k >= nchunks) return;
      for (unsigned spins = 0; !ready(k); ++spins) {
        if (abort.load(std::memory_order_relaxed)) {
          done[k].store(2, std::memory_order_release);
          return;
        }
        if (spins > 64) std::this_thread::yield();
      }
      copy_out(k);
    }
  }
};

// The helper threads of a context.  A call does not wait for those it started; they are joined once they have ended,
// when there are kMost of them, and all of them before the context goes: none outlives it, and so none is left to run
// when the library is unloaded.
class Helpers {
 public:
  static constexpr size_t kMost = 12;
  Helpers() = default;
  Helpers(const Helpers &) = delete;
  Helpers &operator=(const Helpers &) = delete;
  ~Helpers() { join(); }

  // Runs f() on a thread of its own (throws std::exception if there is none to be had).
  template <class F>
  void start(F f) {
    for (size_t k = 0; k < all_.size();) {
      if (all_[k].ended->load(std::memory_order_acquire) || all_.size() >= kMost) {
        all_[k].thread.join();
        all_.erase(all_.begin() + (std::ptrdiff_t)k);
      } else {
        ++k;
      }
    }
    auto ended = std::make_shared<std::atomic<bool>>(false);
    all_.reserve(all_.size() + 1);  // (nothing may throw between a thread's start and its place here)
    all_.push_back(One{std::thread([f, ended]() {
                         f();
                         ended->store(true, std::memory_order_release);
                       }),
                       std::move(ended)});
  }
  void join() {
    for (One &o : all_) o.thread.join();
    all_.clear();
  }
  size_t running() const { return all_.size(); }

 private:
  struct One {
    std::thread thread;
    std::shared_ptr<std::atomic<bool>> ended;
  };
  std::vector<One> all_;
};

}  // namespace ljg
