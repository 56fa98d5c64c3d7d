// A download's ring and the helper threads (autopas_amd/csrc/ljg_ring.h) with a thread in the device's place.
#include <chrono>
#include <cstdio>
#include <cstdlib>

#include "../../autopas_amd/csrc/ljg_ring.h"

using namespace std::chrono_literals;

#define CHECK(x)                                           \
  do {                                                     \
    if (!(x)) {                                            \
      std::printf("line %d: %s\n", __LINE__, #x);          \
      return 1;                                            \
    }                                                      \
  } while (0)

// Nothing a helper does happens after join() or the end of the object, however late the helper is.
static int late() {
  std::atomic<int> runs{0};
  {
    ljg::Helpers h;
    for (int k = 0; k < 3; ++k)
      h.start([&runs]() {
        std::this_thread::sleep_for(30ms);
        runs.fetch_add(1);
      });
    h.join();
    CHECK(runs.load() == 3);
    for (int k = 0; k < 3; ++k)
      h.start([&runs]() {
        std::this_thread::sleep_for(30ms);
        runs.fetch_add(1);
      });
  }
  CHECK(runs.load() == 6);
  return 0;
}

// Helpers that ended go when others start, and there are never more than kMost.
static int bounded() {
  std::atomic<int> runs{0};
  ljg::Helpers h;
  for (int k = 0; k < 100; ++k) {
    h.start([&runs, k]() {
      if (k % 3 == 0) std::this_thread::sleep_for(2ms);
      runs.fetch_add(1);
    });
    CHECK(h.running() <= ljg::Helpers::kMost);
  }
  std::this_thread::sleep_for(50ms);
  h.start([]() {});
  CHECK(h.running() == 1);
  h.join();
  CHECK(runs.load() == 100);
  return 0;
}

// Every value arrives, with helpers that start in time, late or not at all.
static int values(size_t count, size_t chunk, int slots, int helpers, bool late_ones) {
  std::vector<double> dev(9 * count), ring((size_t)slots * chunk), out(9 * count, -1.);
  for (size_t i = 0; i < dev.size(); ++i) dev[i] = (double)i + 0.25;
  std::atomic<unsigned long long> word{0};
  auto shared = std::make_shared<ljg::Download>();
  ljg::Download &d = *shared;
  d.ring = ring.data();
  d.count = count;
  d.total = 9 * count;
  d.chunk = chunk;
  d.nchunks = (int)((d.total + chunk - 1) / chunk);
  d.slots = slots;
  for (int a = 0; a < 9; ++a) d.outs[a] = a == 4 ? nullptr : out.data() + (size_t)a * count;
  d.progress = reinterpret_cast<volatile unsigned long long *>(&word);
  d.base = 0;
  d.done.reset(new std::atomic<char>[(size_t)d.nchunks]);
  for (int k = 0; k < d.nchunks; ++k) d.done[k].store(0);
  std::thread device([&]() {
    for (int k = 0; k < d.nchunks; ++k) {
      while (k >= slots && d.done[k - slots].load(std::memory_order_acquire) == 0) std::this_thread::yield();
      const size_t b = (size_t)k * chunk, n = d.total - b < chunk ? d.total - b : chunk;
      std::memcpy(ring.data() + (size_t)(k % slots) * chunk, dev.data() + b, n * sizeof(double));
      word.store((unsigned long long)k + 1);
    }
  });
  ljg::Helpers h;
  for (int k = 0; k < helpers; ++k)
    h.start([shared, late_ones]() {
      if (late_ones) std::this_thread::sleep_for(20ms);
      shared->help();
    });
  d.help();
  for (int k = 0; k < d.nchunks; ++k)
    while (d.done[k].load(std::memory_order_acquire) == 0) std::this_thread::yield();
  device.join();
  // (the buffers go here, before the helpers are joined: a late one does not touch them)
  for (size_t i = 0; i < out.size(); ++i) CHECK(out[i] == (i / count == 4 ? -1. : dev[i]));
  std::vector<double>().swap(ring);
  std::vector<double>().swap(out);
  h.join();
  return 0;
}

int main() {
  int bad = late() + bounded();
  for (int helpers : {0, 1, 3})
    for (bool l : {false, true})
      for (int slots : {1, 3, 8}) {
        bad += values(1, 16, slots, helpers, l);
        bad += values(777, 64, slots, helpers, l);
        bad += values(1000, 1000, slots, helpers, l);
      }
  if (bad == 0) std::puts("ok ring");
  return bad;
}
