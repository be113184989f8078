// Host checks of the block cache and of the gate between stream captures and
// device synchronisations, over a memory whose allocations, frees and
// synchronisations are counted.  Usage: block_cache_host <check>.
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <thread>
#include <vector>

#include "block_cache.h"
#include "capture_gate.h"

using namespace qop;

#define CHECK(c)                                              \
  do {                                                        \
    if (!(c)) {                                               \
      fprintf(stderr, "line %d: %s\n", __LINE__, #c);         \
      exit(1);                                                \
    }                                                         \
  } while (0)

static void nap(int us) { std::this_thread::sleep_for(std::chrono::microseconds(us)); }

struct Device {
  CaptureGate gate;
  std::atomic<int> capturing{0}, syncs{0}, allocs{0}, frees{0};
  int sync_us = 0;
};
struct Memory {
  Device *d;
  int device() { return 0; }
  void *alloc(size_t n) {
    d->allocs++;
    return malloc(n < 64 ? 64 : n);
  }
  void free(void *p) {
    d->frees++;
    ::free(p);
  }
  bool try_sync() {
    if (!d->gate.sync_begin(false)) return false;
    CHECK(d->capturing == 0);
    nap(d->sync_us);
    CHECK(d->capturing == 0);
    d->syncs++;
    d->gate.sync_end();
    return true;
  }
  [[noreturn]] void out_of_memory(size_t) { throw std::bad_alloc(); }
};
using Cache = BlockCache<Memory>;

// A freed block is handed out again only after a synchronisation, and while
// a stream is captured there is none: the request gets a new block.
static void no_sync_in_capture() {
  Device d;
  Cache c(Memory{&d}, 1 << 20, 8 << 20);
  void *a = c.alloc(4096);
  c.free(a);
  d.gate.capture_begin();
  void *b = c.alloc(4096);
  CHECK(b != a && d.syncs == 0 && d.allocs == 2);
  d.gate.capture_end();
  void *e = c.alloc(4096);
  CHECK(e == a && d.syncs == 1 && d.allocs == 2);
  c.free(b);
  c.free(e);
  c.trim();
  CHECK(d.frees == 2);
}

// Threads that capture beside threads that allocate and free: no capture ever
// overlaps a synchronisation (checked inside try_sync), also of one that waits.
static void captures_and_syncs_exclude_each_other() {
  Device d;
  d.sync_us = 50;
  Cache c(Memory{&d}, 1 << 20, 8 << 20);
  std::atomic<bool> stop{false};
  std::vector<std::thread> ts;
  for (int i = 0; i < 2; i++)
    ts.emplace_back([&] {
      while (!stop) {
        d.gate.capture_begin();
        d.capturing++;
        nap(30);
        d.capturing--;
        d.gate.capture_end();
        nap(30);
      }
    });
  for (int i = 0; i < 3; i++)
    ts.emplace_back([&, i] {
      for (int k = 0; k < 300; k++) {
        void *p = c.alloc(1000 * (i + 1));
        memset(p, i, 1000 * (i + 1));
        c.free(p);
        if (k % 50 == 0) {
          CHECK(d.gate.sync_begin(true));
          CHECK(d.capturing == 0);
          d.gate.sync_end();
        }
      }
    });
  for (size_t i = 2; i < ts.size(); i++) ts[i].join();
  stop = true;
  ts[0].join();
  ts[1].join();
  c.trim();
  CHECK(d.allocs == d.frees);
}

int main(int argc, char **argv) {
  const struct {
    const char *name;
    void (*run)();
  } checks[] = {
      {"no_sync_in_capture", no_sync_in_capture},
      {"captures_and_syncs_exclude_each_other", captures_and_syncs_exclude_each_other},
  };
  for (auto &k : checks)
    if (argc == 2 && !strcmp(argv[1], k.name)) {
      k.run();
      return 0;
    }
  fprintf(stderr, "no such check\n");
  return 2;
}
