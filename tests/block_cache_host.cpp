// Host checks of the block cache over a memory whose allocations, frees and
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
  std::atomic<int> syncs{0}, allocs{0}, frees{0};
  std::atomic<bool> busy{false};  // no synchronisation possible now
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
    if (d->busy) return false;
    nap(d->sync_us);
    d->syncs++;
    return true;
  }
  [[noreturn]] void out_of_memory(size_t) { throw std::bad_alloc(); }
};
using Cache = BlockCache<Memory>;

// A freed block is handed out again only after a synchronisation; where there
// can be none the request gets a new block.
static void freed_blocks_wait_for_a_sync() {
  Device d;
  Cache c(Memory{&d}, 1 << 20, 8 << 20);
  void *a = c.alloc(4096);
  c.free(a);
  d.busy = true;
  void *b = c.alloc(4096);
  CHECK(b != a && d.syncs == 0 && d.allocs == 2);
  d.busy = false;
  void *e = c.alloc(4096);
  CHECK(e == a && d.syncs == 1 && d.allocs == 2);
  c.free(b);
  c.free(e);
  c.trim();
  CHECK(d.frees == 2);
}

int main(int argc, char **argv) {
  const struct {
    const char *name;
    void (*run)();
  } checks[] = {
      {"freed_blocks_wait_for_a_sync", freed_blocks_wait_for_a_sync},
  };
  for (auto &k : checks)
    if (argc == 2 && !strcmp(argv[1], k.name)) {
      k.run();
      return 0;
    }
  fprintf(stderr, "no such check\n");
  return 2;
}
