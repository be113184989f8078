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
  std::atomic<size_t> room{(size_t)1 << 40};  // bytes left
  std::atomic<bool> busy{false};  // no synchronisation possible now
  std::atomic<bool> waiting{false}, release{true};  // synchronisations and frees last until released
  void wait() {
    waiting = true;
    while (!release) std::this_thread::sleep_for(std::chrono::microseconds(20));
    waiting = false;
  }
};
struct Memory {
  Device *d;
  int device() { return 0; }
  void *alloc(size_t n) {
    if (n > d->room) return nullptr;
    d->room -= n;
    d->allocs++;
    size_t *p = (size_t *)malloc(n + 16);
    p[0] = n;
    return p + 2;
  }
  void free(void *p) {
    d->frees++;
    d->wait();
    size_t *q = (size_t *)p - 2;
    d->room += q[0];
    ::free(q);
  }
  bool try_sync() {
    if (d->busy) return false;
    d->wait();
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

// While one thread waits for the device the others allocate and free, and a
// block freed during the wait is not handed out by it.
static void nobody_waits_behind_a_sync() {
  Device d;
  Cache c(Memory{&d}, 1 << 20, 8 << 20);
  void *a = c.alloc(4096), *b = c.alloc(4096);
  c.free(a);
  d.release = false;
  void *got = nullptr;
  std::thread t([&] { got = c.alloc(4096); });
  while (!d.waiting) nap(20);
  std::atomic<bool> done{false};
  std::thread u([&] {
    void *x = c.alloc(100000);
    c.free(x);
    c.free(b);
    done = true;
  });
  for (int i = 0; i < 10000 && !done; i++) nap(100);
  const bool went_on = done;
  d.release = true;
  t.join();
  u.join();
  CHECK(went_on);
  CHECK(got == a && d.syncs == 1);
  void *e = c.alloc(4096);  // b, freed during the wait, needs a sync of its own
  CHECK(e == b && d.syncs == 2);
  c.free(got);
  c.free(e);
  c.trim();
  CHECK(d.allocs == 3 && d.frees == 3);
}

// The same while a thread gives blocks back: one above the bound, and all of
// them in a trim.
static void nobody_waits_behind_a_free() {
  for (int trim = 0; trim < 2; trim++) {
    Device d;
    Cache c(Memory{&d}, 1 << 20, 8 << 20);
    void *big = c.alloc(2 << 20);
    c.free(c.alloc(4096));
    d.release = false;
    std::thread t([&] {
      if (trim) c.trim();
      else c.free(big);
    });
    while (!d.waiting) nap(20);
    std::atomic<bool> done{false};
    std::thread u([&] {
      c.free(c.alloc(100000));
      done = true;
    });
    for (int i = 0; i < 10000 && !done; i++) nap(100);
    const bool went_on = done;
    d.release = true;
    t.join();
    u.join();
    CHECK(went_on);
    if (trim) c.free(big);
    c.trim();
    CHECK(d.allocs == d.frees);
  }
}

// A block is less than 512 bytes larger than asked for; a kept block serves
// only requests of its size.
static void blocks_are_little_larger_than_asked() {
  Device d;
  Cache c(Memory{&d}, 384 << 20, (size_t)8 << 30);
  for (size_t n = 0; n < ((size_t)500 << 20); n = n * 9 / 8 + 37)
    for (size_t m : {n, n + 1, n / 512 * 512}) {
      const size_t s = c.size_of(m);
      CHECK(s >= m && s > 0 && (s < m + 512 || m == 0));
      CHECK(m > ((size_t)384 << 20) ? s == m : s % 512 == 0);
      CHECK(c.size_of(s) == s);
    }
  void *a = c.alloc(64 << 10);
  c.free(a);
  CHECK(c.kept() == 64 << 10);
  void *b = c.alloc(60 << 10);
  CHECK(b != a);
  void *e = c.alloc((64 << 10) - 100);
  CHECK(e == a);
  c.free(b);
  c.free(e);
  c.trim();
}

// Blocks above the bound are not kept, nor any past the total.
static void kept_memory_is_bounded() {
  Device d;
  Cache c(Memory{&d}, 1 << 20, 4 << 20);
  c.free(c.alloc((1 << 20) + 1));
  CHECK(c.kept() == 0 && d.frees == 1);
  std::vector<void *> v;
  for (int i = 0; i < 8; i++) v.push_back(c.alloc(1 << 20));
  for (void *p : v) c.free(p);
  CHECK(c.kept() == 4 << 20 && d.frees == 5);
  c.trim();
  CHECK(c.kept() == 0 && d.frees == 9);
}

// An allocation that fails is tried again without the kept blocks; if it
// fails again the caller hears of it and what it gives back is not kept.
static void failed_allocations_give_kept_blocks_back() {
  Device d;
  d.room = 8 << 20;
  Cache c(Memory{&d}, 2 << 20, 64 << 20);
  std::vector<void *> v;
  for (int i = 0; i < 6; i++) v.push_back(c.alloc(1 << 20));
  for (void *p : v) c.free(p);
  CHECK(c.kept() == 6 << 20 && d.frees == 0);
  void *a = c.alloc(7 << 20);  // fits only without them
  CHECK(c.kept() == 0 && d.frees == 6);
  void *b = c.alloc(1 << 20);
  bool failed = false;
  try {
    c.alloc(1 << 20);
  } catch (const std::bad_alloc &) {
    failed = true;
  }
  CHECK(failed);
  c.free(b);
  CHECK(c.kept() == 0 && d.frees == 7);
  c.free(c.alloc(1 << 20));  // works again, and is kept again
  CHECK(c.kept() == 1 << 20);
  c.free(a);
  c.trim();
  CHECK(d.allocs == d.frees);
}

// Threads that write their blocks and free them: no block has two owners, and
// all go back.
static void blocks_have_one_owner() {
  Device d;
  Cache c(Memory{&d}, 1 << 20, 8 << 20);
  std::vector<std::thread> ts;
  for (int i = 0; i < 4; i++)
    ts.emplace_back([&, i] {
      const size_t n = 1000 * (1 + i % 2);
      for (int k = 0; k < 3000; k++) {
        unsigned char *p = (unsigned char *)c.alloc(n);
        memset(p, i + 1, n);
        for (size_t j = 0; j < n; j++) CHECK(p[j] == i + 1);
        c.free(p);
      }
    });
  for (auto &t : ts) t.join();
  c.trim();
  CHECK(d.allocs == d.frees && c.kept() == 0);
}

int main(int argc, char **argv) {
  const struct {
    const char *name;
    void (*run)();
  } checks[] = {
      {"freed_blocks_wait_for_a_sync", freed_blocks_wait_for_a_sync},
      {"nobody_waits_behind_a_sync", nobody_waits_behind_a_sync},
      {"nobody_waits_behind_a_free", nobody_waits_behind_a_free},
      {"blocks_have_one_owner", blocks_have_one_owner},
      {"blocks_are_little_larger_than_asked", blocks_are_little_larger_than_asked},
      {"kept_memory_is_bounded", kept_memory_is_bounded},
      {"failed_allocations_give_kept_blocks_back", failed_allocations_give_kept_blocks_back},
  };
  for (auto &k : checks)
    if (argc == 2 && !strcmp(argv[1], k.name)) {
      k.run();
      return 0;
    }
  fprintf(stderr, "no such check\n");
  return 2;
}
