// Block cache of dev_alloc / dev_free and host_alloc / host_free.
//
// Solves, link construction and forces take their workspaces at every call;
// hipMalloc and hipFree of a few GB take tens of milliseconds (one asqtad link
// construction at 24^3x48: 8.5 ms of kernels in a 69 ms call), so freed blocks
// are kept and handed out again.
//  * A freed block may still be in use by work enqueued on any stream.  It is
//    pending until a device synchronisation after its free (hipFree waits for
//    the device too) and only then handed out, so a block never passes from
//    one stream or thread to another with work in flight.  The waiting thread
//    holds no lock, here and in the calls of Api: the others allocate and free
//    meanwhile.  Where the device
//    cannot be synchronised now, pending blocks stay pending and a new block
//    is allocated.
//  * Bounded: blocks above `block` bytes go back to the driver at once (the
//    largest kept are the 302 MB matrix fields of 32^3x64), and the kept blocks
//    total at most `total` bytes.  A call on a larger lattice pays for its
//    allocations: little while the card has memory the driver has already
//    cleared, then about 1 s for 35 to 50 GB (asqtad force at 40^3x64, 15 GB
//    of workspace: 81 ms and 430 to 510 ms).
//  * Given back: at QOP_finalize, when a request server ends, and when
//    an allocation fails (it is tried again then, and if it still fails the
//    blocks freed while the failure unwinds are not kept).
//
// Api is the memory behind it (runtime.cpp: HIP device or page-locked memory):
//   int device();                  // the device blocks are allocated on
//   void *alloc(size_t bytes);     // null: out of memory
//   void free(void *p);            // waits for the work that uses p
//   bool try_sync();               // waits for all work of the device; false: not possible now
//   [[noreturn]] void out_of_memory(size_t bytes);
#pragma once
#include <cstddef>
#include <map>
#include <mutex>

namespace qop {

template <class Api>
class BlockCache {
  struct Block {
    size_t bytes;
    int dev;
  };
  struct KeptBlock {
    void *p;
    int dev;
    unsigned long freed;  // epoch of its free
  };
  using Kept = std::multimap<size_t, KeptBlock>;

 public:
  BlockCache(Api api, size_t block, size_t total) : api_(api), block_(block), total_(total) {}
  void *alloc(size_t bytes) {
    const int dev = api_.device();
    const size_t want = size_of(bytes);
    std::unique_lock<std::mutex> lk(mu_);
    void *p = nullptr;
    if (want <= block_) {
      p = take(ready_, dev, want);
      if (!p && fits(pending_, dev, want)) {
        // other threads allocate and free meanwhile; what they free from here
        // on is not settled by this synchronisation
        const unsigned long before = ++epoch_;
        lk.unlock();
        const bool idle = api_.try_sync();
        lk.lock();
        if (idle) settle(dev, before);
        p = take(ready_, dev, want);
      }
    }
    if (!p) {
      lk.unlock();
      p = api_.alloc(want);
      if (!p) {
        trim();
        p = api_.alloc(want);
      }
      lk.lock();
      if (!p) {
        failed_ = true;
        api_.out_of_memory(bytes);
      }
      if (want <= block_) live_[p] = Block{want, dev};
    }
    failed_ = false;
    return p;
  }
  void free(void *p) {
    if (!p) return;
    std::unique_lock<std::mutex> lk(mu_);
    auto it = live_.find(p);
    if (it == live_.end() || failed_ || kept_ + it->second.bytes > total_) {
      if (it != live_.end()) live_.erase(it);
      lk.unlock();
      api_.free(p);
      return;
    }
    kept_ += it->second.bytes;
    pending_.emplace(it->second.bytes, KeptBlock{p, it->second.dev, epoch_});
    live_.erase(it);
  }
  // When it returns, what was kept at the call has gone back, also where
  // another thread's trim had taken it.
  void trim() {
    std::lock_guard<std::mutex> tk(trim_mu_);
    Kept ready, pending;
    {
      std::lock_guard<std::mutex> lk(mu_);
      ready.swap(ready_);
      pending.swap(pending_);
      kept_ = 0;
    }
    for (Kept *k : {&ready, &pending})
      for (auto &b : *k) api_.free(b.second.p);
  }
  // What an allocation of `bytes` takes: whole units of 512 bytes.  Calls come
  // back with the same sizes, so blocks need not serve nearby ones, and a
  // caller's count of what it allocates holds.
  size_t size_of(size_t bytes) const {
    const size_t n = bytes ? (bytes + 511) / 512 * 512 : 512;
    return n <= block_ ? n : bytes;
  }
  size_t kept() {
    std::lock_guard<std::mutex> lk(mu_);
    return kept_;
  }

 private:
  // a kept block of `want` bytes
  static typename Kept::iterator find(Kept &k, int dev, size_t want) {
    for (auto it = k.lower_bound(want); it != k.end() && it->first == want; ++it)
      if (it->second.dev == dev) return it;
    return k.end();
  }
  static bool fits(Kept &k, int dev, size_t want) { return find(k, dev, want) != k.end(); }
  void *take(Kept &k, int dev, size_t want) {
    auto it = find(k, dev, want);
    if (it == k.end()) return nullptr;
    void *p = it->second.p;
    live_[p] = Block{it->first, dev};
    kept_ -= it->first;
    k.erase(it);
    return p;
  }
  // the blocks freed before a synchronisation of their device began
  void settle(int dev, unsigned long before) {
    for (auto it = pending_.begin(); it != pending_.end();) {
      if (it->second.dev == dev && it->second.freed < before) {
        ready_.insert(*it);
        it = pending_.erase(it);
      } else {
        ++it;
      }
    }
  }
  Api api_;
  const size_t block_, total_;
  std::mutex mu_, trim_mu_;
  Kept ready_, pending_;
  std::map<void *, Block> live_;
  size_t kept_ = 0;
  unsigned long epoch_ = 0;
  bool failed_ = false;  // the last allocation failed: its frees are not kept
};

}  // namespace qop
