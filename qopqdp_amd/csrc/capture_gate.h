// Keeps stream captures and device synchronisations apart.  The device must
// not be synchronised while any of its streams is being captured, whichever
// thread captures (thread-local capture mode relaxes only the calls of other
// threads that do not wait for the device).  A capture records host calls
// only, so its window is short; a synchronisation lasts as long as the work
// on the device.
#pragma once
#include <condition_variable>
#include <mutex>

namespace qop {

class CaptureGate {
 public:
  // Before a capture begins: waits for synchronisations in progress.
  void capture_begin() {
    std::unique_lock<std::mutex> lk(mu_);
    cv_.wait(lk, [&] { return syncing_ == 0; });
    capturing_++;
  }
  void capture_end() {
    std::lock_guard<std::mutex> lk(mu_);
    capturing_--;
    cv_.notify_all();
  }
  // Before a device synchronisation: waits for captures in progress, or with
  // wait false gives up (false) when there is one.  The caller must not be
  // capturing itself if it waits.
  bool sync_begin(bool wait) {
    std::unique_lock<std::mutex> lk(mu_);
    if (!wait && capturing_ > 0) return false;
    cv_.wait(lk, [&] { return capturing_ == 0; });
    syncing_++;
    return true;
  }
  void sync_end() {
    std::lock_guard<std::mutex> lk(mu_);
    syncing_--;
    cv_.notify_all();
  }

 private:
  std::mutex mu_;
  std::condition_variable cv_;
  int capturing_ = 0, syncing_ = 0;
};

}  // namespace qop
