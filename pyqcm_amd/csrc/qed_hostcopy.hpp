// A host copy that other threads help with.
#pragma once

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>

namespace qed {

// Makes the caller's pages of [p, p + len) present without changing them: 5 ms for 128 MB of
// fresh pages by one thread, which a call can spend while the device computes.
inline void touch_pages(unsigned char* p, size_t len) {
  volatile unsigned char* v = p;
  for (size_t i = 0; i < len; i += 4096) v[i] = v[i];
  if (len) v[len - 1] = v[len - 1];
}

// Threads that wait for copies to help with. The caller copies too, block by block, and waits
// only for blocks that a helper has begun: a helper that has not been scheduled, could not be
// started or is gone after a fork costs nothing. After a parallel section of the caller's
// program its threads may spin on every core for some 60 ms: threads started for each 16 MB
// piece then took a time slice of 4 ms each to begin, 30 ms for 128 MB where this takes 4 to
// 10 (and 1.6 on idle cores).
class CopyHelpers {
 public:
  // never destroyed: the helpers wait in it until the process ends
  static CopyHelpers& get() {
    static auto* h = new CopyHelpers();
    return *h;
  }
  void copy(unsigned char* dst, const unsigned char* src, size_t len) {
    std::unique_lock<std::mutex> mine(calls_, std::try_to_lock);
    if (!mine || len < (size_t(8) << 20)) {  // helpers are busy with another call, or not worth waking
      std::memcpy(dst, src, len);
      return;
    }
    std::unique_lock<std::mutex> lk(mu_);
    start();
    dst_ = dst;
    src_ = src;
    len_ = len;
    next_ = 0;
    ++busy_;
    wake_.notify_all();
    work(lk);
    done_.wait(lk, [&] { return busy_ == 0; });
  }

 private:
  static constexpr size_t kBlock = size_t(512) << 10;
  // the helpers of this process, on its first copy: as many as there are other cores, seven at most
  void start() {
    if (started_) return;
    started_ = true;
    const int n = std::min(8, (int)std::thread::hardware_concurrency());  // 0 where it is not known
    try {
      for (int t = 1; t < n; ++t) std::thread([this] { help(); }).detach();
    } catch (const std::system_error&) {
    }
  }
  void help() {
    std::unique_lock<std::mutex> lk(mu_);
    for (;;) {
      wake_.wait(lk, [&] { return next_ < len_; });
      ++busy_;
      work(lk);
    }
  }
  // the blocks that are left; lk is held on entry and exit, not during a copy. What a copy is
  // of changes only while busy_ is 0.
  void work(std::unique_lock<std::mutex>& lk) {
    lk.unlock();
    for (size_t o = next_.fetch_add(kBlock); o < len_; o = next_.fetch_add(kBlock))
      std::memcpy(dst_ + o, src_ + o, std::min(kBlock, len_ - o));
    lk.lock();
    if (--busy_ == 0) done_.notify_all();
  }
  std::mutex calls_, mu_;
  std::condition_variable wake_, done_;
  unsigned char* dst_ = nullptr;
  const unsigned char* src_ = nullptr;
  size_t len_ = 0;
  std::atomic<size_t> next_{0};
  int busy_ = 0;  // threads inside a copy
  bool started_ = false;
};

}  // namespace qed
