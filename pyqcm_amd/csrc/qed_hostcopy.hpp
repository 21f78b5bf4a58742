// A host copy by several threads, for pages that are often touched for the first time.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstring>
#include <system_error>
#include <thread>
#include <vector>

namespace qed {

// Threads worth starting for a copy of this size: none below 8 MB, and no more than there
// are cores (hardware_concurrency() is 0 where it is not known).
inline int copy_threads(size_t bytes) {
  if (bytes < (size_t(8) << 20)) return 1;
  const int cores = (int)std::thread::hardware_concurrency();
  return cores > 0 ? std::min(cores, 8) : 1;
}

// Copies len bytes by up to nt threads, the caller's among them. Where a thread cannot be
// started, the caller copies the rest itself.
inline void copy_parallel(unsigned char* dst, const unsigned char* src, size_t len, int nt) {
  struct Joined : std::vector<std::thread> {
    ~Joined() {
      for (auto& t : *this) t.join();
    }
  } threads;
  const size_t per = ((len + nt - 1) / nt + 4095) & ~size_t(4095);
  threads.reserve(nt);
  size_t end = len;  // the caller's part is [0, end): the threads take pieces off its end
  try {
    for (size_t o = per ? (len - (len > 0)) / per * per : 0; o > 0; o -= per) {
      threads.emplace_back([=] { std::memcpy(dst + o, src + o, std::min(per, len - o)); });
      end = o;
    }
  } catch (const std::system_error&) {
  }
  std::memcpy(dst, src, end);
}

}  // namespace qed
