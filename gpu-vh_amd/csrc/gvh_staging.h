// gvh_staging.h -- results from device memory into a caller's host memory.
//
// The runtime moves pageable memory to the host at 17 GB/s on one core, 5 to
// 8 GB/s where the caller's pages are new, over a link that does 57.  Here large
// results come through pinned slots of 1 MiB that a kernel fills and four
// threads empty, so the link, the copies and the page faults overlap: into new
// pages 1.7 MB take 120 against 250 us, 4.2 MB 320 against 550, 33 MB 1.25
// against 6.9 ms (with the runtime's copies into the slots 1.4 ms; slots of 512
// KiB 1.8 ms; six threads 480 us for 4.2 MB).  Copies to the
// device gain nothing by it: the runtime reads pageable memory at 30 GB/s.
#pragma once
#include <hip/hip_runtime.h>

#include <condition_variable>
#include <cstddef>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

namespace gvh {

// One user at a time; work is ordered on the caller's stream and has ended
// when a call returns.  The pinned memory (8 MiB, and 64 KiB for small results)
// is allocated by the first call that needs it and freed with the object, as
// are the three threads beside the caller's; without it, below one slot, or
// into host memory that is pinned itself, the copies are the runtime's.  So is
// an object's first large result, unless it is larger than the slots: to pin
// them and to start the threads takes 0.8 ms, as much as 8 MiB take longer that
// way, and many objects give one such result only.
class Staging {
 public:
  Staging() = default;
  Staging(const Staging &) = delete;
  Staging &operator=(const Staging &) = delete;
  ~Staging();
  hipError_t to_host(void *host, const void *dev, size_t bytes, hipStream_t st);
  // Pinned memory that kernels on the device can write, for a result of at
  // most SMALL bytes; nullptr if there is none.
  void *small(size_t bytes);

  static constexpr size_t SMALL = 1 << 16, SLOT = 1 << 20;
  static constexpr int NSLOT = 8, MAX_THREADS = 4;

 private:
  struct Job;
  bool ready();
  void work();
  hipError_t pipeline(char *host, const char *dev, size_t bytes, hipStream_t st);
  char *mem_ = nullptr;  // the slots, then a flag for each
  char *small_ = nullptr;
  bool failed_ = false, used_ = false;
  unsigned *arrived_ = nullptr;  // per slot, blocks that have their part there
  std::vector<std::thread> pool_;
  std::mutex mutex_;
  std::condition_variable wake_;
  std::shared_ptr<Job> job_;  // the result on its way
  bool quit_ = false;
};

}  // namespace gvh
