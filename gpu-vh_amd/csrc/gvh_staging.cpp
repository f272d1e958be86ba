// gvh_staging.cpp -- see gvh_staging.h.
#include "gvh_staging.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <thread>
#include <vector>

namespace gvh {

namespace {

// Pinned (or device) memory that the runtime copies to and from directly.
bool is_pinned(const void *p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return a.type == hipMemoryTypeHost || a.type == hipMemoryTypeDevice;
}

}  // namespace

Staging::~Staging() {
  for (hipEvent_t e : ev_)
    if (e) (void)hipEventDestroy(e);
  if (mem_) (void)hipHostFree(mem_);
  if (small_) (void)hipHostFree(small_);
}

void *Staging::small(size_t bytes) {
  if (bytes > SMALL) return nullptr;
  if (!small_ && hipHostMalloc((void **)&small_, SMALL) != hipSuccess) {
    (void)hipGetLastError();
    small_ = nullptr;
  }
  return small_;
}

bool Staging::ready() {
  if (mem_ || failed_) return mem_ != nullptr;
  bool ok = true;
  for (hipEvent_t &e : ev_)
    if (!e) ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
  ok = ok && hipHostMalloc((void **)&mem_, NSLOT * SLOT) == hipSuccess;
  if (!ok) {
    (void)hipGetLastError();
    mem_ = nullptr;
    failed_ = true;
  }
  return ok;
}

// Chunks of SLOT bytes go round the slots.  The calling thread issues the
// device copies and waits for their events; it and the others each copy their
// share of a chunk from its slot.  `open` counts the chunks that have arrived,
// done[c] the shares of chunk c that are copied.
hipError_t Staging::pipeline(char *host, const char *dev, size_t bytes, hipStream_t st) {
  const int n = (int)((bytes + SLOT - 1) / SLOT);
  const int nt = std::max(1, std::min({MAX_THREADS, n, (int)std::thread::hardware_concurrency()}));
  std::atomic<int> open{0};
  std::atomic<bool> stop{false};
  std::vector<std::atomic<int>> done(n);
  for (auto &d : done) d = 0;
  auto length = [&](int c) { return std::min(SLOT, bytes - (size_t)c * SLOT); };
  std::atomic<int> threads{1};  // that take part; fixed before the first chunk opens
  auto share = [&](int c, int t) {
    const size_t len = length(c), part = (len / threads + 63) / 64 * 64;
    const size_t a = std::min(len, part * t), b = t == threads - 1 ? len : std::min(len, part * (t + 1));
    if (a < b)
      std::memcpy(host + (size_t)c * SLOT + a, mem_ + (size_t)(c % NSLOT) * SLOT + a, b - a);
    done[c].fetch_add(1, std::memory_order_release);
  };
  auto work = [&](int t) {
    for (int c = 0; c < n; ++c) {
      while (open.load(std::memory_order_acquire) <= c) {
        if (stop) return;
        std::this_thread::yield();
      }
      share(c, t);
    }
  };
  std::vector<std::thread> pool;
  pool.reserve(nt);
  try {
    for (int t = 1; t < nt; ++t) pool.emplace_back(work, t);
  } catch (...) {  // no more threads: those that started take part
  }
  threads = (int)pool.size() + 1;
  auto finish = [&](int c) {
    while (done[c].load(std::memory_order_acquire) < threads) std::this_thread::yield();
  };
  hipError_t e = hipSuccess;
  int issued = 0;
  for (int c = 0; c < n && e == hipSuccess; ++c) {
    for (; issued < n && issued < c + NSLOT && e == hipSuccess; ++issued) {
      if (issued >= NSLOT) finish(issued - NSLOT);
      e = hipMemcpyAsync(mem_ + (size_t)(issued % NSLOT) * SLOT, dev + (size_t)issued * SLOT,
                         length(issued), hipMemcpyDeviceToHost, st);
      if (e == hipSuccess) e = hipEventRecord(ev_[issued % NSLOT], st);
    }
    if (e == hipSuccess) e = hipEventSynchronize(ev_[c % NSLOT]);
    if (e != hipSuccess) break;
    open.store(c + 1, std::memory_order_release);
    share(c, 0);
  }
  if (e == hipSuccess)
    for (int c = std::max(0, n - NSLOT); c < n; ++c) finish(c);
  stop = true;
  for (std::thread &t : pool) t.join();
  const hipError_t s = hipStreamSynchronize(st);
  return e == hipSuccess ? s : e;
}

hipError_t Staging::to_host(void *host, const void *dev, size_t bytes, hipStream_t st) {
  if (bytes >= SLOT && !is_pinned(host) && ready()) {
    try {
      return pipeline(static_cast<char *>(host), static_cast<const char *>(dev), bytes, st);
    } catch (...) {  // no memory for its bookkeeping, before anything was issued
    }
  }
  const hipError_t e = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, st);
  return e == hipSuccess ? hipStreamSynchronize(st) : e;
}

}  // namespace gvh
