// gvh_staging.cpp -- see gvh_staging.h.
#include "gvh_staging.h"

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <thread>
#include <vector>

namespace gvh {

namespace {

constexpr int CHUNK_BLOCKS = 32;

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
  if (arrived_) (void)hipFree(arrived_);
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
  bool ok = hipHostMalloc((void **)&mem_, NSLOT * SLOT + sizeof(unsigned) * NSLOT,
                          hipHostMallocCoherent) == hipSuccess;
  ok = ok && hipMalloc((void **)&arrived_, sizeof(unsigned) * NSLOT) == hipSuccess;
  ok = ok && hipMemset(arrived_, 0, sizeof(unsigned) * NSLOT) == hipSuccess &&
       hipStreamSynchronize(nullptr) == hipSuccess;
  if (!ok) {
    if (mem_) (void)hipHostFree(mem_);
    (void)hipGetLastError();
    mem_ = nullptr;
    failed_ = true;
  }
  return ok;
}

// One chunk of 4-byte words into its slot; the last block to have its part
// there tells the host.  16-byte stores where the chunk's start allows them:
// its words from `n4` 16-byte groups on go one by one.
__global__ __launch_bounds__(256) void chunk_kernel(const unsigned *__restrict__ src,
                                                    unsigned *__restrict__ slot, unsigned words,
                                                    unsigned n4, unsigned *__restrict__ arrived,
                                                    unsigned *__restrict__ flag) {
  const unsigned t = blockIdx.x * 256 + threadIdx.x, nt = gridDim.x * 256;
  for (unsigned i = t; i < n4; i += nt)
    reinterpret_cast<uint4 *>(slot)[i] = reinterpret_cast<const uint4 *>(src)[i];
  for (unsigned i = 4 * n4 + t; i < words; i += nt) slot[i] = src[i];
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x == 0 && atomicAdd(arrived, 1u) == gridDim.x - 1) {
    *arrived = 0;
    __hip_atomic_store(flag, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// Chunks of SLOT bytes go round the slots.  The calling thread launches their
// kernels and waits for their flags; it and the others each copy their share
// of a chunk from its slot.  `open` counts the chunks that have arrived,
// done[c] the shares of chunk c that are copied.  (With the runtime's copies
// and events instead, a thread of the runtime stays busy for milliseconds
// afterwards, and a program whose threads fill the CPUs waits for it.)
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
  unsigned *flags = reinterpret_cast<unsigned *>(mem_ + NSLOT * SLOT);
  auto set = [&](int c) { return __atomic_load_n(flags + c % NSLOT, __ATOMIC_ACQUIRE) != 0u; };
  int issued = 0;
  for (int c = 0; c < n && e == hipSuccess; ++c) {
    for (; issued < n && issued < c + NSLOT && e == hipSuccess; ++issued) {
      if (issued >= NSLOT) finish(issued - NSLOT);
      const int k = issued % NSLOT;
      const char *src = dev + (size_t)issued * SLOT;
      const unsigned words = (unsigned)(length(issued) / 4);
      __atomic_store_n(flags + k, 0u, __ATOMIC_RELEASE);
      chunk_kernel<<<CHUNK_BLOCKS, 256, 0, st>>>(
          reinterpret_cast<const unsigned *>(src), reinterpret_cast<unsigned *>(mem_ + k * SLOT), words,
          reinterpret_cast<uintptr_t>(src) % 16 == 0 ? words / 4 : 0u, arrived_ + k, flags + k);
      e = hipGetLastError();
    }
    // the stream tells of a failed kernel, whose flag would never come
    for (int polls = 1; e == hipSuccess && !set(c); ++polls) {
      if (polls % 4096 == 0) {
        const hipError_t q = hipStreamQuery(st);
        if (q == hipSuccess && !set(c)) e = hipErrorUnknown;
        else if (q != hipSuccess && q != hipErrorNotReady) e = q;
      }
    }
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
  if (bytes >= SLOT && bytes % 4 == 0 && !is_pinned(host) && ready()) {
    try {
      return pipeline(static_cast<char *>(host), static_cast<const char *>(dev), bytes, st);
    } catch (...) {  // no memory for its bookkeeping, before anything was issued
    }
  }
  const hipError_t e = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, st);
  return e == hipSuccess ? hipStreamSynchronize(st) : e;
}

}  // namespace gvh
