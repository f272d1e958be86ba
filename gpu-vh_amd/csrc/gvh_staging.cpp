// gvh_staging.cpp -- see gvh_staging.h.
#include "gvh_staging.h"

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>

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

// A wait of microseconds, as one for another thread's copy is.  It spins, a
// millisecond at most, before it yields.
class Wait {
 public:
  void operator()() {
    if (++n_ < 16384) {
      __builtin_ia32_pause();
    } else {
      n_ = 0;
      std::this_thread::yield();
    }
  }

 private:
  int n_ = 0;
};

}  // namespace

// A result on its way: chunk c has arrived in its slot once open > c, and its
// PARTS parts are copied by whichever thread takes them.
struct Staging::Job {
  static constexpr int PARTS = 4;
  char *host, *slots;
  size_t bytes;
  int n;
  std::vector<std::atomic<int>> copied;  // of each chunk's parts
  std::atomic<int> open{0}, next{0}, total{0};
  std::atomic<bool> over{false};

  Job(char *h, char *m, size_t b, int chunks) : host(h), slots(m), bytes(b), n(chunks), copied(chunks) {
    for (auto &c : copied) c = 0;
  }
  size_t length(int c) const { return std::min(SLOT, bytes - (size_t)c * SLOT); }
  // Copies one part that has arrived; false if there is none left to take.
  bool copy_one() {
    int i = next.load(std::memory_order_relaxed);
    do {
      if (i >= open.load(std::memory_order_acquire) * PARTS) return false;
    } while (!next.compare_exchange_weak(i, i + 1, std::memory_order_acq_rel));
    const int c = i / PARTS, t = i % PARTS;
    const size_t len = length(c), part = (len / PARTS + 63) / 64 * 64;
    const size_t a = std::min(len, part * t), b = t == PARTS - 1 ? len : std::min(len, part * (t + 1));
    if (a < b) std::memcpy(host + (size_t)c * SLOT + a, slots + (size_t)(c % NSLOT) * SLOT + a, b - a);
    copied[c].fetch_add(1, std::memory_order_release);
    total.fetch_add(1, std::memory_order_release);
    return true;
  }
};

// A thread of the pool: sleeps until there is a result on its way.
void Staging::work() {
  std::shared_ptr<Job> last;
  while (true) {
    std::shared_ptr<Job> job;
    {
      std::unique_lock<std::mutex> lock(mutex_);
      wake_.wait(lock, [&] { return quit_ || (job_ && job_ != last); });
      if (quit_) return;
      job = job_;
    }
    Wait wait;
    while (!job->over.load(std::memory_order_acquire))
      if (!job->copy_one()) wait();
    last = job;
  }
}

Staging::~Staging() {
  {
    std::lock_guard<std::mutex> lock(mutex_);
    quit_ = true;
  }
  wake_.notify_all();
  for (std::thread &t : pool_) t.join();
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
// kernels, watches for their flags and copies parts of what has arrived; the
// pool's threads copy too, as soon as they run.  It depends on none of them: a
// thread may first run at the system's next tick, where threads that were each
// given a share of every chunk made 4.8 MB take 2.9 ms instead of 0.4.  (With
// the runtime's copies and events, a thread of the runtime stays busy for
// milliseconds afterwards, and a program whose threads fill the CPUs waits for
// it.)
hipError_t Staging::pipeline(char *host, const char *dev, size_t bytes, hipStream_t st) {
  const int n = (int)((bytes + SLOT - 1) / SLOT);
  const auto job = std::make_shared<Job>(host, mem_, bytes, n);
  try {
    const int threads = std::min(MAX_THREADS, (int)std::thread::hardware_concurrency()) - 1;
    while ((int)pool_.size() < threads) pool_.emplace_back(&Staging::work, this);
  } catch (...) {  // no more threads: those that started take part
  }
  {
    std::lock_guard<std::mutex> lock(mutex_);
    job_ = job;
  }
  wake_.notify_all();
  hipError_t e = hipSuccess;
  unsigned *flags = reinterpret_cast<unsigned *>(mem_ + NSLOT * SLOT);
  auto arrived = [&](int c) { return __atomic_load_n(flags + c % NSLOT, __ATOMIC_ACQUIRE) != 0u; };
  auto emptied = [&](int c) { return job->copied[c].load(std::memory_order_acquire) == Job::PARTS; };
  int issued = 0, open = 0, polls = 0;
  Wait wait;
  while (e == hipSuccess && job->total.load(std::memory_order_acquire) < n * Job::PARTS) {
    if (issued < n && issued < open + NSLOT && (issued < NSLOT || emptied(issued - NSLOT))) {
      const int k = issued % NSLOT;
      const char *src = dev + (size_t)issued * SLOT;
      const unsigned words = (unsigned)(job->length(issued) / 4);
      __atomic_store_n(flags + k, 0u, __ATOMIC_RELEASE);
      chunk_kernel<<<CHUNK_BLOCKS, 256, 0, st>>>(
          reinterpret_cast<const unsigned *>(src), reinterpret_cast<unsigned *>(mem_ + k * SLOT), words,
          reinterpret_cast<uintptr_t>(src) % 16 == 0 ? words / 4 : 0u, arrived_ + k, flags + k);
      e = hipGetLastError();
      ++issued;
    } else if (open < issued && arrived(open)) {
      job->open.store(++open, std::memory_order_release);
      polls = 0;
    } else if (job->copy_one()) {
      polls = 0;
    } else if (open == issued) {  // others copy the last parts
      wait();
    } else if (++polls % 4096 == 0) {
      // the stream tells of a failed kernel, whose flag would never come
      const hipError_t q = hipStreamQuery(st);
      if (q == hipSuccess && !arrived(open)) e = hipErrorUnknown;
      else if (q != hipSuccess && q != hipErrorNotReady) e = q;
    }
  }
  // no part is taken from here on; those that are taken end
  const int taken = job->next.exchange(n * Job::PARTS);
  while (job->total.load(std::memory_order_acquire) < taken) wait();
  job->over.store(true, std::memory_order_release);
  {
    std::lock_guard<std::mutex> lock(mutex_);
    job_.reset();
  }
  const hipError_t s = hipStreamSynchronize(st);
  return e == hipSuccess ? s : e;
}

hipError_t Staging::to_host(void *host, const void *dev, size_t bytes, hipStream_t st) {
  const bool large = bytes >= SLOT && bytes % 4 == 0 && !is_pinned(host);
  const bool pays = used_ || bytes > NSLOT * SLOT;
  used_ = used_ || large;
  if (large && pays && ready()) {
    try {
      return pipeline(static_cast<char *>(host), static_cast<const char *>(dev), bytes, st);
    } catch (...) {  // no memory for its bookkeeping, before anything was issued
    }
  }
  const hipError_t e = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, st);
  return e == hipSuccess ? hipStreamSynchronize(st) : e;
}

}  // namespace gvh
