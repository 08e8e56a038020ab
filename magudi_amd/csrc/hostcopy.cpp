// hostcopy.cpp -- large copies between device memory and a caller's pageable array.
//
// The runtime's own pageable device-to-host copy moves the data with one thread, which also
// takes the page faults of a fresh destination: 10 GB/s.  Here chunks of 2 MiB (the huge page
// that backs large arrays, so no two threads fault on one) arrive in pinned slots and several
// threads copy them out, into a fresh array: 671 MB 64 -> 16.8 ms, 41 MB 4.0 -> 1.3 ms, 8.4 MB
// 0.48 -> 0.32 ms, 5.2 MB 0.29 -> 0.22 ms.  Below kLeast the threads cost more than they save
// (2.4 MB, with the array's allocation, 0.56 -> 0.63 ms).
// The slots are as many as a copy needs, sixteen at most: pinning them takes 0.1 ms per MB
// once.  Host-to-device copies have no faults to share and stay as they are.
#include "hostcopy.h"

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <thread>

namespace mgd {

namespace {
constexpr size_t kLeast = size_t(4) << 20;
constexpr unsigned kMostThreads = 8;

// Copies of all regions in progress.  Small ones beside each other have threads enough of their
// own (4 x 5.2 MB at once 0.6 ms plain, 1.1 through the rings; 16 x 5.2 MB 2.2 and 3.5); large
// ones gain until they fill the link, and lose little then (4 x 41 MB 5.3 and 4.7, 16 x 41 MB 16.4
// and 18, 16 x 164 MB 64 both ways).
constexpr size_t kLeastBeside = size_t(32) << 20;
std::atomic<int> g_copies{0};
struct Copying {
  const int others = g_copies.fetch_add(1);
  ~Copying() { g_copies.fetch_sub(1); }
};

// Whether the runtime knows the destination (pinned, managed or device memory): a copy there is
// one transfer at the link's rate, without faults (671 MB 11.8 ms, 16.6 through the ring).
bool registered(const void* p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return a.type != hipMemoryTypeUnregistered;
}
}  // namespace

HostCopy::~HostCopy() {
  for (hipEvent_t e : ev_)
    if (e) (void)hipEventDestroy(e);
  if (buf_) (void)hipHostFree(buf_);
}

bool HostCopy::prepare(int slots, hipStream_t st) {
  if (slots_ >= slots) return true;
  if (failed_) return false;
  // events are recorded on the stream's device, which need not be the caller's current one
  int current = 0;
  hipDevice_t device = 0;
  if (hipGetDevice(&current) != hipSuccess || hipStreamGetDevice(st, &device) != hipSuccess ||
      (current != device && hipSetDevice(device) != hipSuccess)) {
    (void)hipGetLastError();
    return false;
  }
  const bool ok = make(slots);
  if (current != device) (void)hipSetDevice(current);
  return ok;
}

bool HostCopy::make(int slots) {
  if (buf_) (void)hipHostFree(buf_);
  buf_ = nullptr;
  slots_ = 0;
  void* p = nullptr;
  bool ok = hipHostMalloc(&p, kChunk * slots, hipHostMallocDefault) == hipSuccess;
  for (hipEvent_t& e : ev_) ok = ok && (e || hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess);
  if (!ok) {
    (void)hipGetLastError();     // no pinned memory left: plain copies from here on
    if (p) (void)hipHostFree(p);
    failed_ = true;
    return false;
  }
  buf_ = static_cast<char*>(p);
  slots_ = slots;
  return true;
}

hipError_t HostCopy::to_host(void* host, const void* dev, size_t bytes, hipStream_t st) {
  // chunk c covers [edge(c), edge(c + 1)): the first one ends at a chunk boundary of the address
  const size_t first = kChunk - reinterpret_cast<uintptr_t>(host) % kChunk;
  const long n = bytes > first ? 1 + (long)((bytes - first + kChunk - 1) / kChunk) : 1;
  auto edge = [&](long c) { return c == 0 ? size_t(0) : std::min(bytes, first + (size_t)(c - 1) * kChunk); };
  const unsigned cpus = std::thread::hardware_concurrency();
  const unsigned want = (unsigned)std::min<long>(n, std::min(kMostThreads, cpus / 2));
  const int slots = (int)std::min<long>(n, kMostSlots);
  const Copying now;
  const bool beside = now.others == 0 || bytes >= kLeastBeside;
  if (bytes < kLeast || want < 2 || !beside || registered(host) || !prepare(slots, st)) {
    const hipError_t e = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, st);
    return e != hipSuccess ? e : hipStreamSynchronize(st);
  }
  char* const dst = static_cast<char*>(host);
  const char* const src = static_cast<const char*>(dev);
  std::atomic<long> arrived{0};            // chunks in their slots
  std::atomic<bool> stop{false};
  std::mutex mu;                           // the threads sleep until the first chunk is there: it
  std::condition_variable cv;              // comes after all other work on the stream
  unsigned threads = 0;                    // set then, and once all have started
  std::atomic<long> copied[kMostThreads];  // chunks that each thread has finished
  for (auto& c : copied) c.store(0);
  auto work = [&](unsigned t) {
    unsigned T;
    {
      std::unique_lock<std::mutex> lock(mu);
      cv.wait(lock, [&] { return threads != 0; });
      T = threads;
    }
    for (long c = t; c < n; c += T) {
      while (arrived.load(std::memory_order_acquire) <= c) {
        if (stop.load(std::memory_order_relaxed)) return;
        std::this_thread::yield();
      }
      std::memcpy(dst + edge(c), buf_ + (c % slots) * kChunk, edge(c + 1) - edge(c));
      copied[t].fetch_add(1, std::memory_order_release);
    }
  };
  std::thread pool[kMostThreads];
  unsigned T = 0;
  try {
    for (; T < want; ++T) pool[T] = std::thread(work, T);
  } catch (...) {                          // no thread or no memory: as many as there are
  }
  if (T == 0) {
    const hipError_t e = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, st);
    return e != hipSuccess ? e : hipStreamSynchronize(st);
  }
  auto wake = [&] {
    {
      std::lock_guard<std::mutex> lock(mu);
      threads = T;
    }
    cv.notify_all();
  };
  hipError_t err = hipSuccess;
  auto fetch = [&](long c) {               // chunk c into its slot
    err = hipMemcpyAsync(buf_ + (c % slots) * kChunk, src + edge(c), edge(c + 1) - edge(c),
                         hipMemcpyDeviceToHost, st);
    if (err == hipSuccess) err = hipEventRecord(ev_[c % slots], st);
  };
  for (long c = 0; c < slots && err == hipSuccess; ++c) fetch(c);
  for (long c = 0; c < n && err == hipSuccess; ++c) {
    err = hipEventSynchronize(ev_[c % slots]);
    if (err != hipSuccess) break;
    arrived.store(c + 1, std::memory_order_release);
    if (c == 0) wake();
    // the slot of a chunk half a ring back is free once its thread has copied it out
    const long b = c - slots / 2;
    if (b >= 0 && b + slots < n) {
      while (copied[b % T].load(std::memory_order_acquire) <= b / T) std::this_thread::yield();
      fetch(b + slots);
    }
  }
  if (err != hipSuccess) {
    stop.store(true);
    wake();
  }
  for (unsigned t = 0; t < T; ++t) pool[t].join();
  if (err != hipSuccess) (void)hipStreamSynchronize(st);   // no copy into the slots is left behind
  return err;
}

}  // namespace mgd
