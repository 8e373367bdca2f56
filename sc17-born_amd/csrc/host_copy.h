// host_copy.h -- large copies from the device to pageable host arrays.
//
// On pageable memory hipMemcpyAsync transfers to a pinned buffer and one
// thread empties it: that thread is the bound (17 GB/s for 16 MB; into the
// device, where the runtime pins the caller's pages, 37 GB/s).  Here a few
// threads empty a ring of pinned slots that the transfers fill in turn.
#ifndef BORN_HOST_COPY_H
#define BORN_HOST_COPY_H

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

#include "host_par.h"

namespace born {

class HostCopy {
 public:
  HostCopy() = default;
  HostCopy(const HostCopy &) = delete;
  HostCopy &operator=(const HostCopy &) = delete;

  // host <- dev, ordered on the stream, complete on return
  hipError_t out(void *host, const void *dev, size_t bytes, hipStream_t stream) {
    if (bytes >= kMin && pageable(host) && ring()) {
      bool ran = false;
      const hipError_t e = staged((char *)host, (const char *)dev, bytes, stream, &ran);
      if (ran || e != hipSuccess) return e;
    }
    const hipError_t e = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, stream);
    return e != hipSuccess ? e : hipStreamSynchronize(stream);
  }

  // with no copy in flight
  void release() {
    for (hipEvent_t &e : ev_) {
      if (e) (void)hipEventDestroy(e);
      e = nullptr;
    }
    if (ring_) (void)hipHostFree(ring_);
    ring_ = nullptr;
  }

 private:
  // A transfer costs about 14 us besides its bytes at 55 GB/s: slots of 2 MB.
  // The host share of a slot is split in pieces for the threads.
  static constexpr size_t kSlot = (size_t)2 << 20, kPiece = (size_t)256 << 10;
  static constexpr long kSlots = 4, kPieces = kSlot / kPiece;
  static constexpr int kThreads = 4;
  // below, the threads cost what they gain
  static constexpr size_t kMin = 2 * kSlot;

  // memory that the runtime knows (pinned, managed, device) is left to it
  static bool pageable(const void *host) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, host) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
    (void)hipGetLastError();
    return true;
  }

  // the ring, allocated by the first copy that wants it; without it the
  // runtime does the copy
  bool ring() {
    if (ring_) return true;
    bool ok = hipHostMalloc((void **)&ring_, kSlots * kSlot, hipHostMallocDefault) == hipSuccess;
    if (!ok) ring_ = nullptr;
    for (hipEvent_t &e : ev_)
      if (ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
        e = nullptr;
        ok = false;
      }
    if (!ok) {
      (void)hipGetLastError();
      release();
    }
    return ok;
  }

  // Chunk i passes through slot i % kSlots: the calling thread issues the
  // transfers in order, each once the slot's earlier chunk is emptied, and
  // announces a chunk when its transfer is complete, with the next one under
  // way; the threads take the pieces in order.  No thread waits for a chunk
  // that the calling thread could not reach: a slot is free once pieces of
  // announced chunks are copied.  For the first chunk the threads sleep: the
  // stream may have a whole shot's steps to run before it.  An error stops the
  // threads.  *ran: false if none could be started (nothing was written to
  // host).
  hipError_t staged(char *host, const char *dev, size_t bytes, hipStream_t stream, bool *ran) {
    const long n = (long)((bytes + kSlot - 1) / kSlot);
    const long pieces = (long)((bytes + kPiece - 1) / kPiece);
    std::atomic<long> next{0}, arrived{0};
    std::atomic<bool> stop{false};
    std::mutex m;
    std::condition_variable first;  // a chunk has arrived, or stop
    auto work = [&, host](std::atomic<int> *done) {
      {
        std::unique_lock<std::mutex> lock(m);
        first.wait(lock, [&] { return arrived.load() > 0 || stop.load(); });
      }
      for (long p; (p = next.fetch_add(1)) < pieces;) {
        const long c = p / kPieces;
        while (c >= arrived.load(std::memory_order_acquire)) {
          if (stop.load()) return;
          std::this_thread::yield();
        }
        const size_t at = (size_t)p * kPiece;
        memcpy(host + at, ring_ + (size_t)(c % kSlots) * kSlot + (size_t)(p % kPieces) * kPiece,
               std::min(kPiece, bytes - at));
        done[c].fetch_add(1, std::memory_order_release);
      }
    };
    hipError_t err = hipSuccess;
    auto issue = [&](long i) {
      const size_t at = (size_t)i * kSlot;
      err = hipMemcpyAsync(ring_ + (size_t)(i % kSlots) * kSlot, dev + at,
                           std::min(kSlot, bytes - at), hipMemcpyDeviceToHost, stream);
      if (err == hipSuccess) err = hipEventRecord(ev_[i % kSlots], stream);
    };
    std::vector<std::atomic<int>> done;
    std::vector<std::thread> pool;
    try {
      done = std::vector<std::atomic<int>>(n);
      pool.reserve(kThreads);
      const int want = std::min<int>(kThreads, (int)born_par::threads());
      while ((int)pool.size() < want) pool.emplace_back(work, done.data());
    } catch (const std::exception &) {
      if (pool.empty()) return hipSuccess;
    }
    *ran = true;
    // wakes the threads with a change that they wait for
    auto wake = [&](auto change) {
      {
        std::lock_guard<std::mutex> lock(m);
        change();
      }
      first.notify_all();
    };
    for (long i = 0; i < std::min(n, kSlots) && err == hipSuccess; i++) issue(i);
    for (long i = 1; i <= n && err == hipSuccess; i++) {
      if (i >= kSlots && i < n) {
        while (done[i - kSlots].load(std::memory_order_acquire) < kPieces)
          std::this_thread::yield();
        issue(i);
        if (err != hipSuccess) break;
      }
      err = hipEventSynchronize(ev_[(i - 1) % kSlots]);
      if (err != hipSuccess) break;
      if (i == 1)
        wake([&] { arrived.store(1); });
      else
        arrived.store(i, std::memory_order_release);
    }
    if (err != hipSuccess) wake([&] { stop.store(true); });
    for (std::thread &t : pool) t.join();
    return err;
  }

  char *ring_ = nullptr;
  hipEvent_t ev_[kSlots] = {};
};

}  // namespace born

#endif
