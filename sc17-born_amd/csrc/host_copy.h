// host_copy.h -- copies between pageable host arrays and the device through a
// ring of pinned slots.
//
// hipMemcpyAsync on pageable memory is bound by the one thread that fills or
// empties the runtime's staging buffer (@PLAIN@ GB/s in, @PLAINO@ out for fields of
// 16 MB); here a few threads do that side while the calling thread issues the
// transfers in order (@STAGED@ and @STAGEDO@ GB/s).
#ifndef BORN_HOST_COPY_H
#define BORN_HOST_COPY_H

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstring>
#include <thread>
#include <vector>

#include "host_par.h"

namespace born {

class HostCopy {
 public:
  // dst on the device: on return src may be changed, the transfer is ordered
  // on the stream
  hipError_t in(void *dst, const void *src, size_t bytes, hipStream_t stream) {
    if (!staged(src, bytes))
      return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, stream);
    return run((char *)dst, (char *)src, bytes, stream, true);
  }
  // dst on the host, complete on return
  hipError_t out(void *dst, const void *src, size_t bytes, hipStream_t stream) {
    if (!staged(dst, bytes)) {
      const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream);
      return e != hipSuccess ? e : hipStreamSynchronize(stream);
    }
    return run((char *)src, (char *)dst, bytes, stream, false);
  }
  // with no transfer of this object in flight
  void release() {
    for (hipEvent_t e : ev_) (void)hipEventDestroy(e);
    ev_.clear();
    if (ring_) (void)hipHostFree(ring_);
    ring_ = nullptr;
  }

 private:
  static constexpr size_t kSlot = (size_t)BORN_SLOT_KB << 10;
  static constexpr long kSlots = BORN_SLOTS;  // @RING@
  static constexpr long kLag = kSlots / 2;
  static constexpr size_t kMin = 4 * kSlot;  // @MIN@

  // Large and pageable; memory the runtime knows (pinned, managed, device) is
  // transferred by it directly.  Without the ring the runtime does the copy.
  bool staged(const void *host, size_t bytes) {
    if (bytes < kMin) return false;
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, host) != hipSuccess)
      (void)hipGetLastError();
    else if (a.type != hipMemoryTypeUnregistered)
      return false;
    if (!ring_) {
      if (hipHostMalloc((void **)&ring_, kSlots * kSlot, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        ring_ = nullptr;
        return false;
      }
      for (long k = 0; k < kSlots; k++) {
        hipEvent_t e;
        if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
          (void)hipGetLastError();
          release();
          return false;
        }
        ev_.push_back(e);
      }
    }
    return true;
  }

  // Chunk i of the copy passes through slot i % kSlots.  The workers take
  // chunks in order: going in they fill one whose slot is free, coming out
  // they empty one that has arrived; the calling thread issues the transfers
  // in order and waits for transfer i - kLag after issuing transfer i.  Chunk
  // i + 1 never waits for more than transfer i + 1 - kSlots, so each wait ends;
  // on an error the workers stop at their next wait.
  hipError_t run(char *dev, char *host, size_t bytes, hipStream_t stream, bool in) {
    const long n = (long)((bytes + kSlot - 1) / kSlot);
    auto size = [=](long i) { return std::min(kSlot, bytes - (size_t)i * kSlot); };
    auto slot = [=](long i) { return ring_ + (size_t)(i % kSlots) * kSlot; };
    hipError_t err = hipSuccess;
    // transfers of earlier copies out of the ring
    for (long k = 0; k < std::min(n, kSlots) && err == hipSuccess; k++)
      err = hipEventSynchronize(ev_[k]);
    if (err != hipSuccess) return err;

    std::atomic<long> next{0}, open{in ? kSlots : 0};
    std::atomic<bool> stop{false};
    std::vector<std::atomic<char>> done(n);
    auto work = [&]() {
      for (long i; (i = next.fetch_add(1)) < n;) {
        while (i >= open.load(std::memory_order_acquire)) {
          if (stop.load()) return;
          std::this_thread::yield();
        }
        char *h = host + (size_t)i * kSlot;
        if (in)
          memcpy(slot(i), h, size(i));
        else
          memcpy(h, slot(i), size(i));
        done[i].store(1, std::memory_order_release);
      }
    };
    std::vector<std::thread> pool;
    const long want = std::min<long>(BORN_COPY_THREADS, born_par::threads());
    pool.reserve(want);
    try {
      while ((long)pool.size() < want) pool.emplace_back(work);
    } catch (...) {
      // fewer threads; none: the runtime does the copy
      if (pool.empty()) {
        err = hipMemcpyAsync(in ? dev : host, in ? host : dev, bytes,
                             in ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost, stream);
        return err != hipSuccess || in ? err : hipStreamSynchronize(stream);
      }
    }
    auto wait = [&](long i) {
      while (!done[i].load(std::memory_order_acquire)) std::this_thread::yield();
    };
    auto arrived = [&](long i) {  // transfer i is complete
      if (err == hipSuccess) err = hipEventSynchronize(ev_[i % kSlots]);
      if (err == hipSuccess)
        open.store(in ? i + 1 + kSlots : i + 1, std::memory_order_release);
    };
    for (long i = 0; i < n && err == hipSuccess; i++) {
      if (in)
        wait(i);
      else if (i >= kSlots)
        wait(i - kSlots);
      char *d = dev + (size_t)i * kSlot;
      err = hipMemcpyAsync(in ? d : slot(i), in ? slot(i) : d, size(i),
                           in ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost, stream);
      if (err == hipSuccess) err = hipEventRecord(ev_[i % kSlots], stream);
      if (i >= kLag) arrived(i - kLag);
    }
    if (!in)
      for (long i = std::max(0L, n - kLag); i < n; i++) arrived(i);
    if (err != hipSuccess) stop.store(true);
    for (auto &t : pool) t.join();
    return err;
  }

  char *ring_ = nullptr;
  std::vector<hipEvent_t> ev_;
};

}  // namespace born

#endif
