// fd2_hostcopy.h -- copies between a caller's ordinary (pageable) memory and
// device memory through a small pinned ring, on a few host threads.
//
// The device copies pinned memory at 52 GB/s; one thread fills or empties it at
// 30 GB/s (10 GB/s into pages touched for the first time).  So a large copy goes
// in slices: each worker fills (or empties) its own slots of the ring while the
// device copies the others.  On MI355X: 74 MB to the device in 2.0 ms (one thread
// and one pinned buffer of that size 3.8 ms, and two more passes to check and
// count the events), 13 MB back in 0.46 ms (one hipMemcpy 0.82 ms), with at most
// 16 MB of pinned memory per object.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

#include "../../include/fd2.h"

namespace fd2 {

class HostCopy {
 public:
  ~HostCopy() { release(); }
  void release() {
    for (hipEvent_t& e : ready_) {
      if (e) (void)hipEventDestroy(e);
      e = nullptr;
    }
    if (ring_ && pinned_) (void)hipHostFree(ring_);
    if (ring_ && !pinned_) std::free(ring_);
    ring_ = nullptr;
    cap_ = 0;
  }

  // Copies `bytes` from `src` to device memory in stream order.
  // fill(dst, offset, len) writes the bytes [offset, offset + len) of the
  // source to pinned memory and returns a status; the status of the first slice
  // (in order) that is not FD2_OK ends the copy and is returned.  Returns
  // before the device has finished; the caller waits for the stream before the
  // next call.  `grain` divides every slice.
  template <class Fill>
  int upload(hipStream_t stream, int device, void* dst, size_t bytes, size_t grain, Fill fill) {
    const int rc = reserve(bytes);
    if (rc) return rc;
    const size_t slice = slice_of(bytes) / grain * grain;
    return run(device, bytes, slice, [&](Worker& w, size_t off, size_t len) {
      const int slot = w.next_slot();
      if (w.used[slot] && hipEventSynchronize(ready_[w.base + slot]) != hipSuccess)
        return (int)FD2_E_DEVICE;
      char* s = slot_of(w, slot);
      const int status = fill(s, off, len);
      if (status) return status;
      if (hipMemcpyAsync(static_cast<char*>(dst) + off, s, len, hipMemcpyHostToDevice, stream) !=
          hipSuccess)
        return (int)FD2_E_DEVICE;
      return bytes <= slice ? (int)FD2_OK : w.mark(*this, slot, stream);
    }, [](Worker&) { return (int)FD2_OK; });
  }

  // Copies device memory to `dst` after the work of `stream`, and waits for it.
  int download(hipStream_t stream, int device, void* dst, const void* src, size_t bytes) {
    if (bytes < 2 * kMinSlice) {  // the runtime's own copy is as fast
      if (hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream) != hipSuccess ||
          hipStreamSynchronize(stream) != hipSuccess)
        return FD2_E_DEVICE;
      return FD2_OK;
    }
    // the stream may still read the ring (an upload of the same call), which
    // reserve may give back
    if (hipStreamSynchronize(stream) != hipSuccess) return FD2_E_DEVICE;
    const int rc = reserve(bytes);
    if (rc) return rc;
    char* out = static_cast<char*>(dst);
    auto empty = [&](Worker& w, int slot) {
      if (!w.used[slot]) return (int)FD2_OK;
      w.used[slot] = false;
      if (hipEventSynchronize(ready_[w.base + slot]) != hipSuccess) return (int)FD2_E_DEVICE;
      std::memcpy(out + w.off[slot], slot_of(w, slot), w.len[slot]);
      return (int)FD2_OK;
    };
    return run(device, bytes, slice_of(bytes), [&](Worker& w, size_t off, size_t len) {
      const int slot = w.next_slot();
      int status = empty(w, slot);
      if (status) return status;
      w.off[slot] = off;
      w.len[slot] = len;
      if (hipMemcpyAsync(slot_of(w, slot),
                         static_cast<const char*>(src) + off, len, hipMemcpyDeviceToHost,
                         stream) != hipSuccess)
        return (int)FD2_E_DEVICE;
      return w.mark(*this, slot, stream);
    }, [&](Worker& w) {  // a worker's last slices, the older one first
      const int first = empty(w, w.next_slot());
      const int second = empty(w, w.next_slot());
      return first ? first : second;
    });
  }

 private:
  static constexpr int kWorkers = 4, kSlots = 2;
  static constexpr size_t kMinSlice = (size_t)512 << 10, kMaxSlice = (size_t)2 << 20;
  static constexpr size_t kSmall = (size_t)64 << 10;

  // a slice costs the device 15 us besides its bytes (74 MB in slices of 0.25,
  // 0.5, 1 MB: 5.8, 3.6, 2.5 ms), so at most one per slot while the ring stays
  // small
  static size_t slice_of(size_t bytes) {
    constexpr size_t unit = (size_t)256 << 10;
    const size_t s = (bytes / (kWorkers * kSlots) + unit) / unit * unit;
    return std::min(std::max(s, kMinSlice), kMaxSlice);
  }

  struct Worker {
    int base = 0, turn = 0;
    bool used[kSlots] = {};
    size_t off[kSlots] = {}, len[kSlots] = {};
    int next_slot() { return turn++ % kSlots; }
    int mark(HostCopy& h, int slot, hipStream_t stream) {
      used[slot] = true;
      return hipEventRecord(h.ready_[base + slot], stream) == hipSuccess ? FD2_OK : FD2_E_DEVICE;
    }
  };

  char* slot_of(const Worker& w, int slot) const {
    return ring_ + (size_t)(w.base + slot) * (cap_ / (kWorkers * kSlots));
  }

  // a ring for copies of `bytes`: 64 KB for small ones, else 4 to 16 MB; of
  // ordinary memory if no more can be pinned (the runtime then stages its copies).
  // Freeing that waits for no copy: whoever gets here has waited for the stream.
  int reserve(size_t bytes) {
    const size_t need = bytes <= kSmall ? kSmall : kWorkers * kSlots * slice_of(bytes);
    if (cap_ >= need) return FD2_OK;
    release();
    void* p = nullptr;
    pinned_ = hipHostMalloc(&p, need, hipHostMallocDefault) == hipSuccess;
    if (!pinned_) {
      (void)hipGetLastError();  // answered here
      p = std::malloc(need);
      if (!p) return FD2_E_NOMEM;
    }
    ring_ = static_cast<char*>(p);
    if (need > kSmall)
      for (hipEvent_t& e : ready_)
        if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
          release();
          return FD2_E_DEVICE;
        }
    cap_ = need;
    return FD2_OK;
  }

  // move(worker, offset, length) for every slice, on up to kWorkers threads,
  // then end(worker) on each.  Slices are taken in order, and a failed one stops
  // those after it, so the first failing slice's status is the result.
  template <class Move, class End>
  int run(int device, size_t bytes, size_t slice, Move move, End end) {
    const size_t n = (bytes + slice - 1) / slice;
    std::atomic<size_t> next{0}, bad{n};
    int status = FD2_OK;
    std::mutex mu;
    auto fail = [&](size_t i, int s) {
      std::lock_guard<std::mutex> lock(mu);
      if (status == FD2_OK || i < bad.load()) {
        bad.store(i);
        status = s;
      }
    };
    auto work = [&](int id) {
      Worker w;
      w.base = id * kSlots;
      for (;;) {
        const size_t i = next.fetch_add(1);
        if (i >= bad.load()) break;
        const int s = move(w, i * slice, std::min(slice, bytes - i * slice));
        if (s) {
          fail(i, s);
          break;
        }
      }
      const int s = end(w);
      if (s) fail(n, s);
    };
    const unsigned hw = std::thread::hardware_concurrency();
    size_t threads = std::min<size_t>(kWorkers, (n + 1) / 2);
    if (hw > 0 && threads > hw) threads = hw;
    std::vector<std::thread> others;
    try {
      if (threads > 1) others.reserve(threads - 1);
      for (size_t t = 1; t < threads; ++t)
        others.emplace_back([&work, &fail, device, n, t] {
          if (hipSetDevice(device) == hipSuccess)
            work((int)t);
          else
            fail(n, FD2_E_DEVICE);
        });
    } catch (...) {  // fewer threads do the same slices
    }
    work(0);
    for (std::thread& t : others) t.join();
    return status;
  }

  char* ring_ = nullptr;
  bool pinned_ = false;
  size_t cap_ = 0;
  hipEvent_t ready_[kWorkers * kSlots] = {};
};

}  // namespace fd2
