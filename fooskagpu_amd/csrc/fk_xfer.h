// Host <-> device copies of a context: states, labels and predictions in
// ordinary (pageable) host memory.
//
// One hipMemcpy into a buffer the caller has just allocated runs at 11 GB/s
// (245 MB in 22.7 ms): one thread clears the buffer's fresh pages and copies
// out of the runtime's staging memory.  Large copies therefore go through
// page-locked slots of our own, two to a thread, with the DMA of one slot
// overlapping the host copy of the other, on up to kXferThreads threads: 6.0
// ms into fresh pages, and 5.4 instead of 8.3 ms from the host.  Slots of 4 MB:
// an asynchronous copy costs about 18 us however small (1 MB slots: 8.0 ms).
// Mid sizes use part of a slot, so that a few threads share the copy.
#pragma once
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>

#include "fk_internal.h"

namespace fkx {

// Smaller copies stay one hipMemcpy (starting threads costs about 20 us each).
// To the host: 3.8 MB 232 against 266 us, 6.6 MB 420 against 310.  From the
// host, where the pages are there already: 31 MB 1.00 against 1.06 ms, 84 MB
// 2.92 against 2.08.
constexpr size_t kXferMinDown = (size_t)5 << 20, kXferMinUp = (size_t)48 << 20;

// The slots, 64 MB for the process (page-locking them costs about 2 ms, which
// each new context would otherwise pay in its first copy): allocated by the
// first large copy, freed with the last context, and lent to one copy at a
// time.  A copy that finds them lent is one hipMemcpy.
constexpr size_t kXferSlot = (size_t)4 << 20;
struct XferPool {
  std::mutex mu;
  char *pin = nullptr;
  int contexts = 0;
  bool lent = false;

  void attach() {
    std::lock_guard<std::mutex> lk(mu);
    ++contexts;
  }
  void detach() {
    std::lock_guard<std::mutex> lk(mu);
    if (--contexts > 0 || !pin) return;
    (void)hipHostFree(pin);
    pin = nullptr;
  }
  char *borrow() {
    std::lock_guard<std::mutex> lk(mu);
    if (lent) return nullptr;
    if (!pin && hipHostMalloc(reinterpret_cast<void **>(&pin), 2 * kXferThreads * kXferSlot, hipHostMallocPortable) !=
                    hipSuccess) {
      (void)hipGetLastError();
      pin = nullptr;
    }
    lent = pin != nullptr;
    return pin;
  }
  void give_back() {
    std::lock_guard<std::mutex> lk(mu);
    lent = false;
  }
};
inline XferPool g_xfer;

// The slots for a copy of context c, or null: then the copy is one hipMemcpy.
inline char *xfer_begin(fk_ctx *c) {
  for (hipEvent_t &e : c->xfer.ev)
    if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
      (void)hipGetLastError();
      e = nullptr;
      return nullptr;
    }
  return g_xfer.borrow();
}

inline void xfer_free(fk_ctx *c) {
  for (hipEvent_t &e : c->xfer.ev)
    if (e) (void)hipEventDestroy(e);
  c->xfer = Xfer{};
}

// The chunks of one copy, taken by the threads in order.
struct XferJob {
  fk_ctx *c;
  char *pin, *dev, *host;
  size_t bytes, slot;
  bool down;
  std::atomic<size_t> next{0};
  std::atomic<int> err{0};

  size_t take() { return next.fetch_add(slot); }
  size_t len(size_t at) const { return bytes - at < slot ? bytes - at : slot; }
  bool bad(hipError_t e) {
    if (e != hipSuccess) err.store((int)e);
    return err.load() != 0;
  }
  void work(int t) {
    if (bad(hipSetDevice(c->device))) return;
    char *buf[2];
    hipEvent_t ev[2];
    for (int s = 0; s < 2; ++s) {
      buf[s] = pin + (size_t)(2 * t + s) * kXferSlot;
      ev[s] = c->xfer.ev[2 * t + s];
    }
    if (down) {
      auto fetch = [&](size_t at, int s) {
        return !bad(hipMemcpyAsync(buf[s], dev + at, len(at), hipMemcpyDeviceToHost, c->stream)) &&
               !bad(hipEventRecord(ev[s], c->stream));
      };
      size_t at = take();
      if (at >= bytes || !fetch(at, 0)) return;
      for (int s = 0;; s ^= 1) {
        const size_t nx = take();
        if (nx < bytes && !fetch(nx, s ^ 1)) return;
        if (bad(hipEventSynchronize(ev[s]))) return;
        std::memcpy(host + at, buf[s], len(at));
        if (nx >= bytes) return;
        at = nx;
      }
    }
    int used = 0;
    for (int s = 0;; s ^= 1) {
      const size_t at = take();
      if (at >= bytes) return;
      if (used++ >= 2 && bad(hipEventSynchronize(ev[s]))) return;
      std::memcpy(buf[s], host + at, len(at));
      if (bad(hipMemcpyAsync(dev + at, buf[s], len(at), hipMemcpyHostToDevice, c->stream))) return;
      if (bad(hipEventRecord(ev[s], c->stream))) return;
    }
  }
};

inline int xfer_staged(fk_ctx *c, char *pin, void *dev, void *host, size_t bytes, bool down) {
  XferJob job{c, pin, static_cast<char *>(dev), static_cast<char *>(host), bytes, 0, down};
  job.slot = bytes >= 16 * kXferSlot ? kXferSlot : (bytes >= 4 * kXferSlot ? kXferSlot / 2 : kXferSlot / 4);
  const size_t chunks = (bytes + job.slot - 1) / job.slot;
  const int nt = (int)(chunks / 2 < (size_t)kXferThreads ? chunks / 2 : kXferThreads);
  std::thread th[kXferThreads];
  for (int t = 1; t < nt; ++t) {
    try {
      th[t] = std::thread([&job, t] { job.work(t); });
    } catch (...) {
      break;  // the threads that started, at least this one, do the work
    }
  }
  job.work(0);
  for (std::thread &t : th)
    if (t.joinable()) t.join();
  const hipError_t e = hipStreamSynchronize(c->stream);  // also after an error: nothing uses the slots any more
  g_xfer.give_back();
  if (job.err.load()) return fail(FK_EDEVICE, std::string("copy: ") + hipGetErrorString((hipError_t)job.err.load()));
  if (e != hipSuccess) return fail(FK_EDEVICE, std::string("copy: ") + hipGetErrorString(e));
  return FK_OK;
}

// Synchronous copies, ordered after the work on the context's stream.
inline int copy_down(fk_ctx *c, void *host, const void *dev, size_t bytes) {
  if (bytes >= kXferMinDown)
    if (char *pin = xfer_begin(c)) return xfer_staged(c, pin, const_cast<void *>(dev), host, bytes, true);
  HIPCHK(hipStreamSynchronize(c->stream));
  HIPCHK(hipMemcpy(host, dev, bytes, hipMemcpyDeviceToHost));
  return FK_OK;
}
inline int copy_up(fk_ctx *c, void *dev, const void *host, size_t bytes) {
  if (bytes >= kXferMinUp)
    if (char *pin = xfer_begin(c)) return xfer_staged(c, pin, dev, const_cast<void *>(host), bytes, false);
  HIPCHK(hipStreamSynchronize(c->stream));
  HIPCHK(hipMemcpy(dev, host, bytes, hipMemcpyHostToDevice));
  return FK_OK;
}

}  // namespace fkx
