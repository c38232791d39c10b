// Host <-> device copies of a context: states, labels and predictions in
// ordinary (pageable) host memory.
//
// One hipMemcpy into a buffer the caller has just allocated runs at 11 GB/s
// (245 MB in 22.7 ms): one thread clears the buffer's fresh pages and copies
// out of the runtime's staging memory.  Large copies therefore go through
// page-locked slots of our own, two to a thread on up to kXferThreads threads,
// the transfer of one slot overlapping the host copy of the other.  The
// transfers are kernels that read or write the slots over the link: in 1 MB
// pieces they run at 52 GB/s where hipMemcpyAsync, at about 18 us a piece,
// reaches 38 (4 MB pieces: 54 and 51), and the last block of a piece reports
// it to the waiting thread.  Downloads into fresh memory, us, one hipMemcpy /
// slots: 6.6 MB 420 / 258, 31 MB 1903 / 820, 84 MB 6536 / 1980, 246 MB 23193 /
// 5940; uploads: 41 MB 1370 / 1070, 84 MB 2922 / 1940, 246 MB 8331 / 5160.
#pragma once
#include <atomic>
#include <chrono>
#include <cstring>
#include <mutex>
#include <thread>

#include "fk_internal.h"

namespace fkx {

// Smaller copies stay one hipMemcpy (starting threads costs about 20 us each).
// To the host 3.8 MB take 225 us either way; from the host, where the pages
// are there already, 10 MB 314 and 19 MB 540.
constexpr size_t kXferMinDown = (size_t)5 << 20, kXferMinUp = (size_t)16 << 20;

// The slots, up to 64 MB for the process with a report word each (page-locking
// 64 MB costs about 2 ms, 16 MB 0.1 to 0.2, which each new context would
// otherwise pay in its first copy): allocated by the first large copy at the
// size that it uses, anew by one that uses more, freed with the last context,
// and lent to one copy at a time.  A copy that finds them lent is one hipMemcpy.
// Coherent memory, asked for: the host takes a slot while later kernels of the
// stream run, and refills one for a later kernel without a synchronisation.
constexpr size_t kXferSlot = (size_t)4 << 20;
constexpr int kXferSlots = 2 * kXferThreads;
constexpr size_t kXferReports = 4096;  // at the start of the block, 64 bytes a slot
struct XferPool {
  std::mutex mu;
  char *pin = nullptr;
  size_t cap = 0;
  int contexts = 0;
  bool lent = false;
  std::atomic<unsigned long long> seq{0};

  unsigned long long *report(int slot) {
    return reinterpret_cast<unsigned long long *>(pin) + 8 * slot;
  }
  void attach() {
    std::lock_guard<std::mutex> lk(mu);
    ++contexts;
  }
  void detach() {
    std::lock_guard<std::mutex> lk(mu);
    if (--contexts > 0) return;
    drop();
  }
  void drop() {
    if (pin) (void)hipHostFree(pin);
    pin = nullptr;
    cap = 0;
  }
  // the slots' memory, at least `bytes`
  char *borrow(size_t bytes) {
    std::lock_guard<std::mutex> lk(mu);
    if (lent) return nullptr;
    if (cap < bytes) {
      drop();
      void *p = nullptr;
      if (hipHostMalloc(&p, kXferReports + bytes, kHostCoherent) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
      }
      pin = static_cast<char *>(p);
      cap = bytes;
      std::memset(pin, 0, kXferReports);
    }
    lent = true;
    return pin + kXferReports;
  }
  void give_back() {
    std::lock_guard<std::mutex> lk(mu);
    lent = false;
  }
};
inline XferPool g_xfer;

// n16 16-byte words and `tail` bytes after them from a to b, one of them a
// slot.  The block that ends last releases seq to *report, host memory, behind
// a system-wide fence of every block, and leaves *count at zero.
typedef unsigned int xfer_u4 __attribute__((ext_vector_type(4)));
constexpr unsigned kXferBlocks = 64;
static __global__ void __launch_bounds__(256) xfer_copy(const char *__restrict__ a, char *__restrict__ b, size_t n16,
                                                        int tail, unsigned *__restrict__ count,
                                                        unsigned long long *__restrict__ report,
                                                        unsigned long long seq) {
  const xfer_u4 *src = reinterpret_cast<const xfer_u4 *>(a);
  xfer_u4 *dst = reinterpret_cast<xfer_u4 *>(b);
  for (size_t i = blockIdx.x * (size_t)256 + threadIdx.x; i < n16; i += (size_t)kXferBlocks * 256) dst[i] = src[i];
  if (blockIdx.x == 0 && (int)threadIdx.x < tail) b[16 * n16 + threadIdx.x] = a[16 * n16 + threadIdx.x];
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x != 0) return;
  if (atomicAdd(count, 1u) == kXferBlocks - 1) {
    *count = 0;
    __threadfence_system();
    __hip_atomic_store(report, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

static __global__ void __launch_bounds__(64) xfer_clear(unsigned *__restrict__ count) {
  if ((int)threadIdx.x < kXferSlots) count[threadIdx.x] = 0;
}

// Pieces and threads of a copy: mid sizes in smaller pieces, so that a few
// threads share them; a thread, with two slots, for every two pieces.
struct XferPlan {
  size_t piece;
  int threads;
  explicit XferPlan(size_t bytes)
      : piece(bytes >= 16 * kXferSlot ? kXferSlot : (bytes >= 4 * kXferSlot ? kXferSlot / 2 : kXferSlot / 4)) {
    const size_t half = (bytes + piece - 1) / piece / 2;
    threads = (int)(half < (size_t)kXferThreads ? half : kXferThreads);
  }
};
static_assert(kXferSlots * 64 <= kXferReports, "a report word per slot");

// The slots for a copy of context c, or null: then the copy is one hipMemcpy.
// The counts are cleared on the context's stream, which is not ordered with the
// null stream, and again after a copy that failed.
inline char *xfer_begin(fk_ctx *c, size_t bytes) {
  if (!c->xfer.count) {
    unsigned *p = nullptr;
    if (hipMalloc(&p, kXferSlots * sizeof(unsigned)) != hipSuccess) {
      (void)hipGetLastError();
      return nullptr;
    }
    c->xfer.count = p;
    c->xfer.clear = false;
  }
  const XferPlan plan(bytes);
  char *pin = g_xfer.borrow(2 * plan.threads * plan.piece);
  if (pin && !c->xfer.clear) {
    hipLaunchKernelGGL(xfer_clear, dim3(1), dim3(64), 0, c->stream, c->xfer.count);
    if (hipGetLastError() != hipSuccess) {
      g_xfer.give_back();
      return nullptr;
    }
    c->xfer.clear = true;
  }
  return pin;
}

inline void xfer_free(fk_ctx *c) {
  if (c->xfer.count) (void)hipFree(c->xfer.count);
  c->xfer = Xfer{};
}

// The pieces of one copy, taken by the threads in order.
struct XferJob {
  fk_ctx *c;
  char *pin, *dev, *host;
  size_t bytes;
  bool down;
  size_t piece;
  std::atomic<size_t> next{0};
  std::atomic<int> err{0};

  size_t take() { return next.fetch_add(piece); }
  size_t len(size_t at) const { return bytes - at < piece ? bytes - at : piece; }
  bool bad(hipError_t e) {
    if (e != hipSuccess) err.store((int)e);
    return err.load() != 0;
  }
  char *slot(int s) { return pin + (size_t)s * piece; }
  // starts the transfer of the piece at `at` through slot s; its report in *seq
  bool start(size_t at, int s, unsigned long long *seq) {
    const size_t n = len(at);
    *seq = ++g_xfer.seq;
    const char *a = down ? dev + at : slot(s);
    char *b = down ? slot(s) : dev + at;
    hipLaunchKernelGGL(xfer_copy, dim3(kXferBlocks), dim3(256), 0, c->stream, a, b, n / 16, (int)(n % 16),
                       c->xfer.count + s, g_xfer.report(s), *seq);
    return !bad(hipGetLastError());
  }
  // waits for a report; after 2 s (or an error elsewhere) for the stream
  bool wait(int s, unsigned long long seq) {
    const auto t0 = std::chrono::steady_clock::now();
    for (int k = 0; __atomic_load_n(g_xfer.report(s), __ATOMIC_ACQUIRE) != seq; ++k)
      if ((k & 1023) == 1023 && (err.load() || std::chrono::steady_clock::now() - t0 > std::chrono::seconds(2)))
        return !bad(hipStreamSynchronize(c->stream));
    return true;
  }
  void work(int t) {
    if (bad(hipSetDevice(c->device))) return;
    const int s0 = 2 * t;
    unsigned long long seq[2] = {0, 0};
    if (down) {
      size_t at = take();
      if (at >= bytes || !start(at, s0, &seq[0])) return;
      for (int s = 0;; s ^= 1) {
        const size_t nx = take();
        if (nx < bytes && !start(nx, s0 + (s ^ 1), &seq[s ^ 1])) return;
        if (!wait(s0 + s, seq[s])) return;
        std::memcpy(host + at, slot(s0 + s), len(at));
        if (nx >= bytes) return;
        at = nx;
      }
    }
    for (int s = 0;; s ^= 1) {
      const size_t at = take();
      if (at >= bytes) return;
      if (seq[s] && !wait(s0 + s, seq[s])) return;
      std::memcpy(slot(s0 + s), host + at, len(at));
      if (!start(at, s0 + s, &seq[s])) return;
    }
  }
};

inline int xfer_staged(fk_ctx *c, char *pin, void *dev, void *host, size_t bytes, bool down) {
  const XferPlan plan(bytes);
  XferJob job{c, pin, static_cast<char *>(dev), static_cast<char *>(host), bytes, down, plan.piece};
  const int nt = plan.threads;
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
  c->xfer.clear = !job.err.load() && e == hipSuccess;
  if (job.err.load()) return fail(FK_EDEVICE, std::string("copy: ") + hipGetErrorString((hipError_t)job.err.load()));
  if (e != hipSuccess) return fail(FK_EDEVICE, std::string("copy: ") + hipGetErrorString(e));
  return FK_OK;
}

// Synchronous copies, ordered after the work on the context's stream.  Device
// memory between 16-byte words is not for xfer_copy.
inline bool xfer_aligned(const void *dev) { return reinterpret_cast<uintptr_t>(dev) % 16 == 0; }
inline int copy_down(fk_ctx *c, void *host, const void *dev, size_t bytes) {
  if (bytes >= kXferMinDown && xfer_aligned(dev))
    if (char *pin = xfer_begin(c, bytes)) return xfer_staged(c, pin, const_cast<void *>(dev), host, bytes, true);
  HIPCHK(hipStreamSynchronize(c->stream));
  HIPCHK(hipMemcpy(host, dev, bytes, hipMemcpyDeviceToHost));
  return FK_OK;
}
inline int copy_up(fk_ctx *c, void *dev, const void *host, size_t bytes) {
  if (bytes >= kXferMinUp && xfer_aligned(dev))
    if (char *pin = xfer_begin(c, bytes)) return xfer_staged(c, pin, dev, const_cast<void *>(host), bytes, false);
  HIPCHK(hipStreamSynchronize(c->stream));
  HIPCHK(hipMemcpy(dev, host, bytes, hipMemcpyHostToDevice));
  return FK_OK;
}

}  // namespace fkx
