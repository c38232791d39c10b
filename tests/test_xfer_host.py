"""The large host copies (fk_xfer.h) on a small HIP runtime of the host's own
that keeps to what HIP promises and no more: streams run on their own threads,
a stream that does not block with the null stream is not ordered with it, the
clearing of device memory by the null stream comes late, and new device memory
holds what was there before.  Bytes have to arrive all the same."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CLANG = "/opt/rocm/llvm/bin/clang++"

MOCK = r"""
#pragma once
#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <mutex>
#include <thread>
#define __global__
#define __device__
#define __host__
#define __forceinline__ inline
#define __launch_bounds__(...)
typedef int hipError_t;
enum { hipSuccess = 0 };
enum { hipHostMallocDefault = 0, hipHostMallocPortable = 1, hipHostMallocMapped = 2, hipHostMallocCoherent = 0x40000000 };
enum { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
struct dim3 { unsigned x; dim3(unsigned v) : x(v) {} };
typedef struct Ev *hipEvent_t;
struct Stream {
  std::mutex mu;
  std::condition_variable cv;
  std::deque<std::function<void()>> q;
  bool busy = false;
  void loop() {
    for (;;) {
      std::unique_lock<std::mutex> lk(mu);
      busy = false;
      cv.notify_all();
      cv.wait(lk, [&] { return !q.empty(); });
      auto f = std::move(q.front());
      q.pop_front();
      busy = true;
      lk.unlock();
      f();
    }
  }
  Stream() { std::thread([this] { loop(); }).detach(); }
  void push(std::function<void()> f) {
    std::lock_guard<std::mutex> lk(mu);
    q.push_back(std::move(f));
    cv.notify_all();
  }
  void wait() {
    std::unique_lock<std::mutex> lk(mu);
    cv.wait(lk, [&] { return q.empty() && !busy; });
  }
};
typedef Stream *hipStream_t;
inline thread_local struct { unsigned x; } blockIdx, threadIdx;
inline size_t g_pin_bytes = 0, g_pins = 0;                   // page-locked now, and how often
inline unsigned g_pin_flags = 0, g_memcpys = 0, g_stale = 0;  // g_stale: what new device memory holds
inline std::function<void()> g_late;                         // the null stream's clearing, not done yet
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned flags) {
  g_pin_flags = flags;
  g_pin_bytes = n;
  ++g_pins;
  *p = aligned_alloc(4096, (n + 4095) / 4096 * 4096);
  return hipSuccess;
}
inline hipError_t hipHostFree(void *p) { free(p); g_pin_bytes = 0; return hipSuccess; }
template <typename T>
inline hipError_t hipMalloc(T **p, size_t n) {
  *p = static_cast<T *>(aligned_alloc(4096, (n + 4095) / 4096 * 4096));
  for (size_t i = 0; i < n / 4; ++i) reinterpret_cast<unsigned *>(*p)[i] = g_stale;
  return hipSuccess;
}
inline hipError_t hipFree(void *p) { free(p); return hipSuccess; }
inline hipError_t hipMemset(void *p, int v, size_t n) {
  g_late = [=] { memset(p, v, n); };
  return hipSuccess;
}
inline hipError_t hipMemcpy(void *d, const void *s, size_t n, int) { ++g_memcpys; memcpy(d, s, n); return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t s) { s->wait(); return hipSuccess; }
inline std::atomic<int> g_fail_launches{0};  // that many launches fail from now on
inline thread_local hipError_t g_last = hipSuccess;
inline hipError_t hipGetLastError() { hipError_t e = g_last; g_last = hipSuccess; return e; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline const char *hipGetErrorString(hipError_t) { return ""; }
inline hipError_t hipEventCreate(hipEvent_t *) { return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventElapsedTime(float *, hipEvent_t, hipEvent_t) { return hipSuccess; }
inline void __syncthreads() {}
inline void __threadfence_system() { std::atomic_thread_fence(std::memory_order_seq_cst); }
inline unsigned atomicAdd(unsigned *p, unsigned v) { return __atomic_fetch_add(p, v, __ATOMIC_SEQ_CST); }
#define __HIP_MEMORY_SCOPE_SYSTEM 0
#define __hip_atomic_store(p, v, order, scope) __atomic_store_n(p, v, order)
// a block's threads from the last to the first: thread 0 goes on behind the
// barrier when the others have reached it
template <typename K, typename... A>
inline void mock_launch(K k, unsigned grid, unsigned block, hipStream_t s, A... a) {
  if (g_fail_launches.load() > 0 && g_fail_launches.fetch_sub(1) > 0) {
    g_last = 1;
    return;
  }
  s->push([=] {
    for (unsigned b = 0; b < grid; ++b) {
      for (unsigned t = block; t-- > 0;) {
        blockIdx.x = b;
        threadIdx.x = t;
        k(a...);
      }
      if (b % 16 == 15) std::this_thread::yield();
    }
  });
}
#define hipLaunchKernelGGL(k, g, b, lds, s, ...) mock_launch(k, dim3(g).x, dim3(b).x, s, __VA_ARGS__)
"""

MAIN = r"""
#include <cstdio>
#include <vector>
#include "fk_xfer.h"
using namespace fkx;
// bytes of pattern k
static std::vector<char> pattern(size_t n, unsigned k) {
  std::vector<char> v(n);
  unsigned s = 12345u + k;
  for (char &c : v) c = (char)((s = s * 1664525u + 1013904223u) >> 24);
  return v;
}
static char *device(size_t n) {
  char *p = nullptr;
  (void)hipMalloc(&p, n + 64);
  return p;
}
int main() {
  fk_ctx *c = new fk_ctx;
  c->stream = new Stream;
  g_xfer.attach();
  int wrong = 0;
  auto say = [&](bool ok, const char *what) {
    std::printf("%s: %s\n", what, ok ? "ok" : "wrong");
    wrong += !ok;
  };
BODY
  std::printf("done\n");
  std::fflush(stdout);
  _Exit(wrong ? 1 : 0);
}
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    d = tmp_path_factory.mktemp("xfer")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(MOCK)

    def go(body):
        (d / "main.cpp").write_text(MAIN.replace("BODY", body))
        subprocess.run([CLANG, "-std=c++17", "-O1", "-pthread", "-I" + str(d),
                        "-I" + os.path.join(ROOT, "fooskagpu_amd", "csrc"), str(d / "main.cpp"), "-o",
                        str(d / "main")], check=True)
        r = subprocess.run([str(d / "main")], capture_output=True, text=True, timeout=100)
        assert r.returncode == 0 and r.stdout.endswith("done\n"), r.stdout + r.stderr
        return r.stdout

    return go


def test_slots_are_coherent_memory(run):
    """The host reads a slot while later kernels of the stream still run and
    refills one that a later kernel reads, with no synchronisation in between:
    the memory has to be coherent by request, not by the environment's
    default."""
    run("""
  const size_t n = (size_t)40 << 20;
  char *dev = device(n);
  std::vector<char> in = pattern(n, 1), out(n);
  say(copy_up(c, dev, in.data(), n) == FK_OK && std::memcmp(dev, in.data(), n) == 0, "upload");
  say(copy_down(c, out.data(), dev, n) == FK_OK && out == in, "download");
  say(g_memcpys == 0, "through the slots");
  say((g_pin_flags & hipHostMallocCoherent) && (g_pin_flags & hipHostMallocPortable), "coherent slots");
""")


@pytest.mark.parametrize("stale", [1, 40, 0xabababab])
def test_block_counts_are_cleared_before_the_first_piece(run, stale):
    """The counters of a context's copies start in memory that held something
    else; a count that starts above zero reports a piece before all of its
    blocks have run, garbage never reports it."""
    run(f"""
  g_stale = {stale}u;
  const size_t n = (size_t)40 << 20;
  char *dev = device(n);
  std::vector<char> in = pattern(n, 2), out(n);
  const auto t0 = std::chrono::steady_clock::now();
  for (unsigned k = 0; k < 3; ++k) {{
    in = pattern(n, k);
    say(copy_up(c, dev, in.data(), n) == FK_OK && std::memcmp(dev, in.data(), n) == 0, "upload");
    say(copy_down(c, out.data(), dev, n) == FK_OK && out == in, "download");
  }}
  say(g_memcpys == 0, "through the slots");
  say(std::chrono::steady_clock::now() - t0 < std::chrono::seconds(20), "no piece waits for its time-out");
  say(!g_late, "nothing left to the null stream");
""")


def test_counts_are_cleared_again_after_a_failed_copy(run):
    """A copy that fails leaves its counters to be cleared before the next."""
    run("""
  const size_t n = (size_t)40 << 20;
  char *dev = device(n);
  std::vector<char> in = pattern(n, 3), out(n);
  say(copy_up(c, dev, in.data(), n) == FK_OK, "upload");
  g_fail_launches = 3;
  say(copy_up(c, dev, in.data(), n) != FK_OK, "failed upload");
  g_fail_launches = 0;
  for (int s = 0; s < kXferSlots; ++s) c->xfer.count[s] = 50;
  in = pattern(n, 4);
  say(copy_up(c, dev, in.data(), n) == FK_OK && std::memcmp(dev, in.data(), n) == 0, "next upload");
  say(copy_down(c, out.data(), dev, n) == FK_OK && out == in, "next download");
""")


def test_only_aligned_device_memory_is_copied_in_wide_words(run):
    """The copy kernel moves 16-byte words: a device address between them goes
    to hipMemcpy; any number of bytes, at any host address, through the slots
    (the tail of 1 to 15 bytes by itself)."""
    run("""
  for (int tail : {0, 1, 4, 12, 15}) {
    const size_t n = ((size_t)18 << 20) + tail;
    std::vector<char> in = pattern(n + 3, tail), out(n + 5);
    for (int off : {0, 4, 8, 16}) {
      char *dev = device(n) + off;
      g_memcpys = 0;
      say(copy_up(c, dev, in.data() + 3, n) == FK_OK && std::memcmp(dev, in.data() + 3, n) == 0, "upload");
      say(copy_down(c, out.data() + 5, dev, n) == FK_OK && std::memcmp(out.data() + 5, in.data() + 3, n) == 0, "download");
      say(g_memcpys == (off % 16 ? 2 : 0), off % 16 ? "by hipMemcpy" : "through the slots");
    }
  }
""")


def test_no_more_is_page_locked_than_the_copy_uses(run):
    """Page-locking takes up to 2 ms for 64 MB, which a program's first copy
    pays: it locks what its own pieces go through, a larger copy later what it
    needs, and a smaller one nothing."""
    run("""
  const size_t mb = (size_t)1 << 20;
  std::vector<char> in = pattern(100 * mb + 7, 5), out(100 * mb + 7);
  char *dev = device(100 * mb + 7);
  size_t pins = 0, locked = 0;
  for (size_t n : {6 * mb + 3, 18 * mb, 40 * mb, 7 * mb, 100 * mb + 7, 20 * mb}) {
    say(copy_up(c, dev, in.data(), n) == FK_OK && copy_down(c, out.data(), dev, n) == FK_OK &&
        std::memcmp(out.data(), in.data(), n) == 0, "copied");
    say(g_pin_bytes <= 2 * n && g_pin_bytes <= 65 * mb || g_pins == pins, "locked by need");
    say(g_pin_bytes >= locked, "kept");
    pins = g_pins;
    locked = g_pin_bytes;
  }
  say(pins <= 4, "locked anew for larger copies alone");
  g_xfer.detach();
  say(g_pin_bytes == 0, "given back");
""")
