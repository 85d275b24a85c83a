"""The pinned ring that carries results into the caller's memory (vw_xfer.h), built
on the CPU against a stand-in for the HIP runtime: a stream is a thread that works
through its copies in order, after a kernel that takes 0.3 s."""
import os
import subprocess

from conftest import ROOT

HIP = r"""
#pragma once
#include <chrono>
#include <condition_variable>
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <mutex>
#include <thread>
enum hipError_t { hipSuccess = 0, hipErrorUnknown = 999 };
enum hipMemcpyKind { hipMemcpyDeviceToHost };
enum { hipHostMallocDefault = 0, hipEventDisableTiming = 2 };
struct Stream {
  std::mutex m;
  std::condition_variable cv;
  std::deque<std::function<void()>> q;
  bool stop = false, busy = false;
  std::thread t{[this] {
    std::unique_lock<std::mutex> l(m);
    for (;;) {
      cv.wait(l, [&] { return stop || !q.empty(); });
      if (q.empty()) return;
      auto f = q.front(); q.pop_front(); busy = true;
      l.unlock(); f(); l.lock();
      busy = false; cv.notify_all();
    }
  }};
  void push(std::function<void()> f) { { std::lock_guard<std::mutex> l(m); q.push_back(f); } cv.notify_all(); }
  void wait() { std::unique_lock<std::mutex> l(m); cv.wait(l, [&] { return q.empty() && !busy; }); }
  ~Stream() { { std::lock_guard<std::mutex> l(m); stop = true; } cv.notify_all(); t.join(); }
};
typedef Stream* hipStream_t;
struct Event { std::mutex m; std::condition_variable cv; long rec = 0, done = 0; };
typedef Event* hipEvent_t;
inline std::mutex g_m;
inline bool g_kernel = false; /* the kernel before the results runs */
inline int g_wait = 0, g_max = 0, g_copies = 0, g_fail_at = -1;
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, int) { *p = std::malloc(n); return hipSuccess; }
inline hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, int) { *e = new Event; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
  if (g_copies++ == g_fail_at) return hipErrorUnknown;
  st->push([=] { std::memcpy(d, s, n); });
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t st) {
  long k;
  { std::lock_guard<std::mutex> l(e->m); k = ++e->rec; }
  st->push([=] { { std::lock_guard<std::mutex> l(e->m); e->done = k; } e->cv.notify_all(); });
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
  { std::lock_guard<std::mutex> l(g_m); ++g_wait; if (g_kernel && g_wait > g_max) g_max = g_wait; }
  { std::unique_lock<std::mutex> l(e->m); e->cv.wait(l, [&] { return e->done >= e->rec; }); }
  std::lock_guard<std::mutex> l(g_m); --g_wait;
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) { s->wait(); return hipSuccess; }
"""

MAIN = r"""
#include "vw_xfer.h"
#include <cstdio>
#include <ctime>
int main() {
  Stream st;
  const size_t sizes[] = {100, (8 << 20) - 1, 8 << 20, (9 << 20) + 5, (40 << 20) + 12345};
  VwXfer x;
  x.reserve(64 << 20);
  int bad = 0;
  for (size_t n : sizes)
    for (int seg = 1; seg <= 3; ++seg) {
      std::vector<std::vector<char>> d(seg), h(seg);
      VwXfer::Seg s[3];
      for (int i = 0; i < seg; ++i) {
        d[i].resize(n + 3 * i); h[i].assign(n + 3 * i, 0);
        for (size_t k = 0; k < d[i].size(); ++k) d[i][k] = (char)(k * 2654435761u >> 7) + i;
        s[i] = {h[i].data(), d[i].data(), d[i].size()};
      }
      if (x.out(s, seg, &st) != hipSuccess) ++bad;
      st.wait();
      for (int i = 0; i < seg; ++i) bad += h[i] != d[i];
    }
  std::vector<char> d(20 << 20, 7), h(20 << 20);
  VwXfer::Seg s = {h.data(), d.data(), d.size()};
  g_kernel = true;
  st.push([] { std::this_thread::sleep_for(std::chrono::milliseconds(300)); std::lock_guard<std::mutex> l(g_m); g_kernel = false; });
  const clock_t c0 = clock();
  if (x.out(&s, 1, &st) != hipSuccess) ++bad;
  const double cpu = (double)(clock() - c0) / CLOCKS_PER_SEC;
  st.wait();
  bad += h != d;
  /* a copy that cannot be issued: an error, and the next call works */
  for (int at : {0, 3, 19}) {
    std::vector<char> big(60 << 20, 5), out(60 << 20);
    VwXfer::Seg b = {out.data(), big.data(), big.size()};
    g_copies = 0; g_fail_at = at;
    if (x.out(&b, 1, &st) == hipSuccess) ++bad;
    g_fail_at = -1;
    if (x.out(&b, 1, &st) != hipSuccess) ++bad;
    st.wait();
    bad += out != big;
  }
  std::printf("%d %d %.3f\n", bad, g_max, cpu);
}
"""


def test_ring(tmp_path):
    """every byte arrives, and while the kernel before the results runs one thread waits for it, the caller, at no cost"""
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = tmp_path / "ring"
    csrc = os.path.join(ROOT, "viss_optimize_ws_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", str(tmp_path), "-I", csrc, str(tmp_path / "main.cpp"),
                    "-o", str(exe)], check=True)
    bad, waiting, cpu = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=60).stdout.split()
    assert int(bad) == 0
    assert int(waiting) == 1, f"{waiting} threads waited for the kernel"
    assert float(cpu) < 0.15, f"{cpu} s of CPU time in a wait of 0.3 s"
