/*
 * vw_xfer.h -- device results into the caller's pageable host memory.
 *
 * A plain hipMemcpyAsync to pageable memory goes through the runtime's staging
 * buffer with one thread copying, and with freshly allocated arrays that thread
 * takes every page fault too: about 11 GB/s, 12.5 ms of a 34 ms call that
 * returns 134 MB of maps.  VwXfer keeps a bounded ring of pinned slots per
 * owner: the caller's thread issues the device copies slot by slot, and helper
 * threads move finished slots on, so the faults and the copy run on several
 * cores while the next slots arrive.
 *
 * One owner (context or network) uses its VwXfer from one thread at a time, as
 * it does its streams.  Nothing here throws; where threads or pinned memory
 * cannot be had the copies are plain ones.
 */
#ifndef VW_XFER_H
#define VW_XFER_H

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

class VwXfer {
 public:
  struct Seg {
    void* host;
    const void* dev;
    size_t bytes;
  };
  VwXfer() = default;
  VwXfer(const VwXfer&) = delete;
  VwXfer& operator=(const VwXfer&) = delete;
  ~VwXfer() { release(); }

  /* a pinned ring for results of up to `total` bytes a call (at most 32 MiB) */
  void reserve(size_t total) noexcept {
    const size_t want = std::min(kRing, (total + kChunkMin - 1) / kChunkMin * kChunkMin);
    if (total < kPlain || want <= ring_bytes_) return;
    release_ring();
    if (hipHostMalloc((void**)&ring_, want, hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      ring_ = nullptr;
      return;
    }
    ring_bytes_ = want;
    for (; nev_ < kSlots; ++nev_)
      if (hipEventCreateWithFlags(&ev_[nev_], hipEventDisableTiming) != hipSuccess) {
        (void)hipGetLastError();
        break;
      }
  }

  /* the segments' device memory, as it is when st gets there, into their host
   * memory, which is filled once the caller has waited for st */
  hipError_t out(const Seg* segs, int n, hipStream_t st) noexcept {
    size_t total = 0;
    for (int i = 0; i < n; ++i) total += segs[i].bytes;
    if (!total) return hipSuccess;
    chunk_ = std::min(kChunkMax, std::max(kChunkMin, total / 8 / kChunkMin * kChunkMin));
    nslot_ = (int)std::min<size_t>((size_t)nev_, ring_bytes_ / chunk_);
    if (nslot_ < 2 || total < kPlain || n > kSegs) {
      for (int i = 0; i < n; ++i)
        if (segs[i].bytes) {
          const hipError_t e = hipMemcpyAsync(segs[i].host, segs[i].dev, segs[i].bytes, hipMemcpyDeviceToHost, st);
          if (e != hipSuccess) return e;
        }
      return hipSuccess;
    }
    /* chunk c of segment i: first_[i] <= c < first_[i + 1] */
    nseg_ = n;
    first_[0] = 0;
    for (int i = 0; i < n; ++i) {
      seg_[i] = segs[i];
      first_[i + 1] = first_[i] + (int64_t)((segs[i].bytes + chunk_ - 1) / chunk_);
    }
    nchunk_ = first_[n];
    next_.store(0);
    issued_.store(0);
    err_.store(0);
    for (int s = 0; s < nslot_; ++s) slot_done_[s].store(-1);
    hipError_t e = hipSuccess;
    int64_t c = 0;
    auto issue = [&] {
      const int s = (int)(c % nslot_);
      const Seg g = chunk(c);
      e = hipMemcpyAsync(ring_ + chunk_ * (size_t)s, g.dev, g.bytes, hipMemcpyDeviceToHost, st);
      if (e == hipSuccess) e = hipEventRecord(ev_[s], st);
      if (e == hipSuccess) issued_.store(++c, std::memory_order_release);
    };
    while (c < nslot_ && c < nchunk_ && e == hipSuccess) issue();
    /* the kernels before the results may run for long: until the first chunk is
     * there this thread waits alone, as for a plain copy, and no helper polls */
    if (e == hipSuccess) e = hipEventSynchronize(ev_[0]);
    const bool helped = e == hipSuccess && start();
    while (c < nchunk_ && e == hipSuccess) {
      const int s = (int)(c % nslot_);
      /* the slot's last chunk has to be out: take a chunk on meanwhile */
      while (slot_done_[s].load(std::memory_order_acquire) != c - nslot_) {
        int64_t k = next_.load();
        if (k < c && next_.compare_exchange_strong(k, k + 1)) finish(k);
        else pause();
      }
      issue();
    }
    if (e != hipSuccess) {
      err_.store(1);
      issued_.store(nchunk_, std::memory_order_release);
    }
    for (int64_t k; (k = next_.fetch_add(1)) < nchunk_;) finish(k);
    if (helped) wait_helpers();
    if (e == hipSuccess && err_.load()) e = hipErrorUnknown;
    if (e != hipSuccess) (void)hipStreamSynchronize(st); /* no copy into the ring is left in flight */
    return e;
  }

 private:
  /* Measured into fresh pages, plain copy against this, us: 134 MB 12,500 3,420;
   * 22 MB 2,160 700; 9.4 MB 1,010 430.  Results of a few MB gain only into fresh
   * pages (2.1 MB 473 270), not into a program's recycled arrays (5.5 MB of Nside
   * 128 maps 464 461; with the 1.7 MB of an ordinary training pair the call went
   * from 712 to 814), so they stay plain.  2 MiB chunks keep the copies' launch and event
   * (20 us together, 9.9 ms for 134 MB in 256 KiB chunks) below their 40 us;
   * the smallest results take smaller ones so that four threads share them.
   * 7 or 11 helpers measured the same. */
  static constexpr size_t kPlain = 8 << 20, kChunkMin = 256 << 10, kChunkMax = 2 << 20, kRing = 32 << 20;
  static constexpr int kSlots = 64, kSegs = 8, kThreads = 3;

  char* ring_ = nullptr;
  size_t ring_bytes_ = 0, chunk_ = kChunkMin;
  int nslot_ = 0, nev_ = 0; /* slots of the current call, events */
  hipEvent_t ev_[kSlots] = {};
  Seg seg_[kSegs] = {};
  int64_t first_[kSegs + 1] = {};
  int nseg_ = 0;
  int64_t nchunk_ = 0;
  std::atomic<int64_t> next_{0}, issued_{0}, slot_done_[kSlots] = {};
  std::atomic<int> err_{0};

  std::vector<std::thread> pool_;
  std::mutex mu_;
  std::condition_variable go_, idle_;
  uint64_t job_ = 0;
  int busy_ = 0;
  bool stop_ = false, open_ = false, no_pool_ = false;

  static void pause() { std::this_thread::yield(); }

  Seg chunk(int64_t c) const {
    int i = 0;
    while (c >= first_[i + 1]) ++i;
    const size_t off = chunk_ * (size_t)(c - first_[i]);
    return {(char*)seg_[i].host + off, (const char*)seg_[i].dev + off, std::min(chunk_, seg_[i].bytes - off)};
  }

  /* chunk c, claimed by this thread, from its slot to the caller's memory */
  void finish(int64_t c) {
    while (issued_.load(std::memory_order_acquire) <= c) pause();
    const int s = (int)(c % nslot_);
    if (!err_.load()) {
      if (hipEventSynchronize(ev_[s]) == hipSuccess) {
        const Seg g = chunk(c);
        std::memcpy(g.host, ring_ + chunk_ * (size_t)s, g.bytes);
      } else {
        err_.store(1);
      }
    }
    slot_done_[s].store(c, std::memory_order_release);
  }

  bool start() noexcept {
    if (pool_.empty() && !no_pool_) {
      const int n = std::min<int>(kThreads, (int)std::thread::hardware_concurrency() / 2);
      try {
        for (int i = 0; i < n; ++i) pool_.emplace_back([this] { helper(); });
      } catch (...) {
      }
      no_pool_ = pool_.empty();
    }
    if (pool_.empty()) return false;
    {
      std::lock_guard<std::mutex> lk(mu_);
      ++job_;
      open_ = true;
    }
    go_.notify_all();
    return true;
  }
  /* helpers that have not woken by now stay out of this call */
  void wait_helpers() {
    std::unique_lock<std::mutex> lk(mu_);
    open_ = false;
    idle_.wait(lk, [this] { return busy_ == 0; });
  }
  void helper() {
    uint64_t seen = 0;
    for (;;) {
      {
        std::unique_lock<std::mutex> lk(mu_);
        go_.wait(lk, [&] { return stop_ || (open_ && job_ != seen); });
        if (stop_) return;
        seen = job_;
        ++busy_;
      }
      for (int64_t k; (k = next_.fetch_add(1)) < nchunk_;) finish(k);
      std::lock_guard<std::mutex> lk(mu_);
      if (--busy_ == 0) idle_.notify_one();
    }
  }
  void release_ring() {
    if (ring_) (void)hipHostFree(ring_);
    ring_ = nullptr;
    ring_bytes_ = 0;
  }
  void release() {
    {
      std::lock_guard<std::mutex> lk(mu_);
      stop_ = true;
    }
    go_.notify_all();
    for (std::thread& t : pool_) t.join();
    pool_.clear();
    for (; nev_ > 0; --nev_) (void)hipEventDestroy(ev_[nev_ - 1]);
    release_ring();
  }
};

#endif
