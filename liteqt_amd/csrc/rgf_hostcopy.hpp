// rgf_hostcopy.hpp -- copies between the caller's ordinary host arrays and the device
// through pinned areas.
//
// A copy to or from pageable memory is staged by the runtime on the calling thread, one
// array after the other (5.8 GB/s measured into freshly allocated arrays, whose pages the
// copy touches first), with a synchronisation each.  Here the DMA of one pinned area runs
// while several threads move the other area's contents, and small arrays share an area
// and a synchronisation.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace rgf {

// Two pinned areas, kept between calls (at most 2 x kMax bytes a device) and given back
// with the other buffers.  Used by one call at a time (the caller holds the lock).
struct PinnedAreas {
  static constexpr size_t kMax = size_t(16) << 20, kMin = size_t(256) << 10;
  char* p[2] = {nullptr, nullptr};
  hipEvent_t done[2] = {nullptr, nullptr};
  bool busy[2] = {false, false};  // a DMA of the area may be under way
  size_t bytes = 0;
  // Areas for calls of `total` bytes; none (bytes = 0) where they cannot be allocated.
  hipError_t ensure(size_t total) {
    const size_t want = std::min(kMax, std::max(kMin, (total + 4095) / 4096 * 4096));
    if (want <= bytes) return hipSuccess;
    release();
    for (int i = 0; i < 2; ++i) {
      hipError_t e = hipHostMalloc(reinterpret_cast<void**>(&p[i]), want, hipHostMallocDefault);
      if (e == hipSuccess) e = hipEventCreateWithFlags(&done[i], hipEventDisableTiming);
      if (e != hipSuccess) {
        release();
        return e;
      }
    }
    bytes = want;
    return hipSuccess;
  }
  hipError_t wait(int i) {
    if (!busy[i]) return hipSuccess;
    busy[i] = false;
    return hipEventSynchronize(done[i]);
  }
  void release() {
    for (int i = 0; i < 2; ++i) {
      (void)wait(i);
      if (done[i]) (void)hipEventDestroy(done[i]);
      if (p[i]) (void)hipHostFree(p[i]);
      done[i] = nullptr;
      p[i] = nullptr;
    }
    bytes = 0;
  }
};

// memcpy jobs run by the calling thread and up to kThreads - 1 helpers, which are started
// with the first large batch of a call and end with it.
class CopyTeam {
 public:
  struct Job {
    void* dst;
    const void* src;
    size_t bytes;
  };
  void run(const std::vector<Job>& jobs) {
    size_t total = 0;
    for (const Job& j : jobs) total += j.bytes;
    if (total < kLarge) {
      for (const Job& j : jobs) std::memcpy(j.dst, j.src, j.bytes);
      return;
    }
    start();
    {
      std::lock_guard<std::mutex> lk(mu_);
      parts_.clear();
      for (const Job& j : jobs)
        for (size_t o = 0; o < j.bytes; o += kPart)
          parts_.push_back(Job{static_cast<char*>(j.dst) + o, static_cast<const char*>(j.src) + o, std::min(kPart, j.bytes - o)});
      next_ = 0;
      running_ = (int)team_.size();
      ++round_;
    }
    go_.notify_all();
    work();
    std::unique_lock<std::mutex> lk(mu_);
    idle_.wait(lk, [&] { return running_ == 0; });
  }
  ~CopyTeam() {
    {
      std::lock_guard<std::mutex> lk(mu_);
      stop_ = true;
    }
    go_.notify_all();
    for (std::thread& t : team_) t.join();
  }

 private:
  static constexpr size_t kLarge = size_t(4) << 20, kPart = size_t(512) << 10;
  static constexpr int kThreads = 8;
  std::vector<std::thread> team_;
  std::vector<Job> parts_;
  std::mutex mu_;
  std::condition_variable go_, idle_;
  std::atomic<size_t> next_{0};
  int running_ = 0;
  unsigned round_ = 0;
  bool started_ = false, stop_ = false;
  void work() {
    for (size_t i; (i = next_.fetch_add(1)) < parts_.size();) std::memcpy(parts_[i].dst, parts_[i].src, parts_[i].bytes);
  }
  void start() {
    if (started_) return;
    started_ = true;
    const int want = std::min<int>(kThreads, (int)std::max(1u, std::thread::hardware_concurrency())) - 1;
    try {
      for (int i = 0; i < want; ++i)
        team_.emplace_back([this] {
          unsigned seen = 0;
          for (;;) {
            {
              std::unique_lock<std::mutex> lk(mu_);
              go_.wait(lk, [&] { return stop_ || round_ != seen; });
              if (stop_) return;
              seen = round_;
            }
            work();
            std::lock_guard<std::mutex> lk(mu_);
            if (--running_ == 0) idle_.notify_one();
          }
        });
    } catch (...) {  // fewer helpers: the calling thread takes what is left
    }
  }
};

// A stream's copies through the areas: to_device / to_host queue a copy, finish completes
// the copies to the host (those to the device complete in stream order).  Without areas
// (pinned memory can run out before the host's does) the copies are the runtime's own.
class HostCopier {
 public:
  HostCopier(PinnedAreas& areas, hipStream_t s) : a_(areas), s_(s) {}
  ~HostCopier() { (void)close(); }  // after an error: the next user waits for the queued DMA
  hipError_t to_device(void* dst, const void* src, size_t bytes) {
    if (!a_.bytes) return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s_);
    for (size_t o = 0; o < bytes;) {
      if (hipError_t e = open(false)) return e;
      const size_t b = std::min(bytes - o, a_.bytes - used_);
      char* stage = a_.p[cur_] + used_;
      team_.run({CopyTeam::Job{stage, static_cast<const char*>(src) + o, b}});
      if (hipError_t e = hipMemcpyAsync(static_cast<char*>(dst) + o, stage, b, hipMemcpyHostToDevice, s_)) return e;
      used_ += b;
      o += b;
    }
    return hipSuccess;
  }
  hipError_t to_host(void* dst, const void* src, size_t bytes) {
    if (!a_.bytes) return hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s_);
    for (size_t o = 0; o < bytes;) {
      if (hipError_t e = open(true)) return e;
      const size_t b = std::min(bytes - o, a_.bytes - used_);
      char* stage = a_.p[cur_] + used_;
      if (hipError_t e = hipMemcpyAsync(stage, static_cast<const char*>(src) + o, b, hipMemcpyDeviceToHost, s_)) return e;
      out_[cur_].push_back(CopyTeam::Job{static_cast<char*>(dst) + o, stage, b});
      used_ += (b + 255) / 256 * 256;
      o += b;
    }
    return hipSuccess;
  }
  hipError_t finish() {
    if (!a_.bytes) return hipStreamSynchronize(s_);
    if (hipError_t e = close()) return e;
    if (hipError_t e = land(cur_ ^ 1)) return e;
    return land(cur_);
  }

 private:
  PinnedAreas& a_;
  hipStream_t s_;
  CopyTeam team_;
  std::vector<CopyTeam::Job> out_[2];  // copies waiting for their area's DMA
  int cur_ = 0;
  size_t used_ = 0;
  bool open_ = false;
  // an area with room: the current one, or the other once its DMA is over and its
  // contents are with the caller
  hipError_t open(bool host) {
    if (open_ && used_ < a_.bytes && host_ == host) return hipSuccess;
    if (open_) {
      if (hipError_t e = close()) return e;
      cur_ ^= 1;
    }
    if (hipError_t e = land(cur_)) return e;
    open_ = true;
    host_ = host;
    used_ = 0;
    return hipSuccess;
  }
  hipError_t close() {
    if (!open_) return hipSuccess;
    open_ = false;
    a_.busy[cur_] = true;
    return hipEventRecord(a_.done[cur_], s_);
  }
  hipError_t land(int i) {
    if (hipError_t e = a_.wait(i)) return e;
    team_.run(out_[i]);
    out_[i].clear();
    return hipSuccess;
  }
  bool host_ = false;
};

}  // namespace rgf
