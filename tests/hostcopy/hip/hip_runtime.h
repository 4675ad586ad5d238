// Stand-in for the HIP calls of liteqt_amd/csrc/rgf_hostcopy.hpp, test infrastructure.  One
// stream on the host: a copy of pinned memory runs when the stream or a later event of it is
// waited for, a copy of other memory at once.  Pinned allocations can be made to fail.
#pragma once
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <vector>

typedef int hipError_t;
typedef int hipStream_t;
typedef size_t* hipEvent_t;  // copies queued when it was recorded
enum { hipSuccess = 0, hipErrorOutOfMemory = 2, hipHostMallocDefault = 0, hipEventDisableTiming = 2 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };

struct HostHip {
  struct Copy {
    void* dst;
    const void* src;
    size_t bytes;
  };
  struct Range {
    char* p;
    size_t bytes;
  };
  std::vector<Copy> queue;
  size_t done = 0;
  std::vector<Range> pinned;
  bool fail_pinned = false;
  bool is_pinned(const void* q) const {
    for (const Range& r : pinned)
      if (q >= r.p && q < r.p + r.bytes) return true;
    return false;
  }
  void run_to(size_t n) {
    for (; done < n; ++done) std::memcpy(queue[done].dst, queue[done].src, queue[done].bytes);
  }
};
inline HostHip& host_hip() {
  static HostHip h;
  return h;
}

inline hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
  if (host_hip().fail_pinned) return hipErrorOutOfMemory;
  *p = std::malloc(bytes);
  std::memset(*p, 0x5a, bytes);
  host_hip().pinned.push_back({static_cast<char*>(*p), bytes});
  return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
  std::vector<HostHip::Range>& v = host_hip().pinned;
  for (size_t i = 0; i < v.size(); ++i)
    if (v[i].p == p) v.erase(v.begin() + i);
  std::free(p);
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = new size_t(0);
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
  delete e;
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  *e = host_hip().queue.size();
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
  host_hip().run_to(*e);
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t) {
  host_hip().run_to(host_hip().queue.size());
  return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind, hipStream_t s) {
  HostHip& h = host_hip();
  h.queue.push_back({dst, src, bytes});
  return h.is_pinned(dst) || h.is_pinned(src) ? hipSuccess : hipStreamSynchronize(s);
}
