// Arrays of the given sizes to the device and back, as the host-array entry points copy them.
#include "rgf_hostcopy.hpp"

extern "C" int host_copy(int fail_pinned, int rounds, int n, const size_t* sizes, const char* src, char* dev, char* dst) {
  host_hip().fail_pinned = fail_pinned != 0;
  rgf::PinnedAreas areas;
  size_t total = 0;
  for (int i = 0; i < n; ++i) total += sizes[i];
  (void)areas.ensure(total);
  for (int r = 0; r < rounds; ++r) {
    rgf::HostCopier copier(areas, 0);
    size_t o = 0;
    for (int i = 0; i < n; o += sizes[i++])
      if (int e = copier.to_device(dev + o, src + o, sizes[i])) return e;
    o = 0;
    for (int i = 0; i < n; o += sizes[i++])
      if (int e = copier.to_host(dst + o, dev + o, sizes[i])) return e;
    if (int e = copier.finish()) return e;
  }
  areas.release();
  return 0;
}
