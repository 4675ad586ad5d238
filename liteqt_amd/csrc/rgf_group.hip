// rgf_group.hip -- host side of the group kernels: when a solve uses them, and their launch.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "rgf_group.hpp"

namespace rgf {

namespace {

__global__ void clear_ctl(unsigned* p, int n) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0u;
}

hipError_t clear(const GroupArgs& g, hipStream_t s) {
  const int words = (int)(kGroupCtlBytes / 4) * g.ngroups;
  hipLaunchKernelGGL(clear_ctl, dim3((words + 255) / 256), dim3(256), 0, s, reinterpret_cast<unsigned*>(g.ctl), words);
  return hipGetLastError();
}

}  // namespace

bool group_plan(int n, long long nE, int cus, GroupArgs* g) {
  constexpr int kXcds = 8;
  if (n % 32 != 0 || n < 96 || n > 256 || nE < 1 || cus % kXcds != 0) return false;
  const int per = cus / kXcds;                     // compute units of an XCD
  const int rows = (int)((nE + kXcds - 1) / kXcds);  // groups of an XCD
  if (2 * rows > per) return false;                // two workgroups per energy at the least
  const int tiles = (n / kGrpTile) * (n / kGrpTile);
  g->size = std::min(per / rows, tiles);
  g->per_xcd = rows;
  g->ngroups = (int)nE;
  g->spread = 0;
  g->e0 = 0;
  g->grid = kXcds * rows * g->size;
  g->ctl = nullptr;
  return true;
}

hipError_t launch_sweep_grp(const SweepArgs& a, const GroupArgs& g, bool od, hipStream_t s) {
  if (hipError_t e = clear(g, s)) return e;
  if (od) {
    if (a.n <= 128)
      hipLaunchKernelGGL(rgf_sweep_od_grp<128>, dim3(g.grid), dim3(256), 0, s, a, g);
    else
      hipLaunchKernelGGL(rgf_sweep_od_grp<256>, dim3(g.grid), dim3(256), 0, s, a, g);
  } else if (a.n <= 128) {
    hipLaunchKernelGGL(rgf_sweep_grp<128>, dim3(g.grid), dim3(256), 0, s, a, g);
  } else {
    hipLaunchKernelGGL(rgf_sweep_grp<256>, dim3(g.grid), dim3(256), 0, s, a, g);
  }
  return hipGetLastError();
}

hipError_t launch_adjoint_grp(const AdjArgs& a, const GroupArgs& g, hipStream_t s) {
  if (hipError_t e = clear(g, s)) return e;
  if (a.n <= 128)
    hipLaunchKernelGGL(rgf_adjoint_grp<128>, dim3(g.grid), dim3(256), 0, s, a, g);
  else
    hipLaunchKernelGGL(rgf_adjoint_grp<256>, dim3(g.grid), dim3(256), 0, s, a, g);
  return hipGetLastError();
}

hipError_t launch_wsweep_grp(const WArgs& a, const GroupArgs& g, hipStream_t s) {
  if (hipError_t e = clear(g, s)) return e;
  if (a.n <= 128)
    hipLaunchKernelGGL(rgf_wsweep_grp<128>, dim3(g.grid), dim3(256), 0, s, a, g);
  else
    hipLaunchKernelGGL(rgf_wsweep_grp<256>, dim3(g.grid), dim3(256), 0, s, a, g);
  return hipGetLastError();
}

}  // namespace rgf
