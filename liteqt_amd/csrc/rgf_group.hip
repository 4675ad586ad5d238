// rgf_group.hip -- host side of the group kernels: when a solve uses them, and their launch.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <map>
#include <utility>
#include <vector>

#include "rgf_group.hpp"

namespace rgf {

namespace {

__global__ void clear_ctl(unsigned* p, int n) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0u;
}

hipError_t clear(char* ctl, int ngroups, hipStream_t s) {
  const int words = (int)(kGroupCtlBytes / 4) * ngroups;
  hipLaunchKernelGGL(clear_ctl, dim3((words + 255) / 256), dim3(256), 0, s, reinterpret_cast<unsigned*>(ctl), words);
  return hipGetLastError();
}

// Microseconds of one energy on a group of G workgroups: the measured times of the block
// operations as functions of the block size, a slab of 16 GEMMs and an inverse, 18
// decimation iterations of 6 GEMMs and an inverse per contact, each on half of the group.
// GEMM from 96 orbitals: barrier 4, 1.6 us per 32 x 32 tile and K panel, or 0.33 us per
// 128 x 64 tile and k; inverse: the column steps (134 us at 128, 475 at 256) and 12 (128)
// or 62 us (256) per round of the strips.  32 and 64 orbitals run on one workgroup.
double item_us(int n, int nx, int G) {
  const int t = n / 32;
  auto us = [&](int gemms, int ranks) {
    const double bar = ranks > 1 ? 4.0 : 0.5;
    double gemm = bar + ((t * t + ranks - 1) / ranks) * 1.6 * t;
    const double strip = (n <= 128 ? 12.0 / 16384.0 : 62.0 / 65536.0) * n * n;
    double inv = (n <= 128 ? 1.05 : 1.85) * n + 4 * bar + ((n / 16 + ranks - 1) / ranks) * strip;
    if (n % 128 == 0) gemm = std::min(gemm, bar + ((t * t / 8 + ranks - 1) / ranks) * 0.33 * n);
    if (n < 96) {
      gemm = n == 64 ? 14.0 : 6.0;
      inv = 1.2 * n;
    }
    return gemms * gemm + inv;
  };
  return nx * us(16, G) + 18 * (G > 1 ? us(6, G / 2) : 2 * us(6, 1));
}

}  // namespace

bool group_plan(int n, long long nE, int cus, GroupArgs* g) {
  if (n % 32 != 0 || n < 64 || n > 256 || nE < 1 || cus % kXcds != 0) return false;
  const int per = cus / kXcds;                     // compute units of an XCD
  const int rows = (int)((nE + kXcds - 1) / kXcds);  // groups of an XCD
  if (2 * rows > per) return false;                // two workgroups per energy at the least
  const int tiles = (n / kGrpTile) * (n / kGrpTile);
  g->size = std::min(per / rows, tiles);
  g->per_xcd = rows;
  g->ngroups = (int)nE;
  g->e0 = 0;
  g->grid = kXcds * rows * g->size;
  g->ctl = nullptr;
  return true;
}

bool pair_plan(int n, long long nE, int cus, GroupArgs* g) {
  if (n != 32 || nE < 1 || cus % kXcds != 0) return false;
  const int rows = (int)((nE + kXcds - 1) / kXcds);
  if (2 * rows > cus / kXcds) return false;  // a compute unit for each workgroup
  *g = GroupArgs{(int)nE, 2, rows, 0, kXcds * rows * 2, nullptr};
  return true;
}

static_assert(kPairExtra == kSanchoBlocks, "the right decimation's temporaries");

hipError_t launch_sweep_grp(const SweepArgs& a, const GroupArgs& g, bool od, hipStream_t s) {
  if (hipError_t e = clear(g.ctl, g.ngroups, s)) return e;
  if (a.n == 32) {
    hipLaunchKernelGGL((rgf_sweep_pair<kPair32, 32>), dim3(g.grid), dim3(256), 0, s, a, g);
  } else if (od) {
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
  if (hipError_t e = clear(g.ctl, g.ngroups, s)) return e;
  if (a.n <= 128)
    hipLaunchKernelGGL(rgf_adjoint_grp<128>, dim3(g.grid), dim3(256), 0, s, a, g);
  else
    hipLaunchKernelGGL(rgf_adjoint_grp<256>, dim3(g.grid), dim3(256), 0, s, a, g);
  return hipGetLastError();
}

hipError_t launch_wsweep_grp(const WArgs& a, const GroupArgs& g, hipStream_t s) {
  if (hipError_t e = clear(g.ctl, g.ngroups, s)) return e;
  if (a.n <= 128)
    hipLaunchKernelGGL(rgf_wsweep_grp<128>, dim3(g.grid), dim3(256), 0, s, a, g);
  else
    hipLaunchKernelGGL(rgf_wsweep_grp<256>, dim3(g.grid), dim3(256), 0, s, a, g);
  return hipGetLastError();
}

bool multi_group_plan(const std::vector<int>& n, const std::vector<int>& nx, int cus, MultiGroupPlan* pl) {
  const int count = (int)n.size(), per = cus / kXcds;
  if (count < 1 || count > kMultiGroupItems * cus || cus % kXcds != 0) return false;
  // one workgroup per item: the longest, and the work of all
  double longest = 0.0, work = 0.0;
  std::map<std::pair<int, int>, std::vector<double>> cost;  // (n, nx) -> time by group size
  std::vector<const std::vector<double>*> us(count);
  for (int i = 0; i < count; ++i) {
    std::vector<double>& c = cost[{n[i], nx[i]}];
    if (c.empty()) {
      const int t = n[i] / 32, most = n[i] < 96 ? 1 : std::min(per, t * t);
      for (int G = 1; G <= most; ++G) c.push_back(item_us(n[i], nx[i], G));
    }
    us[i] = &c;
    longest = std::max(longest, c[0]);
    work += c[0];
  }
  struct Bin {
    int size;
    double left;
    std::vector<int> items;
  };
  std::vector<Bin> bins;
  std::vector<int> xcd;
  // first fit of the items, longest first, into groups that end by `limit`: a group that
  // has the time left for the item at its own size, or a new one of the smallest size
  // that makes it; then the groups, largest first, onto the XCDs
  auto fit = [&](double limit) {
    bins.clear();
    int total = 0;
    for (int i = 0; i < count; ++i) {
      const std::vector<double>& c = *us[i];
      Bin* to = nullptr;
      for (Bin& b : bins)
        if (b.size <= (int)c.size() && c[b.size - 1] <= b.left) {
          to = &b;
          break;
        }
      if (!to) {
        int G = 1;
        while (G <= (int)c.size() && c[G - 1] > limit) ++G;
        if (G > (int)c.size() || (total += G) > cus) return false;
        bins.push_back(Bin{G, limit, {}});
        to = &bins.back();
      }
      to->left -= c[to->size - 1];
      to->items.push_back(i);
    }
    std::stable_sort(bins.begin(), bins.end(), [](const Bin& x, const Bin& y) { return x.size > y.size; });
    int used[kXcds] = {};
    xcd.assign(bins.size(), 0);
    for (size_t g = 0; g < bins.size(); ++g) {
      const int x = (int)(std::min_element(used, used + kXcds) - used);
      if (used[x] + bins[g].size > per) return false;
      used[x] += bins[g].size;
      xcd[g] = x;
    }
    return true;
  };
  const double single = std::max(longest, work / cus);
  double lo = 0.0, hi = 2.0 * single;
  if (!fit(hi)) return false;
  for (int k = 0; k < 16; ++k) {
    const double mid = 0.5 * (lo + hi);
    (fit(mid) ? hi : lo) = mid;
  }
  if (hi > 0.9 * single || !fit(hi)) return false;
  pl->block_group.assign(cus, -1);
  pl->first.assign(1, 0);
  int used[kXcds] = {};
  for (size_t g = 0; g < bins.size(); ++g) {
    pl->sizes.push_back(bins[g].size);
    pl->order.insert(pl->order.end(), bins[g].items.begin(), bins[g].items.end());
    pl->first.push_back((int)pl->order.size());
    for (int r = 0; r < bins[g].size; ++r) pl->block_group[kXcds * used[xcd[g]]++ + xcd[g]] = (int)g;
  }
  return true;
}

hipError_t launch_multi_grp(const MultiGroupArgs& m, int blocks, hipStream_t s) {
  if (hipError_t e = clear(m.ctl, m.ngroups, s)) return e;
  hipLaunchKernelGGL(rgf_sweep_multi_grp, dim3(blocks), dim3(256), 0, s, m);
  return hipGetLastError();
}

}  // namespace rgf
