// rgf_group_api.hpp -- launching one energy on a group of workgroups (rgf_group.hpp).
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

namespace rgf {

constexpr size_t kCtlBytes = 2048;  // control words of a group, of each of its halves
constexpr size_t kGroupCtlBytes = 3 * kCtlBytes;
constexpr int kXcds = 8;

constexpr int kGrpTile = 32;  // output tile of a group GEMM: 4 waves of one 16 x 16 MFMA tile

// Where the block is a multiple of 128 and the ranks are few, the 128 x 64 tiles of the
// one-workgroup GEMM are the better split: they read a third of the operands' panels and
// run at 80% of the MFMA rate against 54%, so one of them takes as long as 6.5 of the
// small ones (42 and 6.5 us at K = 128), not 8.
__host__ __device__ inline bool large_tiles(int n, int size) {
  if (n % 128 != 0) return false;
  const int small = (n / kGrpTile) * (n / kGrpTile), large = small / 8;
  return 13 * ((large + size - 1) / size) < 2 * ((small + size - 1) / size);
}

struct GroupArgs {
  int ngroups, size, per_xcd;
  int e0;       // first energy of the launch
  int grid;
  char* ctl;    // ngroups control areas of kGroupCtlBytes
};

struct SweepArgs;
struct AdjArgs;
struct WArgs;

// Many devices with at most kMultiGroupItems (device, energy) items per compute unit:
// groups of workgroups with lists of items, sizes and lists by the items' costs.
constexpr int kMultiGroupItems = 2;
struct MultiGroupArgs {
  const SweepArgs* jobs;
  const int2* items;       // (device, energy), group by group
  const int* first;        // group g runs items first[g] .. first[g + 1] - 1
  const int* sizes;        // workgroups of each group
  const int* block_group;  // group of each block, -1: none
  int ngroups;
  char* ctl;
  double2* ws;
  long long ws_slot;
};
struct MultiGroupPlan {
  std::vector<int> sizes, first, block_group;
  std::vector<int> order;  // the items, group by group
};

// Groups for nE energies of n orbitals on `cus` compute units; false where one workgroup
// per energy is the faster (or only) form.
bool group_plan(int n, long long nE, int cus, GroupArgs* g);
// 32 orbitals: two workgroups for each of nE energies (launch_sweep_grp, without
// block-tridiagonal Sigma); a slot has kPairExtra more blocks.
bool pair_plan(int n, long long nE, int cus, GroupArgs* g);
constexpr int kPairExtra = 11;

// Clear the control areas and launch.  The areas belong to the launch until it ends.
hipError_t launch_sweep_grp(const SweepArgs& a, const GroupArgs& g, bool od, hipStream_t s);
hipError_t launch_adjoint_grp(const AdjArgs& a, const GroupArgs& g, hipStream_t s);
hipError_t launch_wsweep_grp(const WArgs& a, const GroupArgs& g, hipStream_t s);

// The groups for items of n[i] orbitals and nx[i] slabs, longest first; false where one
// workgroup per item is as fast.
bool multi_group_plan(const std::vector<int>& n, const std::vector<int>& nx, int cus, MultiGroupPlan* pl);
// Tile parameter (32 T, 4: 128 x 64) of the GEMMs that such a launch runs for n orbitals in a
// group of `size`.
inline int group_tile_T(int n, int size) { return n == 64 ? 2 : large_tiles(n, size) ? 4 : 1; }
hipError_t launch_multi_grp(const MultiGroupArgs& m, int blocks, hipStream_t s);

}  // namespace rgf
