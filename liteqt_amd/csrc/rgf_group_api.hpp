// rgf_group_api.hpp -- launching one energy on a group of workgroups (rgf_group.hpp).
#pragma once
#include <hip/hip_runtime.h>

namespace rgf {

constexpr size_t kGroupCtlBytes = 2048;

struct GroupArgs {
  int ngroups, size, per_xcd, spread;
  int e0;       // first energy of the launch
  int grid;
  char* ctl;    // ngroups control areas of kGroupCtlBytes
};

struct SweepArgs;
struct AdjArgs;
struct WArgs;

// Groups for nE energies of n orbitals on `cus` compute units; false where one workgroup
// per energy is the faster (or only) form.
bool group_plan(int n, long long nE, int cus, GroupArgs* g);

// Clear the control areas (a kernel, so that the launch can be captured) and launch.
hipError_t launch_sweep_grp(const SweepArgs& a, const GroupArgs& g, bool od, hipStream_t s);
hipError_t launch_adjoint_grp(const AdjArgs& a, const GroupArgs& g, hipStream_t s);
hipError_t launch_wsweep_grp(const WArgs& a, const GroupArgs& g, hipStream_t s);

}  // namespace rgf
