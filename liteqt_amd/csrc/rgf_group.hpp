// rgf_group.hpp -- one energy solved by a group of workgroups.
//
// The block program of an energy (solve_energy, solve_energy_od, adjoint_energy,
// w_energy) is a serial chain of block operations, which one workgroup runs on one
// compute unit.  With fewer energies than compute units the others idle, so here a group
// of workgroups runs the same program: every rank follows the whole control flow, a
// block operation's output tiles are dealt to the ranks, and the operation ends with a
// barrier of the group in place of the workgroup's.  The program is compiled unchanged
// with GroupN as the type of its block dimension (Dim<kGrp>), which selects the
// overloads below.
//
// Results do not depend on the number of ranks: an output element is formed by one wave
// from the same products in the same order as in the one-workgroup kernels, reductions
// over a block are formed by every rank for itself, and the one sum that is split (the sum of
// |C_ij| that the decimation and the contacts' Stein equations compare with their tolerances)
// is made of the same parts, one per 32 x 32 tile, added in the order of the tiles, whatever
// the GEMM's tiles are.  (The one-workgroup kernels add it in another order, so that next to
// the tolerance the two may differ by an iteration.)
//
// Membership.  A group is formed by the workgroups that have arrived when its first one
// closes it, so no workgroup ever waits for one that is not running, whatever else
// occupies the GPU: the first arrival (rank 0) waits for the others at most kJoinTicks,
// then publishes the number of members; a later arrival finds the group closed and
// leaves.  The members wait for rank 0's word, and at the barriers for each other, all of
// them resident workgroups that reach every barrier.  With rank 0 alone the program runs
// as in the one-workgroup kernels.
//
// A group barrier costs 4 us, 7 to 9 us with the write-back and refetch of the blocks
// (256 workgroups, groups of 2 to 32), against 84 us for a 128-orbital GEMM and 570 us
// for a 256-orbital one in one workgroup, 18 us for a 64-orbital and 8 for a 32-orbital one:
// groups are for blocks of 64 to 256 orbitals (64 orbitals, 20 slabs against a lone workgroup
// with a second one for the right contact: one energy 5.6 -> 3.9 ms, 60 energies 7.0 -> 5.5,
// 100 in groups of two 7.1 either way).  Members on one XCD share its L2, so their
// barriers leave the write-back out (read from the hardware when the group closes; 128
// orbitals, 18 slabs, one energy 9.9 -> 8.9 ms, 40 energies 17.7 -> 15.4; 96 orbitals, 120
// energies 28.0 -> 24.2).
#pragma once
#include "rgf_adjoint.hpp"
#include "rgf_group_api.hpp"
#include "rgf_offdiag.hpp"
#include "rgf_small.hpp"
#include "rgf_sweep.hpp"
#include "rgf_wsweep.hpp"

namespace rgf {

constexpr int kGrp = 64;          // variant code of the group kernels
constexpr int kGrpK = 32;         // its K panel
constexpr int kJoinTicks = 20000; // 200 us of the 100 MHz clock
constexpr int kMaxTiles = (256 / kGrpTile) * (256 / kGrpTile);

// Control words of one group, zero before the launch.
struct GroupCtl {
  unsigned arrivals, pad0[31];  // workgroups arrived, their XCDs (kXcdShift), kClosed: no more join
  unsigned members, pad1[31];   // the number of members and kOneXcd, written once
  unsigned barrier, pad2[31];   // arrivals at the barriers, all of them
  double part[2][kMaxTiles];    // partial sums of a GEMM's tiles, by barrier parity
  int lead[2][3];               // a contact's iterations, limit flag, singular inverses
};
// Arrivals: count in bits 0 .. 6, kClosed, then the sum of the arrivals' XCD numbers and the
// sum of their squares: the XCDs are equal where count * squares = sum^2.
constexpr unsigned kCount = 127u, kClosed = 1u << 7, kOneXcd = 1u << 16;
constexpr int kXcdShift = 8, kXcdSqShift = 17;  // up to 32 members: 9 and 12 bits
static_assert(sizeof(GroupCtl) <= kCtlBytes, "control area of a group");

struct GroupCtx {  // in LDS, one per workgroup
  GroupCtl* ctl;
  int rank, size;
  unsigned epoch;  // barriers passed
  unsigned half_epoch;  // barriers of this workgroup's half
  int one_xcd;          // the members share an L2
};

__device__ __forceinline__ GroupCtx* group_ctx() {
  __shared__ GroupCtx c;
  return &c;
}

// The block dimension of a group's program.
struct GroupN {
  int v;
  __device__ __forceinline__ GroupN(int n) : v(n) {}
  __device__ __forceinline__ operator int() const { return v; }
};
template <>
struct Dim<kGrp> {
  typedef GroupN type;
};

template <typename V>
__device__ __forceinline__ V agent_load(const V* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename V>
__device__ __forceinline__ void agent_store(V* p, V v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ int group_rank(GroupN) { return uni(group_ctx()->rank); }
__device__ __forceinline__ int group_size(GroupN) { return uni(group_ctx()->size); }
__device__ __forceinline__ bool group_leader(GroupN) { return group_ctx()->rank == 0; }
__device__ __forceinline__ int group_parity(GroupN) { return uni((int)(group_ctx()->epoch & 1u)); }

// Barrier of the group: every wave's stores are complete (in the L2) before the workgroup
// barrier, then one thread writes them back where the members do not share the L2 (agent
// release), counts the workgroup in and waits for the others, and drops the stale cache
// lines (agent acquire) before anyone reads on.
__device__ __noinline__ void group_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  __syncthreads();
  GroupCtx* c = group_ctx();
  if (threadIdx.x == 0) {
    const unsigned target = ++c->epoch * (unsigned)c->size;
    if (!c->one_xcd) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    __hip_atomic_fetch_add(&c->ctl->barrier, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    while ((int)(agent_load(&c->ctl->barrier) - target) < 0) __builtin_amdgcn_s_sleep(1);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  }
  __syncthreads();
}
__device__ __forceinline__ void group_sync(GroupN) { group_barrier(); }

// Join a group of `size` workgroups at control area ctl; false when it is closed (the
// workgroup leaves).
__device__ __forceinline__ bool group_join(char* area, int size) {
  GroupCtx* c = group_ctx();
  if (threadIdx.x == 0) {
    GroupCtl* ctl = reinterpret_cast<GroupCtl*>(area);
    const unsigned x = __builtin_amdgcn_s_getreg((31 << 11) | 20) & (kXcds - 1);  // XCC_ID
    const unsigned a = __hip_atomic_fetch_add(&ctl->arrivals, 1u + (x << kXcdShift) + (x * x << kXcdSqShift),
                                              __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    c->ctl = ctl;
    c->epoch = c->half_epoch = 0;
    c->rank = (int)(a & kCount);
    c->size = 0;
    unsigned m = 0;
    if (a == 0) {
      const unsigned long long t0 = wall_clock64();
      while ((agent_load(&ctl->arrivals) & kCount) < (unsigned)size &&
             wall_clock64() - t0 < (unsigned long long)kJoinTicks)
        __builtin_amdgcn_s_sleep(1);
      const unsigned f = __hip_atomic_fetch_add(&ctl->arrivals, kClosed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const unsigned sum = (f >> kXcdShift) & 511u, sq = f >> kXcdSqShift;
      m = f & kCount;
      if (m * sq == sum * sum) m |= kOneXcd;
      agent_store(&ctl->members, m);
    } else if (!(a & kClosed)) {
      while ((m = agent_load(&ctl->members)) == 0) __builtin_amdgcn_s_sleep(1);
    }
    c->size = (int)(m & kCount);
    c->one_xcd = (m & kOneXcd) != 0;
  }
  __syncthreads();
  return uni(c->size) > 0;
}

// The same by block index.  Workgroups are dealt to the XCDs in turn, so a group takes
// blocks of equal index mod 8: its ranks share an L2.
__device__ __forceinline__ bool group_join(const GroupArgs& g, int& grp) {
  const int b = blockIdx.x, q = (b / kXcds) / g.size;
  grp = q < g.per_xcd ? q * kXcds + b % kXcds : g.ngroups;
  if (grp >= g.ngroups) return false;
  return group_join(g.ctl + (size_t)grp * kGroupCtlBytes, g.size);
}

// ------------------------------------------------------------------- GEMM
// One 32 x 32 tile of C per workgroup and turn, K panels of 32 double-buffered in LDS and
// requested two panels ahead, across the rank's tiles: after a barrier the operands come
// from another CU's writes, and one panel's MFMAs (0.87 us) do not cover that latency.
// The tile is small so that a group of 16 covers a 128-orbital block.  The epilogue's D
// terms are requested with the tile's first panel.  The arithmetic of an element is
// wg_gemm_k's.
struct GrpGemm {
  static constexpr int LDR = kGrpTile + PAD, LDC = kGrpK + 2;  // row- / k-contiguous strides
  static constexpr int PLANE = (kGrpK * LDR > kGrpTile * LDC) ? kGrpK * LDR : kGrpTile * LDC;
  static constexpr int STAGE = 4 * PLANE, PER = kGrpTile * kGrpK / 256;
};
template <>
struct Cfg<kGrp> : Cfg<1> {};
template <>
struct GemmLds<kGrp> {
  static constexpr int DOUBLES = 2 * GrpGemm::STAGE > GemmLds<4>::DOUBLES ? 2 * GrpGemm::STAGE : GemmLds<4>::DOUBLES;
};

// The parts of a sum, one per tile (at most a wave's lanes), added in the order of the tiles.
__device__ __forceinline__ double tile_sum(const double* part, int ntiles) {
  static_assert(kMaxTiles <= 64, "a lane for each tile");
  const int lane = threadIdx.x & 63;
  const double v = lane < ntiles ? agent_load(part + lane) : 0.0;
  double s = 0.0;
  for (int t = 0; t < ntiles; ++t) s += lane_f64(v, t);
  return s;
}

__device__ __forceinline__ double group_abs(double2 v) { return sqrt(fma(v.y, v.y, v.x * v.x)); }

// Those parts from the 128 x 64 tiles: a wave's 64 x 32 part is two of the sum's tiles, each
// added as grp_gemm's four waves add it.
struct GroupSums {
  double* parts;
  int nt;
  double sum = 0.0, part = 0.0;  // of the 16 x 16 tile at work; lane b: of tile b
  __device__ __forceinline__ void add(double2 v) { sum += group_abs(v); }
  __device__ __forceinline__ void tile(int b) {
    sum = wave_sum(sum);
    part = (int)(threadIdx.x & 63) == b ? sum : part;
    sum = 0.0;
  }
  __device__ __forceinline__ void done(int row, int col) {
    static_assert(Cfg<4>::TA == 4 && Cfg<4>::TB == 2, "two 32 x 32 tiles per wave");
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      const double s = ((lane_f64(part, 4 * a) + lane_f64(part, 4 * a + 2)) + lane_f64(part, 4 * a + 1)) +
                       lane_f64(part, 4 * a + 3);
      if ((threadIdx.x & 63) == 0) agent_store(parts + row / kGrpTile + a + col / kGrpTile * nt, s);
    }
  }
};

template <int OPA, int OPB, int CRM>
__device__ __noinline__ double grp_gemm_large(GroupN n_, const double2* __restrict__ A, const double2* __restrict__ B,
                                              void* Cout, Epi ep, ldsd* lds) {
  const int rank = group_rank(n_), size = group_size(n_), parity = group_parity(n_);
  GroupCtl* ctl = uni(group_ctx()->ctl);
  const int nt = uni((int)n_) / kGrpTile;
  gemm_tiles<4, OPA, OPB, CRM>((int)n_, A, B, Cout, ep, lds, rank, size, GroupSums{ctl->part[parity], nt});
  group_barrier();
  return uni(ep.abs_sum) ? tile_sum(ctl->part[parity], nt * nt) : 0.0;
}

template <int OPA, int OPB, int CRM>
__device__ __noinline__ double grp_gemm(GroupN n_, const double2* __restrict__ A_, const double2* __restrict__ B_,
                                        void* Cout_, Epi ep_, ldsd* lds) {
  using L = GrpGemm;
  constexpr bool AKC = (OPA != OP_N), BKC = (OPB == OP_N);
  constexpr int LA = AKC ? L::LDC : L::LDR, LB = BKC ? L::LDC : L::LDR;
  const int n = uni((int)n_), rank = group_rank(n_), size = group_size(n_);
  const double2* A = uni(A_);
  const double2* B = uni(B_);
  void* Cout = uni(Cout_);
  Epi ep;
  ep.diag = uni(ep_.diag); ep.sacc = uni(ep_.sacc);
  ep.D1 = uni(ep_.D1); ep.s1 = uni(ep_.s1);
  ep.D2 = uni(ep_.D2); ep.s2 = uni(ep_.s2);
  ep.D3 = uni(ep_.D3); ep.s3 = uni(ep_.s3);
  ep.real_out = uni(ep_.real_out); ep.abs_sum = uni(ep_.abs_sum);
  const int parity = group_parity(n_);
  GroupCtl* ctl = uni(group_ctx()->ctl);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nt = n / kGrpTile, ntiles = nt * nt, np = n / kGrpK;
  const int arow = (wave & 1) * 16, bcol = (wave >> 1) * 16;
  const int m = lane & 15, kq = lane >> 4;
  // element q of a thread: fast index tid % 32, slow index tid / 32 + 8 q
  const int f = tid & 31, w8 = tid >> 5;
  // a rank's steps: panel s % np of its tile s / np.  Panel s is in LDS stage s & 1, panel
  // s + 1 in the other register set (requested a step ago), panel s + 2 being requested
  double2 ra[2][L::PER], rb[2][L::PER];
  const int mine = rank < ntiles ? (ntiles - rank + size - 1) / size : 0, steps = mine * np;
  int ftile = rank, fp = 0;  // tile and panel of the next fetch
  auto fetch = [&](double2 (&xa)[L::PER], double2 (&xb)[L::PER]) {
    const int row0 = (ftile % nt) * kGrpTile, col0 = (ftile / nt) * kGrpTile, k0 = fp * kGrpK;
    const double2* Ao = OPA == OP_N ? A + row0 + (size_t)k0 * n : A + k0 + (size_t)row0 * n;
    const double2* Bo = OPB == OP_N ? B + k0 + (size_t)col0 * n : B + col0 + (size_t)k0 * n;
#pragma unroll
    for (int q = 0; q < L::PER; ++q) {
      // op(A)(row0 + i, k0 + k): N reads down a column (i fast), C / T along k; B likewise
      xa[q] = ldgb(Ao, 16u * (uint32_t)(f + (w8 + 8 * q) * n));
      if (OPA == OP_C) xa[q] = cconj(xa[q]);
      xb[q] = ldgb(Bo, 16u * (uint32_t)(f + (w8 + 8 * q) * n));
      if (OPB == OP_C) xb[q] = cconj(xb[q]);
    }
    if (++fp == np) {
      fp = 0;
      ftile += size;
    }
  };
  auto store = [&](ldsd* st, const double2 (&xa)[L::PER], const double2 (&xb)[L::PER], int part) {
#pragma unroll
    for (int q = 0; q < L::PER; ++q) {
      if (part >= 0 && q != part) continue;
      const int s = w8 + 8 * q;  // k-contiguous panels are [i][k], the others [k][i]
      st[s * LA + f] = xa[q].x;
      st[L::PLANE + s * LA + f] = xa[q].y;
      st[2 * L::PLANE + s * LB + f] = xb[q].x;
      st[3 * L::PLANE + s * LB + f] = xb[q].y;
    }
  };
  static_assert(L::PER == 4, "one panel element per MFMA group");
  if (steps > 0) {
    fetch(ra[0], rb[0]);
    if (steps > 1) fetch(ra[1], rb[1]);
    store(lds, ra[0], rb[0], -1);
  }
  __syncthreads();
  int tile = rank, p = 0;
  d4 cr[1][1], ci[1][1];
  double2 d1[4], d2[4], d3[4];  // the D terms of the lane's 4 elements, requested at the tile's first panel
  auto element = [&](int r, int& i, int& j) {
    i = (tile % nt) * kGrpTile + arow + (CRM ? 4 * r + kq : m);
    j = (tile / nt) * kGrpTile + bcol + (CRM ? m : 4 * r + kq);
  };
  auto step = [&](auto par, int s) {
    constexpr int PAR = decltype(par)::value;
    ldsd* cur = lds + PAR * L::STAGE;
    ldsd* nxt = lds + (PAR ^ 1) * L::STAGE;
    if (s + 2 < steps) fetch(ra[PAR], rb[PAR]);
    if (p == 0) {
      cr[0][0] = d4{0, 0, 0, 0};
      ci[0][0] = d4{0, 0, 0, 0};
      auto terms = [&](const double2* D, double2 (&d)[4], bool transposed) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          int i, j;
          element(r, i, j);
          d[r] = ldgb(D, 16u * (uint32_t)(transposed ? j + i * n : i + j * n));
        }
      };
      if (ep.D1) terms(ep.D1, d1, false);
      if (ep.D2) terms(ep.D2, d2, false);
      if (ep.D3) terms(ep.D3, d3, true);
    }
    mma_steps<1, 1, CRM, kGrpK / 4, AKC, BKC>(cr, ci, cur, cur + L::PLANE, LA, arow, cur + 2 * L::PLANE,
                                              cur + 3 * L::PLANE, LB, bcol,
                                              [&](int g) { store(nxt, ra[PAR ^ 1], rb[PAR ^ 1], g); });
    __syncthreads();
    if (++p < np) return;
    p = 0;
    double asum = 0.0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      int i, j;
      element(r, i, j);
      double2 v = make_double2(ep.sacc * cr[0][0][r], ep.sacc * ci[0][0][r]);
      const double2 vd = cadd(v, ep.diag);
      v.x = (i == j) ? vd.x : v.x;
      v.y = (i == j) ? vd.y : v.y;
      if (ep.D1) v = cadd(v, cmul(ep.s1, d1[r]));
      if (ep.D2) v = cadd(v, cmul(ep.s2, d2[r]));
      if (ep.D3) v = cadd(v, cmul(ep.s3, cconj(d3[r])));
      if (ep.abs_sum) asum += group_abs(v);
      const uint32_t u = (uint32_t)(CRM ? j + i * n : i + j * n);
      if (ep.real_out)
        stgb_re((double*)Cout, 8u * u, v.x);
      else
        stgb((double2*)Cout, 16u * u, v);
    }
    if (ep.abs_sum) {
      // the stage just multiplied is free until the next step's stores
      const double t = block_sum(asum, cur);
      if (tid == 0) agent_store(&ctl->part[parity][tile], t);
    }
    tile += size;
  };
#pragma unroll
  for (int r = 0; r < 4; ++r) d1[r] = d2[r] = d3[r] = make_double2(0, 0);
  for (int s = 0; s < steps; s += 2) {
    step(Index<0>(), s);
    if (s + 1 < steps) step(Index<1>(), s + 1);
  }
  group_barrier();
  return ep.abs_sum ? tile_sum(ctl->part[parity], ntiles) : 0.0;
}

template <int T, int OPA, int OPB, int CRM>
__device__ __forceinline__ double wg_gemm_k(GroupN n, const double2* A, const double2* B, void* C, Epi ep, ldsd* lds) {
  static_assert(T == kGrp, "group program");
  if (large_tiles((int)n, group_size(n))) return grp_gemm_large<OPA, OPB, CRM>(n, A, B, C, ep, lds);
  return grp_gemm<OPA, OPB, CRM>(n, A, B, C, ep, lds);
}

template <int T>
__device__ __forceinline__ double wg_gemm(GroupN n, int opA, const double2* A, int opB, const double2* B, void* C,
                                          int c_rowmajor, Epi ep, ldsd* lds) {
  if (c_rowmajor) {
    if (opA == OP_N) {
      if (opB == OP_N) return wg_gemm_k<T, OP_N, OP_N, 1>(n, A, B, C, ep, lds);
      return wg_gemm_k<T, OP_N, OP_C, 1>(n, A, B, C, ep, lds);
    }
    if (opB == OP_N) return wg_gemm_k<T, OP_C, OP_N, 1>(n, A, B, C, ep, lds);
    return wg_gemm_k<T, OP_C, OP_C, 1>(n, A, B, C, ep, lds);
  }
  if (opA == OP_N) {
    if (opB == OP_N) return wg_gemm_k<T, OP_N, OP_N, 0>(n, A, B, C, ep, lds);
    return wg_gemm_k<T, OP_N, OP_C, 0>(n, A, B, C, ep, lds);
  }
  if (opB == OP_N) return wg_gemm_k<T, OP_C, OP_N, 0>(n, A, B, C, ep, lds);
  return wg_gemm_k<T, OP_C, OP_C, 0>(n, A, B, C, ep, lds);
}

// ----------------------------------------------------- elementwise, reductions
__device__ __noinline__ void wg_ew(GroupN n_, double2* out, int out_rowmajor, double2 diag, const double2* D1, double2 s1,
                                   const double2* D2, double2 s2, const double2* D3, double2 s3) {
  ew_elements(uni((int)n_), out, uni(out_rowmajor), diag, D1, s1, D2, s2, D3, s3, group_rank(n_), group_size(n_));
  group_barrier();
}

__device__ __forceinline__ void wg_antiherm(GroupN n, const double2* X, double2* out, ldsd* lds) {
  antiherm_pairs(uni((int)n), X, out, lds, group_rank(n), group_size(n));
  group_barrier();
}

__device__ __noinline__ void wg_imag_part(GroupN n_, const double2* X, double2* Y, double2* Z) {
  const int n = uni((int)n_), nn = n * n, step = 256 * group_size(n_);
  for (int idx = group_rank(n_) * 256 + threadIdx.x; idx < nn; idx += step) {
    const double2 v = gc(X)[idx];
    gw(Y)[idx] = make_double2(0.0, v.y);
    if (Z) gw(Z)[idx] = v;
  }
  group_barrier();
}

// Every rank reads the whole blocks; the barrier keeps a faster rank from overwriting them.
__device__ __forceinline__ double wg_retrace_prod(GroupN n, const double2* X, const double2* Y, ldsd* red) {
  const double s = wg_retrace_prod((int)n, X, Y, red);
  group_barrier();
  return s;
}

// ------------------------------------------------------------------ inverse
// Every rank sweeps the panels (the column steps are serial) and updates its own strips; at 64
// orbitals every rank sweeps the whole block in registers and rank 0 stores it.
template <int NMAX>
struct InvLds<kGrp, NMAX> {
  static constexpr int DOUBLES = InvStripLds<NMAX>::DOUBLES;
};

template <int T, int NMAX>
__device__ __forceinline__ int wg_inverse(GroupN n, double2* W, double2* out, ldsd* lds) {
  static_assert(T == kGrp && (NMAX == 128 || NMAX == 256), "group program");
  if (NMAX == 128 && (int)n == 64) {
    const int info = wg_inverse_reg<2, 64>(W, out, lds, group_rank(n) == 0);
    group_barrier();
    return info;
  }
  return wg_inverse_strip<NMAX>(n, W, out, lds);
}

// ----------------------------------------------------------------- contacts
// The decimations of the two contacts do not depend on each other and are half of a solve's
// inverses, which do not get faster with the ranks: each half of the group runs one.
// Between the split and the merge a workgroup is a rank of its half, which has a control
// area of its own.
template <int NMAX>
struct Leads<kGrp, NMAX> : LeadsBase {
  static __device__ __noinline__ bool run(GroupN n, double E, double eta, double tol, int nmax, Lead& L, Lead& R,
                                          ldsd* lds, ldsd* red) {
    const int size = group_size(n), rank = group_rank(n), first = (size + 1) / 2;
    if (size == 1) {
      for (int h = 0; h < 2; ++h) one(n, E, eta, tol, nmax, h ? R : L, lds, red);
      return false;
    }
    const int h = rank >= first ? 1 : 0;
    GroupCtx* c = group_ctx();
    GroupCtl* ctl = uni(c->ctl);
    const unsigned epoch = uni((int)c->epoch);
    __syncthreads();
    if (threadIdx.x == 0) {
      c->ctl = reinterpret_cast<GroupCtl*>(reinterpret_cast<char*>(ctl) + kCtlBytes * (1 + h));
      c->rank = h ? rank - first : rank;
      c->size = h ? size - first : first;
      c->epoch = c->half_epoch;
    }
    __syncthreads();
    Lead& m = h ? R : L;
    one(n, E, eta, tol, nmax, m, lds, red);
    __syncthreads();
    if (threadIdx.x == 0) {
      if (c->rank == 0) {
        agent_store(&ctl->lead[h][0], m.it);
        agent_store(&ctl->lead[h][1], m.hit);
        agent_store(&ctl->lead[h][2], m.fails);
      }
      c->half_epoch = c->epoch;
      c->ctl = ctl;
      c->rank = rank;
      c->size = size;
      c->epoch = epoch;
    }
    group_barrier();
    for (int k = 0; k < 2; ++k) {
      Lead& x = k ? R : L;
      x.it = uni(agent_load(&ctl->lead[k][0]));
      x.hit = uni(agent_load(&ctl->lead[k][1]));
      x.fails = uni(agent_load(&ctl->lead[k][2]));
    }
    return false;
  }

  static __device__ __noinline__ void one(GroupN n, double E, double eta, double tol, int nmax, Lead& m, ldsd* lds,
                                          ldsd* red) {
    m.hit = m.fails = 0;
    m.it = wg_sancho<kGrp, NMAX>(n, E, eta, tol, nmax, m.H00, m.C, m.left, m.G, m.tb, lds, red, m.hit, m.fails);
  }
};

// At 32 orbitals a block operation is too short to share, but the right contact's
// decimation is not needed before the forward sweep is over: in a group of two, rank 1 runs
// it and leaves, rank 0 runs the rest of the program.
template <int T, int NMAX>
struct PairLeads {
  static constexpr int kRightTemp = kTmpBlocks;
  static __device__ __forceinline__ bool left() { return uni(group_ctx()->rank) == 0; }
  static __device__ __forceinline__ bool right() { return uni(group_ctx()->rank) == 1 || uni(group_ctx()->size) == 1; }
  static __device__ bool run(typename Dim<T>::type n, double E, double eta, double tol, int nmax, Lead& L, Lead& R,
                             ldsd* lds, ldsd* red) {
    const int rank = uni(group_ctx()->rank), size = uni(group_ctx()->size);
    for (int h = rank; h < 2; h += size) {
      Lead& m = h ? R : L;
      m.hit = m.fails = 0;
      m.it = wg_sancho<T, NMAX>(n, E, eta, tol, nmax, m.H00, m.C, m.left, m.G, m.tb, lds, red, m.hit, m.fails);
    }
    if (rank == 0) return false;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    __syncthreads();
    if (threadIdx.x == 0) {
      GroupCtl* ctl = group_ctx()->ctl;
      agent_store(&ctl->lead[1][0], R.it);
      agent_store(&ctl->lead[1][1], R.hit);
      agent_store(&ctl->lead[1][2], R.fails);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
      agent_store(&ctl->barrier, 1u);
    }
    return true;
  }
  static __device__ __forceinline__ void finish(Lead& R) {
    if (uni(group_ctx()->size) == 1) return;
    GroupCtl* ctl = uni(group_ctx()->ctl);
    if (threadIdx.x == 0) {
      while (agent_load(&ctl->barrier) == 0u) __builtin_amdgcn_s_sleep(1);
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    __syncthreads();
    R.it = uni(agent_load(&ctl->lead[1][0]));
    R.hit = uni(agent_load(&ctl->lead[1][1]));
    R.fails = uni(agent_load(&ctl->lead[1][2]));
  }
};
template <>
struct Leads<kPair32, 32> : PairLeads<kPair32, 32> {};

// ------------------------------------------------------------------ kernels
template <int T, int NMAX>
__global__ __launch_bounds__(256, 1) void rgf_sweep_pair(SweepArgs a, GroupArgs g) {
  __shared__ __attribute__((aligned(16))) double lds[SweepLds<T, NMAX>::DOUBLES];
  int grp;
  if (!group_join(g, grp)) return;
  solve_energy<T, NMAX>(a, g.e0 + grp, a.ws + (size_t)grp * (size_t)a.ws_slot, (ldsd*)lds, (ldsd*)lds);
}

template <int NMAX>
__global__ __launch_bounds__(256, 1) void rgf_sweep_grp(SweepArgs a, GroupArgs g) {
  __shared__ __attribute__((aligned(16))) double lds[SweepLds<kGrp, NMAX>::DOUBLES];
  int grp;
  if (!group_join(g, grp)) return;
  double2* ws = a.ws + (size_t)grp * (size_t)a.ws_slot;
  for (int e = g.e0 + grp; e < a.nE; e += g.ngroups) {
    solve_energy<kGrp, NMAX>(a, e, ws, (ldsd*)lds, (ldsd*)lds);
    group_barrier();
  }
}

template <int NMAX>
__global__ __launch_bounds__(256, 1) void rgf_sweep_od_grp(SweepArgs a, GroupArgs g) {
  __shared__ __attribute__((aligned(16))) double lds[SweepLds<kGrp, NMAX>::DOUBLES];
  int grp;
  if (!group_join(g, grp)) return;
  double2* ws = a.ws + (size_t)grp * (size_t)a.ws_slot;
  for (int e = g.e0 + grp; e < a.nE; e += g.ngroups) {
    solve_energy_od<kGrp, NMAX>(a, e, ws, (ldsd*)lds, (ldsd*)lds);
    group_barrier();
  }
}

template <int NMAX>
__global__ __launch_bounds__(256, 1) void rgf_adjoint_grp(AdjArgs a, GroupArgs g) {
  __shared__ __attribute__((aligned(16))) double lds[SweepLds<kGrp, NMAX>::DOUBLES];
  int grp;
  if (!group_join(g, grp)) return;
  double2* ws = a.ws + (size_t)grp * (size_t)a.ws_slot;
  double2* dH = a.dH + (size_t)grp * a.nx * (size_t)a.n * a.n;
  for (int e = g.e0 + grp; e < a.nE; e += g.ngroups) {
    adjoint_energy<kGrp, NMAX>(a, e, ws, dH, (ldsd*)lds, (ldsd*)lds);
    group_barrier();
  }
}

template <int NMAX>
__global__ __launch_bounds__(256, 1) void rgf_wsweep_grp(WArgs a, GroupArgs g) {
  __shared__ __attribute__((aligned(16))) double lds[SweepLds<kGrp, NMAX>::DOUBLES];
  int grp;
  if (!group_join(g, grp)) return;
  double2* ws = a.ws + (size_t)grp * (size_t)a.ws_slot;
  for (int e = g.e0 + grp; e < a.nE; e += g.ngroups) {
    w_energy<kGrp, NMAX>(a, e, ws, (ldsd*)lds);
    group_barrier();
  }
}

// Several devices on groups of unequal size, each running its list of (device, energy)
// items.
struct MultiGroupLds {
  static constexpr int A = SweepLds<kGrp, 256>::DOUBLES, B = SweepLds<kGrp, 128>::DOUBLES;
  static constexpr int C = SweepLds<2, 64>::DOUBLES;
  static constexpr int AB = A > B ? A : B, DOUBLES = AB > C ? AB : C;
};

__global__ __launch_bounds__(256, 1) void rgf_sweep_multi_grp(MultiGroupArgs m) {
  __shared__ __attribute__((aligned(16))) double lds[MultiGroupLds::DOUBLES];
  const int grp = uni(m.block_group[blockIdx.x]);
  if (grp < 0 || !group_join(m.ctl + (size_t)grp * kGroupCtlBytes, uni(m.sizes[grp]))) return;
  double2* ws = m.ws + (size_t)grp * (size_t)m.ws_slot;
  ldsd* L = (ldsd*)lds;
  for (int i = uni(m.first[grp]); i < uni(m.first[grp + 1]); ++i) {
    const int job = uni(m.items[i].x), e = uni(m.items[i].y);
    const SweepArgs& a = m.jobs[job];
    if (a.n == 32)  // in groups of one workgroup only
      solve_energy<kReg32, 32>(a, e, ws, L, L);
    else if (a.n == 64)
      solve_energy<2, 64>(a, e, ws, L, L);
    else if (a.n <= 128)
      solve_energy<kGrp, 128>(a, e, ws, L, L);
    else
      solve_energy<kGrp, 256>(a, e, ws, L, L);
    group_barrier();
  }
}

}  // namespace rgf
