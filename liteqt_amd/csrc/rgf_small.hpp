// rgf_small.hpp -- block operations for 32 orbitals, with blocks in LDS.
//
// At 32 orbitals a GEMM is 0.87 us of MFMAs on a CU while a block is 16 KB, so the
// programs were bounded by their temporaries' trips through memory (1.2 MB per slab and
// energy at 4.4 TB/s with 1000 energies in flight) and, for one energy, by the latency of
// each trip.  Here the hottest temporaries live in LDS (Temp<kReg32>), two workgroups per
// CU.  A block operation takes each operand where it is: its pointer is generic, and
// one uniform test per operand chooses LDS or global accesses.  LDS blocks have a column
// stride of 33: fragment reads along either index, transposed and diagonal accesses then
// spread over all banks.
// The programs are compiled unchanged with SmallN as the type of their block dimension.
#pragma once
#include "rgf_sweep.hpp"

namespace rgf {

constexpr int kReg32 = 9;      // variant code: two workgroups per CU
constexpr int kPair32 = 65;    // the same program with a second workgroup for the right contact
constexpr int kSmallLd = 33;   // column stride of a block in LDS (elements)
constexpr int kSmallBlk = 2 * 32 * kSmallLd;  // doubles of an LDS block
constexpr int kSmallScratch = 1024;           // doubles below the blocks: exchanges and sums

struct SmallN {
  int v;
  __device__ __forceinline__ SmallN(int n) : v(n) {}
  __device__ __forceinline__ operator int() const { return 32; }
};
template <>
struct Dim<kReg32> {
  typedef SmallN type;
};
template <>
struct Dim<kPair32> {
  typedef SmallN type;
};
__device__ __forceinline__ bool group_leader(SmallN) { return true; }

template <>
struct GemmLds<kReg32> {
  static constexpr int DOUBLES = 64;
};
template <>
struct InvLds<kReg32, 32> {
  static constexpr int DOUBLES = GjLds<1, 4, 2>::DOUBLES + 32 + 8;  // exchange, then piv and its inverse
};
template <>
struct GemmLds<kPair32> : GemmLds<kReg32> {};
template <>
struct InvLds<kPair32, 32> : InvLds<kReg32, 32> {};
static_assert(InvLds<kReg32, 32>::DOUBLES <= kSmallScratch, "scratch below the LDS blocks");
template <>
struct SweepLds<kReg32, 32> {
  static constexpr int DOUBLES = kSmallScratch + 4 * kSmallBlk;
};

template <>
struct SweepLds<kPair32, 32> : SweepLds<kReg32, 32> {};

// The four LDS blocks by the temporaries' reads and writes per slab: T0 and T1 (6, 5), T2
// of the forward with X of the backward sweep (3, 4), W with P7 (2, 3); the latter pairs
// are never live together (the backward sweep's T2 is spent before X is formed, and a
// segment recompute runs while X and P7 are dead).  The decimation, which runs while all
// of them are dead, has its A, B, B2 and W there.
template <>
struct Temp<kReg32> {
  static __device__ __forceinline__ double2* at(double2* tb, size_t nn, int k, ldsd* lds) {
    const int slot = k == 7 || k == kTmpSancho + 6   ? 0
                     : k == 8 || k == kTmpSancho + 7 ? 1
                     : k == 9 || k == 11 || k == kTmpSancho + 9 ? 2
                     : k == 5 || k == 12 || k == kTmpSancho + 10 ? 3
                                                                 : -1;
    if (slot < 0) return tb + (size_t)k * nn;
    return (double2*)(lds + kSmallScratch + slot * kSmallBlk);
  }
};
template <>
struct Temp<kPair32> : Temp<kReg32> {};

// A block where it is: element (i, j) at i + j ld.
struct SmallBlk {
  double2* p;
  bool sh;
  int ld;
  __device__ __forceinline__ explicit SmallBlk(const void* q) {
    p = (double2*)uni((const double2*)q);
#if defined(__HIP_DEVICE_COMPILE__)
    sh = __builtin_amdgcn_is_shared((const __attribute__((address_space(0))) void*)p);
#else
    sh = false;
#endif
    ld = sh ? kSmallLd : 32;
  }
  // f(load, store): a loader of element indexes and, for stores, a writer
  template <typename F>
  __device__ __forceinline__ void with(const F& f) const {
    if (sh) {
      ldsv* q = (ldsv*)p;
      f([&](int o) { const dvec2 v = q[o]; return make_double2(v.x, v.y); },
        [&](int o, double2 v) { dvec2 w; w.x = v.x; w.y = v.y; q[o] = w; });
    } else {
      f([&](int o) { return ldgb(p, 16u * (uint32_t)o); }, [&](int o, double2 v) { stgb(p, 16u * (uint32_t)o, v); });
    }
  }
};

// GEMM: one 16 x 16 tile per wave, its MFMA fragments loaded straight from the operands,
// all 16 loads of a lane in flight at once (panels through LDS paid the latency three
// times, with a barrier each).  The products are summed in the order of mma_steps.
template <int OPA, int OPB, int CRM>
__device__ __noinline__ double gemm_reg32(const double2* A_, const double2* B_, void* C_, Epi ep_, ldsd* lds) {
  constexpr int NK = 8;
  const SmallBlk A(A_), B(B_);
  Epi ep;
  ep.diag = uni(ep_.diag); ep.sacc = uni(ep_.sacc);
  ep.D1 = uni(ep_.D1); ep.s1 = uni(ep_.s1);
  ep.D2 = uni(ep_.D2); ep.s2 = uni(ep_.s2);
  ep.D3 = uni(ep_.D3); ep.s3 = uni(ep_.s3);
  ep.real_out = uni(ep_.real_out); ep.abs_sum = uni(ep_.abs_sum);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m = lane & 15, kq = lane >> 4;
  const int arow = (wave & 1) * 16, bcol = (wave >> 1) * 16;
  // op(A)(arow + m, 4 ks + kq), op(B)(4 ks + kq, bcol + m)
  double2 a[NK], b[NK];
  A.with([&](auto load, auto) {
    const int o = OPA == OP_N ? arow + m + kq * A.ld : kq + (arow + m) * A.ld, d = OPA == OP_N ? 4 * A.ld : 4;
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) a[ks] = load(o + ks * d);
  });
  B.with([&](auto load, auto) {
    const int o = OPB == OP_N ? kq + (bcol + m) * B.ld : bcol + m + kq * B.ld, d = OPB == OP_N ? 4 : 4 * B.ld;
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) b[ks] = load(o + ks * d);
  });
  // element r of the lane: (i0 + 4 r, j0) when CRM, else (i0, j0 + 4 r)
  const int i0 = arow + (CRM ? kq : m), j0 = bcol + (CRM ? m : kq);
  auto terms = [&](const double2* D, bool transposed, double2 (&d)[4]) {
    const SmallBlk X(D);
    X.with([&](auto load, auto) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = CRM ? i0 + 4 * r : i0, j = CRM ? j0 : j0 + 4 * r;
        d[r] = load(transposed ? j + i * X.ld : i + j * X.ld);
      }
    });
  };
  double2 d1[4], d2[4], d3[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) d1[r] = d2[r] = d3[r] = make_double2(0, 0);
  if (ep.D1) terms(ep.D1, false, d1);
  if (ep.D2) terms(ep.D2, false, d2);
  if (ep.D3) terms(ep.D3, true, d3);
  d4 cr = d4{0, 0, 0, 0}, ci = d4{0, 0, 0, 0};
#pragma unroll
  for (int ks = 0; ks < NK; ++ks) {
    const double ar = a[ks].x, ai = OPA == OP_C ? -a[ks].y : a[ks].y;
    const double br = b[ks].x, bi = OPB == OP_C ? -b[ks].y : b[ks].y;
    if (CRM) {
      cr = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, br, cr, 0, 0, 0);
      ci = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, bi, ci, 0, 0, 0);
      cr = __builtin_amdgcn_mfma_f64_16x16x4f64(-ai, bi, cr, 0, 0, 0);
      ci = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, br, ci, 0, 0, 0);
    } else {
      cr = __builtin_amdgcn_mfma_f64_16x16x4f64(br, ar, cr, 0, 0, 0);
      ci = __builtin_amdgcn_mfma_f64_16x16x4f64(bi, ar, ci, 0, 0, 0);
      cr = __builtin_amdgcn_mfma_f64_16x16x4f64(bi, -ai, cr, 0, 0, 0);
      ci = __builtin_amdgcn_mfma_f64_16x16x4f64(br, ai, ci, 0, 0, 0);
    }
  }
  double asum = 0.0;
  double2 v[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = CRM ? i0 + 4 * r : i0, j = CRM ? j0 : j0 + 4 * r;
    v[r] = make_double2(ep.sacc * cr[r], ep.sacc * ci[r]);
    const double2 vd = cadd(v[r], ep.diag);
    v[r].x = (i == j) ? vd.x : v[r].x;
    v[r].y = (i == j) ? vd.y : v[r].y;
    if (ep.D1) v[r] = cadd(v[r], cmul(ep.s1, d1[r]));
    if (ep.D2) v[r] = cadd(v[r], cmul(ep.s2, d2[r]));
    if (ep.D3) v[r] = cadd(v[r], cmul(ep.s3, cconj(d3[r])));
    if (ep.abs_sum) asum += sqrt(v[r].y * v[r].y + v[r].x * v[r].x);
  }
  if (ep.real_out) {  // a caller's array
    double* C = uni((double*)C_);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = CRM ? i0 + 4 * r : i0, j = CRM ? j0 : j0 + 4 * r;
      stgb_re(C, 8u * (uint32_t)(CRM ? j + i * 32 : i + j * 32), v[r].x);
    }
  } else {
    const SmallBlk C(C_);
    C.with([&](auto, auto store) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = CRM ? i0 + 4 * r : i0, j = CRM ? j0 : j0 + 4 * r;
        store(CRM ? j + i * C.ld : i + j * C.ld, v[r]);
      }
    });
  }
  double s = 0.0;
  if (ep.abs_sum) s = block_sum(asum, lds);
  __syncthreads();
  return s;
}

template <int T, int OPA, int OPB, int CRM>
__device__ __forceinline__ double wg_gemm_k(SmallN, const double2* A, const double2* B, void* C, Epi ep, ldsd* lds) {
  static_assert(T == kReg32 || T == kPair32, "32-orbital program");
  return gemm_reg32<OPA, OPB, CRM>(A, B, C, ep, lds);
}

template <int T>
__device__ __forceinline__ double wg_gemm(SmallN n, int opA, const double2* A, int opB, const double2* B, void* C,
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

// Elementwise operations: thread t has rows t % 32 of columns t / 32 + 8 u, u < 4.
__device__ __noinline__ void small_ew(double2* out_, int out_rowmajor_, double2 diag_, const double2* D1_, double2 s1_,
                                      const double2* D2_, double2 s2_, const double2* D3_, double2 s3_) {
  const SmallBlk out(out_);
  const bool rm = uni(out_rowmajor_) != 0;
  const double2 diag = uni(diag_), s1 = uni(s1_), s2 = uni(s2_), s3 = uni(s3_);
  const int f = threadIdx.x & 31, w = threadIdx.x >> 5;  // f runs along the output's contiguous index
  double2 v[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) v[u] = make_double2(f == w + 8 * u ? diag.x : 0.0, f == w + 8 * u ? diag.y : 0.0);
  auto term = [&](const double2* D_, double2 s, bool conj_t) {
    const double2* D = uni(D_);
    if (!D) return;
    const SmallBlk X(D);
    X.with([&](auto load, auto) {
      double2 d[4];
      const bool swap = rm != conj_t;  // the element's row is the slow index
#pragma unroll
      for (int u = 0; u < 4; ++u) d[u] = load(swap ? w + 8 * u + f * X.ld : f + (w + 8 * u) * X.ld);
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = cadd(v[u], cmul(s, conj_t ? cconj(d[u]) : d[u]));
    });
  };
  term(D1_, s1, false);
  term(D2_, s2, false);
  term(D3_, s3, true);
  out.with([&](auto, auto store) {
#pragma unroll
    for (int u = 0; u < 4; ++u) store(f + (w + 8 * u) * out.ld, v[u]);
  });
  __syncthreads();
}
__device__ __forceinline__ void wg_ew(SmallN, double2* out, int out_rowmajor, double2 diag, const double2* D1, double2 s1,
                                      const double2* D2, double2 s2, const double2* D3, double2 s3) {
  small_ew(out, out_rowmajor, diag, D1, s1, D2, s2, D3, s3);
}

__device__ __forceinline__ void wg_antiherm(SmallN, const double2* X, double2* out, ldsd*) {
  small_ew(out, 0, make_double2(0, 0), X, make_double2(0.5, 0), nullptr, make_double2(0, 0), X, make_double2(-0.5, 0));
}

__device__ __forceinline__ void wg_imag_part(SmallN, const double2* X, double2* Y, double2* Z) {
  wg_imag_part(32, X, Y, Z);  // the screened interaction's blocks are all in memory
}

__device__ __noinline__ double small_retrace(const double2* X_, const double2* Y_, ldsd* red) {
  const SmallBlk X(X_), Y(Y_);
  const int f = threadIdx.x & 31, w = threadIdx.x >> 5;
  double2 x[4], y[4];
  X.with([&](auto load, auto) {
#pragma unroll
    for (int u = 0; u < 4; ++u) x[u] = load(f + (w + 8 * u) * X.ld);
  });
  Y.with([&](auto load, auto) {
#pragma unroll
    for (int u = 0; u < 4; ++u) y[u] = load(w + 8 * u + f * Y.ld);
  });
  double s = 0.0;
#pragma unroll
  for (int u = 0; u < 4; ++u) s += x[u].x * y[u].x - x[u].y * y[u].y;
  return block_sum(s, red);
}
__device__ __forceinline__ double wg_retrace_prod(SmallN, const double2* X, const double2* Y, ldsd* red) {
  return small_retrace(X, Y, red);
}

__device__ __forceinline__ double wg_imtrace(SmallN, const double2* X_, ldsd* red) {
  const SmallBlk X(X_);
  double s = 0.0;
  if (threadIdx.x < 32) X.with([&](auto load, auto) { s = load((int)threadIdx.x * (X.ld + 1)).y; });
  return block_sum(s, red);
}

// The register inverse, each element stored straight to its place: out(pinv[i], piv[c])
// = W[i][c] (a store of 32 lanes fills one column, in the order of the pivots).
__device__ __noinline__ int small_inverse(const double2* W_, double2* out_, ldsd* lds) {
  const SmallBlk W(W_), out(out_);
  ldsi* piv = (ldsi*)(lds + GjLds<1, 4, 2>::DOUBLES);
  ldsi* pinv = piv + 32;
  const int tid = threadIdx.x, i = tid & 31, cb = tid >> 5;
  double2 a[1][4];
  W.with([&](auto load, auto) {
#pragma unroll
    for (int c = 0; c < 4; ++c) a[0][c] = load(i * W.ld + cb * 4 + c);
  });
  unsigned used = 0;
  const int info = gj_sweep<1, 4, 2>(a, 32, used, piv, lds);
  if (tid < 32) pinv[piv[tid]] = tid;
  __syncthreads();
  // (a singular block has no permutation: zeros to the elements' own places)
  const int r = info ? i : pinv[i];
  out.with([&](auto, auto store) {
#pragma unroll
    for (int c = 0; c < 4; ++c)
      store(r + (info ? cb * 4 + c : piv[cb * 4 + c]) * out.ld, info ? make_double2(0, 0) : a[0][c]);
  });
  __syncthreads();
  return info;
}

template <int T, int NMAX>
__device__ __forceinline__ int wg_inverse(SmallN, double2* W, double2* out, ldsd* lds) {
  static_assert((T == kReg32 || T == kPair32) && NMAX == 32, "32-orbital program");
  return small_inverse(W, out, lds);
}

}  // namespace rgf
