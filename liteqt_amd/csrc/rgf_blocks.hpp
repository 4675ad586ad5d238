// rgf_blocks.hpp -- workgroup-level complex-FP64 building blocks for gfx950.
//
// One workgroup (256 threads = 4 wave64) owns one energy and runs every matrix
// operation of the RGF on it: complex GEMMs on FP64 MFMA
// (v_mfma_f64_16x16x4_f64) with LDS-staged K panels, a blocked Gauss-Jordan
// inverse with partial (row) pivoting, elementwise combinations and
// reductions.  Matrices live in HBM/L2 (workspace or caller arrays); all
// operations end with a workgroup barrier so the next one sees their results.
//
// MFMA f64 16x16x4 lane layout (measured on gfx950): lane l supplies
// X[l%16][l/16] of the 16x4 operand and Y[l/16][l%16] of the 4x16 operand and
// holds D[4r + l/16][l%16] in accumulator element r.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace rgf {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int PAD = 16;   // LDS row padding (doubles): row stride = 16 mod 32 doubles
constexpr int KP = 16;    // K panel depth (complex)
// Row stride (doubles) of an LDS panel stored k-contiguous ([row][k]): 2 mod 32, so
// the fragment reads of 16 rows x 2 k-steps per half-wave hit distinct 8-byte bank pairs.
constexpr int LDK = KP + 2;

enum { OP_N = 0, OP_C = 1, OP_T = 2 };  // op(X) = X, X^H, X^T

// Explicit address spaces: global (1) and LDS (3).  Pointers that reach a
// non-inlined function as generic pointers would be accessed with FLAT
// instructions, which count against both the vector-memory and the LDS wait
// counters and so serialise the global prefetch with the LDS fragment reads.
// The host pass only parses device code, so it sees the unqualified types.
#if defined(__HIP_DEVICE_COMPILE__)
typedef __attribute__((address_space(3))) double ldsd;
typedef __attribute__((address_space(3))) int ldsi;
typedef __attribute__((address_space(1))) double2 gd2;
typedef __attribute__((address_space(1))) const double2 gcd2;
typedef __attribute__((address_space(1))) double gd;
#else
typedef double ldsd;
typedef int ldsi;
typedef double2 gd2;
typedef const double2 gcd2;
typedef double gd;
#endif

__device__ __forceinline__ gcd2* gc(const double2* p) { return (gcd2*)p; }
__device__ __forceinline__ gd2* gw(double2* p) { return (gd2*)p; }

// 16-byte complex load through a native vector type (one global_load_dwordx4).
typedef double dvec2 __attribute__((ext_vector_type(2)));
#if defined(__HIP_DEVICE_COMPILE__)
typedef __attribute__((address_space(1))) const dvec2 gcv2;
#else
typedef const dvec2 gcv2;
#endif
__device__ __forceinline__ double2 ldg(const double2* p, size_t i) {
  const dvec2 v = ((gcv2*)p)[i];
  return make_double2(v.x, v.y);
}

// Loads and stores at a wave-uniform base plus a 32-bit byte offset: the base
// stays in scalar registers and the address is one VGPR (global_* saddr form).
#if defined(__HIP_DEVICE_COMPILE__)
typedef __attribute__((address_space(1))) const char gcb;
typedef __attribute__((address_space(1))) char gwb;
typedef __attribute__((address_space(1))) dvec2 gv2;
#else
typedef const char gcb;
typedef char gwb;
typedef dvec2 gv2;
#endif
__device__ __forceinline__ double2 ldgb(const double2* base, uint32_t boff) {
  const dvec2 v = *(gcv2*)((gcb*)base + boff);
  return make_double2(v.x, v.y);
}
__device__ __forceinline__ void stgb(double2* base, uint32_t boff, double2 v) {
  dvec2 w;
  w.x = v.x;
  w.y = v.y;
  *(gv2*)((gwb*)base + boff) = w;
}
__device__ __forceinline__ void stgb_re(double* base, uint32_t boff, double v) { *(gd*)((gwb*)base + boff) = v; }

// A block dimension of type int is a lone workgroup's: it has every tile, and its
// operations end with the workgroup barrier (rgf_group.hpp has the other kind).
__device__ __forceinline__ int group_rank(int) { return 0; }
__device__ __forceinline__ int group_size(int) { return 1; }
__device__ __forceinline__ void group_sync(int) { __syncthreads(); }

// Uniform values arrive in VGPRs through the calling convention of a
// non-inlined function; moving them to SGPRs frees those VGPRs.
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ double uni(double v) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)b);
  const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(b >> 32));
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
template <typename P>
__device__ __forceinline__ P* uni(P* p) {
  const unsigned long long b = (unsigned long long)(uintptr_t)p;
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)b);
  const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(b >> 32));
  return (P*)(uintptr_t)(((unsigned long long)hi << 32) | lo);
}
__device__ __forceinline__ double2 uni(double2 v) { return make_double2(uni(v.x), uni(v.y)); }

__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 cconj(double2 a) { return make_double2(a.x, -a.y); }
// Smith's algorithm for 1/b.
__device__ __forceinline__ double2 crecip(double2 b) {
  if (fabs(b.x) >= fabs(b.y)) {
    double t = b.y / b.x, d = b.x + b.y * t;
    return make_double2(1.0 / d, -t / d);
  } else {
    double t = b.x / b.y, d = b.x * t + b.y;
    return make_double2(t / d, -1.0 / d);
  }
}

// 1/b for a wave-uniform b: where |b| is far from the ends of the exponent range (high
// words of the components below 2^500, the larger above 2^-500) b* / |b|^2 with the
// hardware's reciprocal refined by two Newton steps, 8 dependent operations against the
// two divisions in a row of the general form; else the general form.
__device__ __forceinline__ double2 crecip_uniform(double2 b) {
  const unsigned hx = (unsigned)(__builtin_bit_cast(unsigned long long, b.x) >> 32) & 0x7fffffffu;
  const unsigned hy = (unsigned)(__builtin_bit_cast(unsigned long long, b.y) >> 32) & 0x7fffffffu;
  const unsigned h = uni((int)(hx > hy ? hx : hy));
  constexpr unsigned lo = (1023u - 500u) << 20, hi = (1023u + 500u) << 20;
  if (h >= lo && h < hi) {
    const double d = fma(b.x, b.x, b.y * b.y);
    double r = __builtin_amdgcn_rcp(d);
    r = fma(r, fma(-d, r, 1.0), r);
    r = fma(r, fma(-d, r, 1.0), r);
    return make_double2(b.x * r, -b.y * r);
  }
  return crecip(b);
}

// out(i,j) = sacc*acc(i,j) + diag*[i==j] + s1*D1(i,j) + s2*D2(i,j) + s3*conj(D3(j,i))
// D1 may alias the output (each element is read and written by one thread);
// D3 must not.  real_out stores Re(value) into a double array.
struct Epi {
  double2 diag;
  double sacc;
  const double2* D1;
  double2 s1;
  const double2* D2;
  double2 s2;
  const double2* D3;
  double2 s3;
  int real_out;
  int abs_sum;  // accumulate sum_ij |value| (returned by the GEMM)
};

__device__ __forceinline__ Epi epi_store() {
  Epi e;
  e.diag = make_double2(0, 0); e.sacc = 1.0;
  e.D1 = nullptr; e.s1 = make_double2(1, 0);
  e.D2 = nullptr; e.s2 = make_double2(1, 0);
  e.D3 = nullptr; e.s3 = make_double2(1, 0);
  e.real_out = 0; e.abs_sum = 0;
  return e;
}

__device__ __forceinline__ double2 epi_value(const Epi& ep, int n, int i, int j, double ar, double ai) {
  double2 v = make_double2(ep.sacc * ar, ep.sacc * ai);
  if (i == j) v = cadd(v, ep.diag);
  if (ep.D1) v = cadd(v, cmul(ep.s1, gc(ep.D1)[i + (size_t)j * n]));
  if (ep.D2) v = cadd(v, cmul(ep.s2, gc(ep.D2)[i + (size_t)j * n]));
  if (ep.D3) v = cadd(v, cmul(ep.s3, cconj(gc(ep.D3)[j + (size_t)i * n])));
  return v;
}

// ---------------------------------------------------------------- reductions
// DPP lane exchange of a double within a row of 16 lanes (CTRL: a DPP pattern that
// reads only lanes of the same row).
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, 0xf, 0xf, false);
  return __builtin_bit_cast(double, ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}

__device__ __forceinline__ double lane_f64(double v, int l) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = __builtin_amdgcn_readlane((unsigned)b, l);
  const unsigned hi = __builtin_amdgcn_readlane((unsigned)(b >> 32), l);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// Maximum over the wave (uniform result): quad swaps, half-row and row mirrors,
// one 16-lane swap, then the two 32-lane halves.
__device__ __forceinline__ double wave_max(double v) {
  v = fmax(v, dpp_f64<0xB1>(v));   // quad_perm [1,0,3,2]
  v = fmax(v, dpp_f64<0x4E>(v));   // quad_perm [2,3,0,1]
  v = fmax(v, dpp_f64<0x141>(v));  // row_half_mirror
  v = fmax(v, dpp_f64<0x140>(v));  // row_mirror
  v = fmax(v, __shfl_xor(v, 16, 64));
  return fmax(lane_f64(v, 0), lane_f64(v, 32));
}

__device__ __forceinline__ double wave_sum(double v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// Sum over the workgroup; result valid in every thread.  red: >= 8 doubles of LDS.
__device__ __forceinline__ double block_sum(double v, ldsd* red) {
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) red[wave] = v;
  __syncthreads();
  double s = 0.0;
  for (int w = 0; w < (int)(blockDim.x >> 6); ++w) s += red[w];
  __syncthreads();
  return s;
}

// Argmax of v over the workgroup, ties to the smallest index.
__device__ __forceinline__ void block_argmax(double& v, int& idx, ldsd* redv, ldsi* redi) {
  for (int off = 32; off > 0; off >>= 1) {
    double ov = __shfl_xor(v, off, 64);
    int oi = __shfl_xor(idx, off, 64);
    if (ov > v || (ov == v && oi < idx)) { v = ov; idx = oi; }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) { redv[wave] = v; redi[wave] = idx; }
  __syncthreads();
  v = redv[0]; idx = redi[0];
  for (int w = 1; w < (int)(blockDim.x >> 6); ++w) {
    double ov = redv[w]; int oi = redi[w];
    if (ov > v || (ov == v && oi < idx)) { v = ov; idx = oi; }
  }
  __syncthreads();
}

// ------------------------------------------------------------ tile configs
// Per block-size variant V = T + 8 (OCC - 1): a pass computes an MR x MC macro
// tile of C with NW waves in a WR x WC grid, each wave owning TA x TB MFMA tiles
// of 16x16 complex (2*TA*TB accumulators of 4 doubles).  T = 4 (n = 128, 256)
// uses a 128 x 64 macro tile: 64 x 32 per wave keeps a wave at 128 accumulator
// registers, so nothing spills with one wave per SIMD.  Smaller T use square
// (32T)^2 tiles.  OCC is the number of workgroups per CU the variant's kernels
// are compiled for (their launch bounds): the same code at OCC = 2 is a
// separate instantiation of every block function, so the register budget of
// two workgroups per CU applies to it alone.
template <int V>
struct Cfg {
  static constexpr int T = V & 7;
  static constexpr int OCC = 1 + (V >> 3);
  static constexpr int MR = 32 * T;
  static constexpr int MC = (T == 4) ? 64 : 32 * T;
  static constexpr int NW = 4;
  static constexpr int WR = 2;
  static constexpr int WC = 2;
  static constexpr int TA = MR / (16 * WR);
  static constexpr int TB = MC / (16 * WC);
  static constexpr int NTH = 64 * NW;
  static constexpr int LDA = MR + PAD;  // LDS row stride of the op(A) panel
  static constexpr int LDB = MC + PAD;  // LDS row stride of the op(B) panel
  static constexpr int STAGE = 2 * KP * LDA + 2 * KP * LDB;  // re/im planes of both panels
  static constexpr int PERA = (MR * KP) / NTH;
  static constexpr int PERB = (MC * KP) / NTH;
  static_assert(TA * 16 * WR == MR && TB * 16 * WC == MC, "wave grid must tile the macro tile");
  static_assert((MR * KP) % NTH == 0 && (MC * KP) % NTH == 0, "panels must split evenly");
  static_assert(MR * LDK <= KP * LDA && MC * LDK <= KP * LDB, "k-contiguous panels fit the planes");
};

// ----------------------------------------------------------- MFMA micro-tile
// Accumulate NKS k-steps (4 complex k each) of a wave's TA x TB grid of 16x16
// complex tiles.  A values at Ar/Ai[k*lda + arow + m], B at Br/Bi[k*ldb + bcol + m].
// ROWMAJ=0: lane holds C[arow + ti*16 + l%16][bcol + tj*16 + 4r + l/16];
// ROWMAJ=1: lane holds C[arow + ti*16 + 4r + l/16][bcol + tj*16 + l%16].
// AKC / BKC: the panel is stored k-contiguous (A at Ar[(arow + m) * lda + k], B at
// Br[(bcol + m) * ldb + k]) instead of row-contiguous (A at Ar[k * lda + arow + m]).
struct NoMid {
  __device__ void operator()(int) const {}
};

// mid(g), g = 0..3, runs after the g-th group of MFMAs of the last k-step, pinned
// there, so work of the caller (the LDS stores of the next panel) issues while
// the MFMA pipe is still busy.
template <int TA, int TB, int ROWMAJ, int NKS, bool AKC = false, bool BKC = false, typename Mid = NoMid>
__device__ __forceinline__ void mma_steps(d4 (&cr)[TA][TB], d4 (&ci)[TA][TB],
                                          const ldsd* Ar, const ldsd* Ai, int lda, int arow,
                                          const ldsd* Br, const ldsd* Bi, int ldb, int bcol,
                                          const Mid& mid = Mid()) {
  constexpr bool kMid = !__is_same(Mid, NoMid);
  const int lane = threadIdx.x & 63;
  const int m = lane & 15, kq = lane >> 4;
  // fragments of k-step ks + 1 are read while the MFMAs of k-step ks run
  double ar[2][TA], ai[2][TA], br[2][TB], bi[2][TB];
  auto frag = [&](int ks, int s) {
    const int k = ks * 4 + kq;
#pragma unroll
    for (int t = 0; t < TA; ++t) {
      const int ia = AKC ? (arow + t * 16 + m) * lda + k : k * lda + arow + t * 16 + m;
      ar[s][t] = Ar[ia];
      ai[s][t] = Ai[ia];
    }
#pragma unroll
    for (int t = 0; t < TB; ++t) {
      const int ib = BKC ? (bcol + t * 16 + m) * ldb + k : k * ldb + bcol + t * 16 + m;
      br[s][t] = Br[ib];
      bi[s][t] = Bi[ib];
    }
  };
  frag(0, 0);
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) {
    const int s = ks & 1;
    if (ks + 1 < NKS) frag(ks + 1, s ^ 1);
    double nai[TA];
#pragma unroll
    for (int t = 0; t < TA; ++t) nai[t] = -ai[s][t];
    const bool hook = kMid && ks == NKS - 1;
#pragma unroll
    for (int ti = 0; ti < TA; ++ti)
#pragma unroll
      for (int tj = 0; tj < TB; ++tj)
        cr[ti][tj] = ROWMAJ ? __builtin_amdgcn_mfma_f64_16x16x4f64(ar[s][ti], br[s][tj], cr[ti][tj], 0, 0, 0)
                            : __builtin_amdgcn_mfma_f64_16x16x4f64(br[s][tj], ar[s][ti], cr[ti][tj], 0, 0, 0);
    if (hook) { __builtin_amdgcn_sched_barrier(0); mid(0); __builtin_amdgcn_sched_barrier(0); }
#pragma unroll
    for (int ti = 0; ti < TA; ++ti)
#pragma unroll
      for (int tj = 0; tj < TB; ++tj)
        ci[ti][tj] = ROWMAJ ? __builtin_amdgcn_mfma_f64_16x16x4f64(ar[s][ti], bi[s][tj], ci[ti][tj], 0, 0, 0)
                            : __builtin_amdgcn_mfma_f64_16x16x4f64(bi[s][tj], ar[s][ti], ci[ti][tj], 0, 0, 0);
    if (hook) { __builtin_amdgcn_sched_barrier(0); mid(1); __builtin_amdgcn_sched_barrier(0); }
#pragma unroll
    for (int ti = 0; ti < TA; ++ti)
#pragma unroll
      for (int tj = 0; tj < TB; ++tj)
        cr[ti][tj] = ROWMAJ ? __builtin_amdgcn_mfma_f64_16x16x4f64(nai[ti], bi[s][tj], cr[ti][tj], 0, 0, 0)
                            : __builtin_amdgcn_mfma_f64_16x16x4f64(bi[s][tj], nai[ti], cr[ti][tj], 0, 0, 0);
    if (hook) { __builtin_amdgcn_sched_barrier(0); mid(2); __builtin_amdgcn_sched_barrier(0); }
#pragma unroll
    for (int ti = 0; ti < TA; ++ti)
#pragma unroll
      for (int tj = 0; tj < TB; ++tj)
        ci[ti][tj] = ROWMAJ ? __builtin_amdgcn_mfma_f64_16x16x4f64(ai[s][ti], br[s][tj], ci[ti][tj], 0, 0, 0)
                            : __builtin_amdgcn_mfma_f64_16x16x4f64(br[s][tj], ai[s][ti], ci[ti][tj], 0, 0, 0);
    if (hook) { __builtin_amdgcn_sched_barrier(0); mid(3); __builtin_amdgcn_sched_barrier(0); }
  }
}

// ------------------------------------------------------------------- GEMM
// C = op(A) op(B) (+ epilogue), n x n column-major (or row-major C when CRM),
// n a multiple of MR, MC and 32.  K panels of 16 are double-buffered in LDS; the
// next panel is fetched into registers while the current one is multiplied,
// then stored to the other stage before the single barrier of the panel.  The
// last panel of a tile fetches panel 0 of the next tile, so only the first tile
// has an exposed prologue.  Global addresses are a wave-uniform origin (scalar
// registers, advanced per panel and tile) plus a 32-bit byte offset per thread
// that is fixed for the whole GEMM.  Returns sum |C_ij| when ep.abs_sum (same
// value in every thread).
template <int T>
struct GemmLds {
  static constexpr int DOUBLES = 2 * Cfg<T>::STAGE;  // two stages (the abs-sum reduction reuses stage 0)
};

// Byte offset of each of a thread's panel elements from the panel origin.
template <int T, int OPA, int OPB>
__device__ __forceinline__ void gemm_panel_offsets(int n, uint32_t (&oa)[Cfg<T>::PERA],
                                                   uint32_t (&ob)[Cfg<T>::PERB]) {
  constexpr int MR = Cfg<T>::MR, MC = Cfg<T>::MC, NTH = Cfg<T>::NTH;
  const int tid = threadIdx.x;
#pragma unroll
  for (int q = 0; q < Cfg<T>::PERA; ++q) {
    const int idx = q * NTH + tid;
    if (OPA == OP_N) {
      const int i = idx % MR, k = idx / MR;  // A(row0 + i, k0 + k)
      oa[q] = (uint32_t)(i + k * n) * 16u;
    } else {
      const int k = idx % KP, i = idx / KP;  // conj A(k0 + k, row0 + i)
      oa[q] = (uint32_t)(k + i * n) * 16u;
    }
  }
#pragma unroll
  for (int q = 0; q < Cfg<T>::PERB; ++q) {
    const int idx = q * NTH + tid;
    if (OPB == OP_N) {
      const int k = idx % KP, j = idx / KP;  // B(k0 + k, col0 + j)
      ob[q] = (uint32_t)(k + j * n) * 16u;
    } else {
      const int j = idx % MC, k = idx / MC;  // conj B(col0 + j, k0 + k)
      ob[q] = (uint32_t)(j + k * n) * 16u;
    }
  }
}

template <int T, int OPA, int OPB>
__device__ __forceinline__ void gemm_load_panel(const double2* Ao, const double2* Bo,
                                                const uint32_t (&oa)[Cfg<T>::PERA], const uint32_t (&ob)[Cfg<T>::PERB],
                                                double2 (&ra)[Cfg<T>::PERA], double2 (&rb)[Cfg<T>::PERB]) {
#pragma unroll
  for (int q = 0; q < Cfg<T>::PERA; ++q) {
    ra[q] = ldgb(Ao, oa[q]);
    if (OPA == OP_C) ra[q] = cconj(ra[q]);
  }
#pragma unroll
  for (int q = 0; q < Cfg<T>::PERB; ++q) {
    rb[q] = ldgb(Bo, ob[q]);
    if (OPB == OP_C) rb[q] = cconj(rb[q]);
  }
}

// part = -1: the whole panel; 0..3: the elements q with q % 4 == part
template <int T, int OPA, int OPB>
__device__ __forceinline__ void gemm_store_panel(ldsd* st, const double2 (&ra)[Cfg<T>::PERA],
                                                 const double2 (&rb)[Cfg<T>::PERB], int part = -1) {
  constexpr int MR = Cfg<T>::MR, MC = Cfg<T>::MC, LDA = Cfg<T>::LDA, LDB = Cfg<T>::LDB, NTH = Cfg<T>::NTH;
  ldsd* Ar = st;
  ldsd* Ai = Ar + KP * LDA;
  ldsd* Br = Ai + KP * LDA;
  ldsd* Bi = Br + KP * LDB;
  const int tid = threadIdx.x;
#pragma unroll
  for (int q = 0; q < Cfg<T>::PERA; ++q) {
    if (part >= 0 && q % 4 != part) continue;
    const int idx = q * NTH + tid;
    int i, k;
    if (OPA == OP_N) { i = idx % MR; k = idx / MR; } else { k = idx % KP; i = idx / KP; }
    // k-contiguous layout when the global read runs along k (OP_C): conflict-free stores
    const int o = (OPA == OP_N) ? k * LDA + i : i * LDK + k;
    Ar[o] = ra[q].x;
    Ai[o] = ra[q].y;
  }
#pragma unroll
  for (int q = 0; q < Cfg<T>::PERB; ++q) {
    if (part >= 0 && q % 4 != part) continue;
    const int idx = q * NTH + tid;
    int j, k;
    if (OPB == OP_N) { k = idx % KP; j = idx / KP; } else { j = idx % MC; k = idx / MC; }
    const int o = (OPB == OP_N) ? j * LDK + k : k * LDB + j;
    Br[o] = rb[q].x;
    Bi[o] = rb[q].y;
  }
}

template <int M>
struct EpiMode {
  static constexpr int value = M;
};

// What becomes of sum |C_ij| in gemm_tiles: the thread's part of it (the result), or with
// another Sums the parts of each macro tile (add: an element, tile: the b-th 16 x 16 tile of
// the wave's part is complete, done: the part, at its row and column).  The epilogue takes it
// as an argument: captured, it changed the register allocation of the one-workgroup kernels
// (Born step at 64 orbitals 0.3% slower).
struct NoSums {
  __device__ void add(double2) {}
  __device__ void tile(int) {}
  __device__ void done(int, int) {}
};

// The output tiles rank, rank + size, ...; returns this thread's part of sum |C_ij|.
template <int T, int OPA, int OPB, int CRM, typename Sums = NoSums>
__device__ __forceinline__ double gemm_tiles(int n_, const double2* __restrict__ A_, const double2* __restrict__ B_,
                                             void* Cout_, Epi ep_, ldsd* lds, int rank, int size,
                                             Sums sums = Sums()) {
  using C = Cfg<T>;
  constexpr int MR = C::MR, MC = C::MC, LDA = C::LDA, LDB = C::LDB, STAGE = C::STAGE, TA = C::TA, TB = C::TB;
  constexpr bool AKC = (OPA != OP_N), BKC = (OPB == OP_N);
  const int n = uni(n_);
  const double2* A = uni(A_);
  const double2* B = uni(B_);
  void* Cout = uni(Cout_);
  Epi ep;
  ep.diag = uni(ep_.diag); ep.sacc = uni(ep_.sacc);
  ep.D1 = uni(ep_.D1); ep.s1 = uni(ep_.s1);
  ep.D2 = uni(ep_.D2); ep.s2 = uni(ep_.s2);
  ep.D3 = uni(ep_.D3); ep.s3 = uni(ep_.s3);
  ep.real_out = uni(ep_.real_out); ep.abs_sum = uni(ep_.abs_sum);
  const int emode = (ep.D2 || ep.D3 || ep.real_out || ep.abs_sum) ? 2 : (ep.D1 ? 1 : 0);
  const ldsd* s0Ar = lds;
  const ldsd* s0Ai = s0Ar + KP * LDA;
  const ldsd* s0Br = s0Ai + KP * LDA;
  const ldsd* s0Bi = s0Br + KP * LDB;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int arow = (wave % C::WR) * 16 * TA, bcol = (wave / C::WR) * 16 * TB;
  const int ntr = n / MR, ntiles = ntr * (n / MC), npan = n / KP;  // npan is even
  uint32_t oa[C::PERA], ob[C::PERB];
  gemm_panel_offsets<T, OPA, OPB>(n, oa, ob);
  // panel origins: A rows row0.. / B columns col0.., k from k0
  auto a_org = [&](int row0, int k0) -> const double2* {
    return OPA == OP_N ? A + row0 + (size_t)k0 * n : A + k0 + (size_t)row0 * n;
  };
  auto b_org = [&](int col0, int k0) -> const double2* {
    return OPB == OP_N ? B + k0 + (size_t)col0 * n : B + col0 + (size_t)k0 * n;
  };
  // epilogue: the thread's element of (ti, tj, r) is (row0 + it + di, col0 + jt + dj)
  const int m = lane & 15, kq = lane >> 4;
  const int it = CRM ? arow + kq : arow + m;
  const int jt = CRM ? bcol + m : bcol + kq;
  const uint32_t t_cm = (uint32_t)(it + jt * n), t_tr = (uint32_t)(jt + it * n);
  const uint32_t t_out = CRM ? t_tr : t_cm;
  double asum = 0.0;
  if (rank >= ntiles) return 0.0;
  double2 ra[C::PERA], rb[C::PERB];
  gemm_load_panel<T, OPA, OPB>(a_org((rank % ntr) * MR, 0), b_org((rank / ntr) * MC, 0), oa, ob, ra, rb);
  gemm_store_panel<T, OPA, OPB>(lds, ra, rb);
  __syncthreads();
  for (int tile = rank; tile < ntiles; tile += size) {
    const int row0 = (tile % ntr) * MR, col0 = (tile / ntr) * MC;
    const int tn = tile + size < ntiles ? tile + size : tile;  // the last tile refetches its own panel 0
    const int nrow0 = (tn % ntr) * MR, ncol0 = (tn / ntr) * MC;
    d4 cr[TA][TB], ci[TA][TB];
#pragma unroll
    for (int a = 0; a < TA; ++a)
#pragma unroll
      for (int b = 0; b < TB; ++b) { cr[a][b] = d4{0, 0, 0, 0}; ci[a][b] = d4{0, 0, 0, 0}; }
    for (int p = 0; p < npan; p += 2) {
      // stage 0 holds panel p; panel p + 1 goes to stage 1
      gemm_load_panel<T, OPA, OPB>(a_org(row0, (p + 1) * KP), b_org(col0, (p + 1) * KP), oa, ob, ra, rb);
      mma_steps<TA, TB, CRM, KP / 4, AKC, BKC>(cr, ci, s0Ar, s0Ai, AKC ? LDK : LDA, arow, s0Br, s0Bi, BKC ? LDK : LDB, bcol,
                                              [&](int g) { gemm_store_panel<T, OPA, OPB>(lds + STAGE, ra, rb, g); });
      __syncthreads();
      // stage 1 holds panel p + 1; panel p + 2 (or panel 0 of the next tile) goes to stage 0
      const bool last = p + 2 == npan;
      gemm_load_panel<T, OPA, OPB>(last ? a_org(nrow0, 0) : a_org(row0, (p + 2) * KP),
                                   last ? b_org(ncol0, 0) : b_org(col0, (p + 2) * KP), oa, ob, ra, rb);
      mma_steps<TA, TB, CRM, KP / 4, AKC, BKC>(cr, ci, s0Ar + STAGE, s0Ai + STAGE, AKC ? LDK : LDA, arow, s0Br + STAGE,
                                              s0Bi + STAGE, BKC ? LDK : LDB, bcol,
                                              [&](int g) { gemm_store_panel<T, OPA, OPB>(lds, ra, rb, g); });
      __syncthreads();
    }
    // epilogue, in batches of one 16x16 tile (4 elements per thread); the D-term
    // loads of the next batch are issued before the current batch is combined.
    // The variant is chosen once per tile (no per-element tests of the epilogue
    // fields): 0 = scale (+ diagonal) and store, 1 = plus s1*D1, 2 = general.
    const size_t cm0 = row0 + (size_t)col0 * n, tr0 = col0 + (size_t)row0 * n;
    auto di = [&](int ti, int r) { return CRM ? ti * 16 + 4 * r : ti * 16; };
    auto dj = [&](int tj, int r) { return CRM ? tj * 16 : tj * 16 + 4 * r; };
    auto epilogue = [&](auto mode, auto& acc) {
      constexpr int MODE = decltype(mode)::value;
      constexpr bool kSums = !__is_same(decltype(acc), NoSums&);
      auto load_d = [&](int b, double2 (&d1)[4], double2 (&d2)[4], double2 (&d3)[4]) {
        const int ti = b / TB, tj = b % TB;
        if (MODE == 1 || (MODE == 2 && ep.D1)) {
#pragma unroll
          for (int r = 0; r < 4; ++r) d1[r] = ldgb(ep.D1 + cm0 + di(ti, r) + (size_t)dj(tj, r) * n, 16u * t_cm);
        }
        if (MODE == 2 && ep.D2) {
#pragma unroll
          for (int r = 0; r < 4; ++r) d2[r] = ldgb(ep.D2 + cm0 + di(ti, r) + (size_t)dj(tj, r) * n, 16u * t_cm);
        }
        if (MODE == 2 && ep.D3) {
#pragma unroll
          for (int r = 0; r < 4; ++r) d3[r] = ldgb(ep.D3 + tr0 + dj(tj, r) + (size_t)di(ti, r) * n, 16u * t_tr);
        }
      };
      double2 n1[4], n2[4], n3[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) n1[r] = n2[r] = n3[r] = make_double2(0, 0);
      if (MODE > 0) load_d(0, n1, n2, n3);
#pragma unroll
      for (int b = 0; b < TA * TB; ++b) {
        const int ti = b / TB, tj = b % TB;
        double2 c1[4], c2[4], c3[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) { c1[r] = n1[r]; c2[r] = n2[r]; c3[r] = n3[r]; }
        if (MODE > 0 && b + 1 < TA * TB) load_d(b + 1, n1, n2, n3);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = row0 + it + di(ti, r), j = col0 + jt + dj(tj, r);
          double2 v = make_double2(ep.sacc * cr[ti][tj][r], ep.sacc * ci[ti][tj][r]);
          const double2 vd = cadd(v, ep.diag);
          v.x = (i == j) ? vd.x : v.x;
          v.y = (i == j) ? vd.y : v.y;
          if (MODE == 1) v = cadd(v, cmul(ep.s1, c1[r]));
          if (MODE == 2) {
            if (ep.D1) v = cadd(v, cmul(ep.s1, c1[r]));
            if (ep.D2) v = cadd(v, cmul(ep.s2, c2[r]));
            if (ep.D3) v = cadd(v, cmul(ep.s3, cconj(c3[r])));
            if (ep.abs_sum) {
              if constexpr (kSums) acc.add(v);
              else asum += sqrt(v.y * v.y + v.x * v.x);
            }
          }
          const size_t u = CRM ? tr0 + dj(tj, r) + (size_t)di(ti, r) * n : cm0 + di(ti, r) + (size_t)dj(tj, r) * n;
          if (MODE == 2 && ep.real_out)
            stgb_re((double*)Cout + u, 8u * t_out, v.x);
          else
            stgb((double2*)Cout + u, 16u * t_out, v);
        }
        if constexpr (MODE == 2 && kSums) {
          if (ep.abs_sum) acc.tile(b);
        }
      }
    };
    if (emode == 0)
      epilogue(EpiMode<0>(), sums);
    else if (emode == 1)
      epilogue(EpiMode<1>(), sums);
    else
      epilogue(EpiMode<2>(), sums);
    if (!__is_same(Sums, NoSums) && ep.abs_sum) sums.done(row0 + arow, col0 + bcol);
  }
  return asum;
}

template <int T, int OPA, int OPB, int CRM>
__device__ __noinline__ double wg_gemm_k(int n, const double2* __restrict__ A, const double2* __restrict__ B, void* Cout,
                                         Epi ep, ldsd* lds) {
  const double asum = gemm_tiles<T, OPA, OPB, CRM>(n, A, B, Cout, ep, lds, 0, 1);
  double s = 0.0;
  // stage 0 is free after the last panel's barrier
  if (uni(ep.abs_sum)) s = block_sum(asum, lds);
  __syncthreads();
  return s;
}

template <int T>
__device__ __forceinline__ double wg_gemm(int n, int opA, const double2* A, int opB, const double2* B, void* Cout,
                                          int c_rowmajor, Epi ep, ldsd* lds) {
  if (c_rowmajor) {
    if (opA == OP_N) {
      if (opB == OP_N) return wg_gemm_k<T, OP_N, OP_N, 1>(n, A, B, Cout, ep, lds);
      return wg_gemm_k<T, OP_N, OP_C, 1>(n, A, B, Cout, ep, lds);
    }
    if (opB == OP_N) return wg_gemm_k<T, OP_C, OP_N, 1>(n, A, B, Cout, ep, lds);
    return wg_gemm_k<T, OP_C, OP_C, 1>(n, A, B, Cout, ep, lds);
  }
  if (opA == OP_N) {
    if (opB == OP_N) return wg_gemm_k<T, OP_N, OP_N, 0>(n, A, B, Cout, ep, lds);
    return wg_gemm_k<T, OP_N, OP_C, 0>(n, A, B, Cout, ep, lds);
  }
  if (opB == OP_N) return wg_gemm_k<T, OP_C, OP_N, 0>(n, A, B, Cout, ep, lds);
  return wg_gemm_k<T, OP_C, OP_C, 0>(n, A, B, Cout, ep, lds);
}

// --------------------------------------------------------------- elementwise
// out(i,j) = diag*[i==j] + s1*D1(i,j) + s2*D2(i,j) + s3*conj(D3(j,i)); row-major
// output when out_rowmajor.  D1/D2 may alias out (not D3).
// The elements of share `rank` of `size`: a thread takes four at a time with all their
// loads in flight (one at a time the operation is as long as its loads' latencies), and
// steps its row and column instead of dividing the index.
__device__ __forceinline__ void ew_elements(int n, double2* out_, int out_rowmajor, double2 diag, const double2* D1_,
                                            double2 s1, const double2* D2_, double2 s2, const double2* D3_, double2 s3,
                                            int rank, int size) {
  constexpr int U = 4;
  const int nn = n * n, step = 256 * size, first = rank * 256 + (int)threadIdx.x;
  const int dslow = step / n, dfast = step - dslow * n;
  int slow = first / n, fast = first - slow * n;  // (j, i), or (i, j) when row-major
  double2* out = uni(out_);
  const double2 *D1 = uni(D1_), *D2 = uni(D2_), *D3 = uni(D3_);
  for (int idx = first; idx < nn; idx += U * step) {
    uint32_t o[U], t[U];  // offsets of the element and of its transpose, column-major
    bool in[U], dg[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      in[u] = idx + u * step < nn;
      const int i = in[u] ? (out_rowmajor ? slow : fast) : 0, j = in[u] ? (out_rowmajor ? fast : slow) : 0;
      o[u] = 16u * (uint32_t)(i + j * n);
      t[u] = 16u * (uint32_t)(j + i * n);
      dg[u] = i == j;
      fast += dfast;
      slow += dslow;
      if (fast >= n) {
        fast -= n;
        ++slow;
      }
    }
    double2 d1[U], d2[U], d3[U];
    if (D1) {
#pragma unroll
      for (int u = 0; u < U; ++u) d1[u] = ldgb(D1, o[u]);
    }
    if (D2) {
#pragma unroll
      for (int u = 0; u < U; ++u) d2[u] = ldgb(D2, o[u]);
    }
    if (D3) {
#pragma unroll
      for (int u = 0; u < U; ++u) d3[u] = ldgb(D3, t[u]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      double2 v = make_double2(dg[u] ? diag.x : 0.0, dg[u] ? diag.y : 0.0);
      if (D1) v = cadd(v, cmul(s1, d1[u]));
      if (D2) v = cadd(v, cmul(s2, d2[u]));
      if (D3) v = cadd(v, cmul(s3, cconj(d3[u])));
      if (in[u]) stgb(out, out_rowmajor ? t[u] : o[u], v);
    }
  }
}

__device__ __noinline__ void wg_ew(int n, double2* out, int out_rowmajor, double2 diag,
                                   const double2* D1, double2 s1, const double2* D2, double2 s2,
                                   const double2* D3, double2 s3) {
  ew_elements(uni(n), out, uni(out_rowmajor), diag, D1, s1, D2, s2, D3, s3, 0, 1);
  __syncthreads();
}

// out = (X - X^H) / 2, the anti-Hermitian part of X (n a multiple of 32, out must not
// alias X).  The 32 x 32 tile pairs (I, J), (J, I), I <= J, are read down their
// columns into LDS, the pair's two output tiles are written down their columns; the
// next pair's elements are loaded into registers while the current pair is combined.
// LDS: kAntihermLds doubles; 256 threads.
constexpr int kAntihermLds = 4 * 32 * 33;
// Pairs q = rank, rank + size, ...
__device__ __noinline__ void antiherm_pairs(int n, const double2* X_, double2* out_, ldsd* lds, int rank, int size) {
  constexpr int TS = 32, LD = TS + 1, PER = TS * TS / 256;
  static_assert(4 * TS * LD == kAntihermLds, "LDS size");
  const gcd2* X = gc(X_);
  gd2* out = gw(out_);
  ldsd* Ar = lds;
  ldsd* Ai = Ar + TS * LD;
  ldsd* Br = Ai + TS * LD;
  ldsd* Bi = Br + TS * LD;
  const int nt = n / TS, npair = nt * (nt + 1) / 2;
  const int tid = threadIdx.x;  // element k of a tile: row tid % 32, column tid / 32 + 8k
  const int r = tid % TS, c0 = tid / TS;
  auto pair_of = [&](int q, int& I, int& J) {  // q-th pair (I <= J), row by row
    I = 0;
    while (q >= nt - I) { q -= nt - I; ++I; }
    J = I + q;
  };
  double2 ra[PER], rb[PER];
  auto load = [&](int q) {
    int I, J;
    pair_of(q, I, J);
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int c = c0 + 8 * k;
      ra[k] = X[(size_t)(I * TS + r) + (size_t)(J * TS + c) * n];
      rb[k] = X[(size_t)(J * TS + r) + (size_t)(I * TS + c) * n];
    }
  };
  if (rank < npair) load(rank);
  for (int q = rank; q < npair; q += size) {
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int c = c0 + 8 * k;
      Ar[c * LD + r] = ra[k].x; Ai[c * LD + r] = ra[k].y;
      Br[c * LD + r] = rb[k].x; Bi[c * LD + r] = rb[k].y;
    }
    __syncthreads();
    if (q + size < npair) load(q + size);
    int I, J;
    pair_of(q, I, J);
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int c = c0 + 8 * k;
      // A = X[I-tile rows, J-tile cols] at (c, r) of the LDS tile, B likewise
      out[(size_t)(I * TS + r) + (size_t)(J * TS + c) * n] =
          make_double2(0.5 * (Ar[c * LD + r] - Br[r * LD + c]), 0.5 * (Ai[c * LD + r] + Bi[r * LD + c]));
      if (I != J)
        out[(size_t)(J * TS + r) + (size_t)(I * TS + c) * n] =
            make_double2(0.5 * (Br[c * LD + r] - Ar[r * LD + c]), 0.5 * (Bi[c * LD + r] + Ai[r * LD + c]));
    }
    __syncthreads();
  }
}
__device__ __forceinline__ void wg_antiherm(int n, const double2* X, double2* out, ldsd* lds) {
  antiherm_pairs(n, X, out, lds, 0, 1);
}

// Y = i Im X (real parts zeroed); Z = X as well when Z is given.  Y, Z must not alias X.
__device__ __noinline__ void wg_imag_part(int n, const double2* X, double2* Y, double2* Z) {
  const int nn = n * n;
  for (int idx = threadIdx.x; idx < nn; idx += blockDim.x) {
    const double2 v = gc(X)[idx];
    gw(Y)[idx] = make_double2(0.0, v.y);
    if (Z) gw(Z)[idx] = v;
  }
  __syncthreads();
}

// Re sum_ij X(i,j) Y(j,i) = Re Tr(X Y).
__device__ __noinline__ double wg_retrace_prod(int n, const double2* X, const double2* Y, ldsd* red) {
  double s = 0.0;
  const int nn = n * n;
  for (int idx = threadIdx.x; idx < nn; idx += blockDim.x) {
    const int i = idx % n, j = idx / n;
    double2 x = gc(X)[i + (size_t)j * n], y = gc(Y)[j + (size_t)i * n];
    s += x.x * y.x - x.y * y.y;
  }
  return block_sum(s, red);
}

// Im Tr(X).
__device__ __forceinline__ double wg_imtrace(int n, const double2* X, ldsd* red) {
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += blockDim.x) s += gc(X)[i + (size_t)i * n].y;
  return block_sum(s, red);
}

// --------------------------------------------------- Gauss-Jordan column steps
// Maximum over the wave of an int, uniform result: DPP swaps within rows of 16 lanes,
// then lane 15 of rows 0 / 2 into rows 1 / 3 and lane 31 into rows 2, 3; lane 63 holds
// the maximum of all.
__device__ __forceinline__ int wave_max_i32(int v) {
  // (old values chosen so that each exchange folds into its maximum)
  constexpr int lowest = (int)0x80000000;
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xf, 0xf, true));   // quad_perm [1,0,3,2]
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xf, 0xf, true));   // quad_perm [2,3,0,1]
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, true));  // row_half_mirror
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x140, 0xf, 0xf, true));  // row_mirror
  v = max(v, __builtin_amdgcn_update_dpp(lowest, v, 0x142, 0xa, 0xf, false));  // row_bcast:15 into rows 1, 3
  v = max(v, __builtin_amdgcn_update_dpp(lowest, v, 0x143, 0xc, 0xf, false));  // row_bcast:31 into rows 2, 3
  return __builtin_amdgcn_readlane(v, 63);
}

// Row of the largest v >= 0 over the wave, the lowest row among equal values; -1 when
// every v is negative or zero.  Each lane brings its own largest value and its row.
// Non-negative doubles order like their bit patterns, so the high words decide unless
// several lanes share the largest one (or it is zero), where the low words do.
__device__ __forceinline__ int wave_pivot(double v, int row) {
  const long long bits = __builtin_bit_cast(long long, v);
  const int hi = (int)(bits >> 32);
  const int mh = wave_max_i32(hi);
  if (mh < 0) return -1;
  unsigned long long hit = __ballot(hi == mh);
  if (mh == 0 || __builtin_popcountll(hit) > 1) {
    // unsigned order of the low words as signed ints
    const int lo = (hi == mh) ? (int)((unsigned)bits ^ 0x80000000u) : (int)0x80000000;
    const int ml = wave_max_i32(lo);
    if (mh == 0 && ml == (int)0x80000000) return -1;
    const bool top = hi == mh && lo == ml;
    const int r = wave_max_i32(top ? -row : (int)0x80000000);
    return -r;
  }
  return __builtin_amdgcn_readlane(row, __builtin_ctzll(hit));
}

// f(Index<i>()) for a wave-uniform i in [LO, HI): the registers that f reads keep static
// indexes, one of log2 uniform branches is taken at each level.
template <int I>
struct Index {
  static constexpr int value = I;
};
template <int LO, int HI, typename F>
__device__ __forceinline__ void at_index(int i, const F& f) {
  if constexpr (HI - LO == 1) {
    f(Index<LO>());
  } else {
    constexpr int MID = (LO + HI) / 2;
    if (i < MID)
      at_index<LO, MID>(i, f);
    else
      at_index<MID, HI>(i, f);
  }
}

#if defined(__HIP_DEVICE_COMPILE__)
typedef __attribute__((address_space(3))) dvec2 ldsv;
#else
typedef dvec2 ldsv;
#endif

template <int RT, int CT, int HV>
struct GjLds {
  static constexpr int ROWS = (64 / HV) * RT;
  static constexpr int COL = 2 * ROWS + 4;            // the column, its pivot, the pivot's row
  static constexpr int ROW = HV == 2 ? 2 * CT * HV : 0;  // a wave's part of the pivot row
  static constexpr int DOUBLES = 2 * COL + 4 * ROW;   // columns by parity, rows by wave
};

// Gauss-Jordan sweep of 4 HV CT columns held in registers by 4 waves: lane l of wave w
// holds rows (l mod 64/HV) + (64/HV) r, r < RT, of the CT columns of column block
// cb = w HV + l / (64/HV).  Per column k the wave that holds it chooses the pivot row p
// (the first maximum of |Re| + |Im| over the rows not yet used, as izamax in zgetrf) and
// publishes the column through LDS with a zero in the pivot's place, then restarts its
// registers of the column from the unit vector of p; after one barrier every wave takes
// its own part of row p from the lane that holds it (readlane, no second exchange) and
// updates a_ij -= (a_ik / a_pk) a_pj.  Row p itself is left as it is (its factor is the
// published zero) and scaled by 1 / a_pk after the last column, which commutes with the
// later updates of the row.  Only the holding wave's part depends on the column's
// register, so the code of a step is short (the fully unrolled sweep of a 256 x 32 panel
// was 130 KB and ran from L2).  Column buffers alternate by column parity: a column's
// reads are over before the barrier after which the next write to them starts.
// A column step is a serial chain (pivot search, exchange, reciprocal, update), so its
// length counts, not its operations; this split needs one barrier and no broadcast of
// the pivot row.  Inverse of 256 blocks, one per CU, against one panel row per thread
// (four candidate rows of 16 exchanged and scaled in every thread): n = 32 35 -> 27 us,
// 64 159 -> 77, 96 300 -> 185, 128 449 -> 298.
// Returns 0 or the 1-based column without a nonzero pivot; piv[c] is the row of column c.
template <int RT, int CT, int HV>
__device__ __forceinline__ int gj_sweep(double2 (&a)[RT][CT], int nrow, unsigned& used, ldsi* piv, ldsd* xch) {
  constexpr int RL = 64 / HV;
  static_assert(HV == 1 || RT == 1, "half waves hold one row per lane");
  const int lane = threadIdx.x & 63, wave = uni((int)(threadIdx.x >> 6));
  const int row = lane % RL, half = lane / RL;
  double2 sc[RT];       // 1 / pivot of a row that has been one in this sweep
  unsigned here = 0;    // bit r: it has
  int fail = 0;
  ldsv* prow_mine = (ldsv*)(xch + 2 * GjLds<RT, CT, HV>::COL) + (wave * HV + half) * CT;
#pragma unroll
  for (int r = 0; r < RT; ++r) sc[r] = make_double2(1, 0);
#pragma unroll 1
  for (int k = 0; k < 4 * HV * CT; ++k) {
    ldsd* xc = xch + (k & 1) * (GjLds<RT, CT, HV>::COL);
    ldsv* col = (ldsv*)xc;
    ldsv* pivot = (ldsv*)(xc + 2 * RL * RT);
    ldsi* prow = (ldsi*)(xc + 2 * RL * RT + 2);
    const int h = k / CT;  // column block
    if (wave == h / HV) {
      const bool mine = half == h % HV;
      at_index<0, CT>(k % CT, [&](auto ix) {
        constexpr int cc = decltype(ix)::value;
        double bv = -1.0;
        int br = 0;
#pragma unroll
        for (int r = 0; r < RT; ++r) {
          const double v = fabs(a[r][cc].x) + fabs(a[r][cc].y);
          if (mine && row + RL * r < nrow && !((used >> r) & 1u) && v > bv) { bv = v; br = r; }
        }
        const int p = wave_pivot(bv, row + RL * br);
#pragma unroll
        for (int r = 0; r < RT; ++r) {
          const bool isp = row + RL * r == p;
          dvec2 v;
          v.x = a[r][cc].x;
          v.y = a[r][cc].y;
          if (mine) {
            if (isp) *pivot = v;
            v.x = isp ? 0.0 : v.x;
            v.y = isp ? 0.0 : v.y;
            col[row + RL * r] = v;
            a[r][cc].x = isp ? 1.0 : 0.0;
            a[r][cc].y = 0.0;
          }
        }
        if (lane == 0) {
          *prow = p;
          piv[k] = p < 0 ? 0 : p;
        }
      });
    }
    __syncthreads();
    const int p0 = *prow;
    const dvec2 pv = *pivot;
    double2 g[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const dvec2 v = col[row + RL * r];
      g[r] = make_double2(v.x, v.y);
    }
    // a column without a pivot is noted and the sweep runs on (its results are not used):
    // a branch here would put the reads above behind the row's
    const int pu = uni(p0);
    if (pu < 0 && !fail) fail = k + 1;
    const int p = pu < 0 ? 0 : pu;
    // row p's entries of this wave's columns
    const int pl = p % RL;
    double2 rw[CT];
    if constexpr (HV == 2) {
      // through LDS (a wave's LDS operations are in order, so without a barrier): the
      // half waves read different columns
      if (row == pl) {
#pragma unroll
        for (int c = 0; c < CT; ++c) {
          dvec2 v;
          v.x = a[0][c].x;
          v.y = a[0][c].y;
          prow_mine[c] = v;
        }
      }
      // (the fences emit nothing: they keep the compiler from moving the reads up)
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        const dvec2 v = prow_mine[c];
        rw[c] = make_double2(v.x, v.y);
      }
    } else {
      // (through LDS one lane's 16 writes alone take longer than 64 readlanes)
      at_index<0, RT>(p / RL, [&](auto ix) {
        constexpr int pr = decltype(ix)::value;
#pragma unroll
        for (int c = 0; c < CT; ++c) rw[c] = make_double2(lane_f64(a[pr][c].x, pl), lane_f64(a[pr][c].y, pl));
      });
    }
    const double2 ainv = crecip_uniform(make_double2(pv.x, pv.y));
    const unsigned bit = row == pl ? 1u << (p / RL) : 0u;
    used |= bit;
    here |= bit;
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      sc[r].x = row + RL * r == p ? ainv.x : sc[r].x;
      sc[r].y = row + RL * r == p ? ainv.y : sc[r].y;
      g[r] = cmul(g[r], ainv);
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        a[r][c].x = fma(g[r].y, rw[c].y, fma(-g[r].x, rw[c].x, a[r][c].x));
        a[r][c].y = fma(-g[r].y, rw[c].x, fma(-g[r].x, rw[c].y, a[r][c].y));
      }
    }
  }
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    if ((here >> r) & 1u) {
#pragma unroll
      for (int c = 0; c < CT; ++c) a[r][c] = cmul(a[r][c], sc[r]);
    }
  }
  return fail;
}

// ------------------------------------------------------------------ inverse
// In-place blocked Gauss-Jordan inverse with partial row pivoting (pivot =
// first maximum of |Re|+|Im| among the rows not yet used, the izamax choice of
// zgetrf) and logical row exchanges.  W is row-major n x n and is destroyed;
// the inverse is written column-major to out.  Returns 0, or k+1 when column k
// has no nonzero pivot, in which case out is zeroed (src/green_rgf.f90:4429-4437).
//
// Panel step (32 columns K, pivot rows P): the panel is swept in registers
// (gj_sweep), giving F_P = A_PK^-1 and F_R = -A_RK A_PK^-1; the other
// columns J are updated on MFMA, W[:,J] += (F - E) W[P,J] with E the pivot
// incidence (accumulating onto the loaded tiles of W), and columns K take F.
// out (a separate n x n buffer) receives inv(i, q) = W[piv[i]][pinv[q]] after the
// last panel.
//
// 65 to 256 rows.  From 129 on the panel updates read and write the whole of W from HBM
// (256 workgroups hold 256 MB), so the number of passes counts: 32 columns halve those of
// a 16-column panel.  The swept panel M = F - E (32 x n)
// fills the LDS; W is updated in strips of 16 columns, each with its part of the pivot
// rows staged beside M, and the next strip is loaded while the current one is multiplied
// (without that overlap the 32-column panels are slower: 1844 us, below).
// Rows of M alternate by 16 doubles (row k's index is xored with 16 (k & 1)) in place of a
// padded stride, which LDS has no room for: the four k of a fragment read then fall on
// distinct banks as with a stride of 16 mod 32.
// Strips belong to the ranks of a group in turn (a lone workgroup has all); every rank
// sweeps the panel for itself.  A panel's own columns take F one step late, after the
// ranks have all read the panel.  256 blocks, one per CU, 16-column panels -> this: n = 160
// 587 -> 553 us, 192 767 -> 776, 224 1287 -> 1159, 256 1624 -> 1527.  At 96 and 128 against
// whole tiles with all of the pivot rows beside M: 184 -> 182 and 304 -> 288 us (8 blocks:
// 153 -> 149, 245 -> 229): the strips' loads run under the MFMAs, and a panel's own columns
// are not multiplied.
template <int NMAX>
struct InvStripLds {
  static constexpr int KPI = 32, SC = 16;
  static constexpr int S1 = 2 * KPI * SC;  // re / im planes of a strip's pivot rows, two buffers
  static constexpr int OFF_S = 2 * KPI * NMAX, OFF_PIV = OFF_S + 2 * S1;
  static constexpr int DOUBLES = OFF_PIV + NMAX;  // + piv, pinv (2 NMAX ints)
};

template <int NMAX, typename N>
__device__ __noinline__ int wg_inverse_strip(N n_, double2* W_, double2* out_, ldsd* lds) {
  using L = InvStripLds<NMAX>;
  constexpr int KPI = L::KPI, SC = L::SC, NTH = 256;
  constexpr int RT = NMAX / 64, CT = KPI / 4, PS = KPI * SC / NTH;
  static_assert(NMAX % 64 == 0 && NMAX <= NTH, "four waves of row tiles");
  static_assert(GjLds<RT, CT, 1>::DOUBLES <= 2 * L::S1, "the column exchange fits the pivot-row area");
  const int n = uni((int)n_), rank = uni(group_rank(n_)), size = uni(group_size(n_));
  double2* Wp = uni(W_);
  gd2* out = gw(uni(out_));
  ldsd* Mr = lds;
  ldsd* Mi = lds + KPI * NMAX;
  ldsd* S = lds + L::OFF_S;
  ldsi* piv = (ldsi*)(lds + L::OFF_PIV);
  ldsi* pinv = piv + NMAX;
  const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6);
  const int m = lane & 15, kq = lane >> 4;
  auto mix = [&](int k, int i) { return k * NMAX + (i ^ ((k & 1) << 4)); };
  // columns k0.. of W take F = M + E
  auto late = [&](int k0) {
    if ((k0 / SC + (wave >> 1)) % size != rank) return;  // waves 0, 1 hold the first strip
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const int i = lane + 64 * r;
      if (i < n) {
#pragma unroll
        for (int c = 0; c < CT; ++c) {
          const int k = wave * CT + c;
          double2 f = make_double2(Mr[mix(k, i)], Mi[mix(k, i)]);
          f.x += piv[k0 + k] == i ? 1.0 : 0.0;
          stgb(Wp + k0 + k, 16u * (uint32_t)(i * n), f);
        }
      }
    }
  };
  int info = 0, k0 = 0;
  unsigned used = 0;  // bit r: row lane + 64 r has been a pivot
  for (; k0 < n; k0 += KPI) {
    double2 a[RT][CT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int c = 0; c < CT; ++c)
        a[r][c] = lane + 64 * r < n ? ldgb(Wp + k0 + wave * CT + c, 16u * (uint32_t)((lane + 64 * r) * n)) : make_double2(0, 0);
    if (k0) late(k0 - KPI);
    info = gj_sweep<RT, CT, 1>(a, n, used, piv + k0, S);
    if (info) {
      info += k0;
      break;
    }
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int c = 0; c < CT; ++c)
        if (lane + 64 * r < n) {
          Mr[mix(wave * CT + c, lane + 64 * r)] = a[r][c].x;
          Mi[mix(wave * CT + c, lane + 64 * r)] = a[r][c].y;
        }
    __syncthreads();
    if (tid < KPI) Mr[mix(tid, piv[k0 + tid])] -= 1.0;  // M = F - E
    // the rank's strips but the panel's own; -1: none left
    auto next = [&](int s) {
      while (s < n / SC && s / (KPI / SC) == k0 / KPI) s += size;
      return s < n / SC ? s : -1;
    };
    double2 v[PS];             // the pivot rows' part of a strip, before they are updated
    d4 cr[RT], ci[RT];         // the strip: rows (wave + 4 q) 16 + 4 r + kq, column m
    const uint32_t t_off = 16u * (uint32_t)(kq * n + m);
    auto fetch = [&](int s, double2 (&pv)[PS], d4 (&xr)[RT], d4 (&xi)[RT]) {
      const double2* Ws = Wp + s * SC;
#pragma unroll
      for (int q = 0; q < PS; ++q) {
        const int idx = q * NTH + tid, c = idx / SC, j = idx % SC;
        pv[q] = ldgb(Ws, 16u * (uint32_t)(piv[k0 + c] * n + j));
      }
#pragma unroll
      for (int q = 0; q < RT; ++q) {
        if ((wave + 4 * q) * 16 < n) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const double2 o = ldgb(Ws + (size_t)((wave + 4 * q) * 16 + 4 * r) * n, t_off);
            xr[q][r] = o.x;
            xi[q][r] = o.y;
          }
        }
      }
    };
    int s = next(rank), buf = 0;
    if (s >= 0) fetch(s, v, cr, ci);
    while (s >= 0) {
      ldsd* Sr = S + buf * L::S1;
      ldsd* Si = Sr + KPI * SC;
#pragma unroll
      for (int q = 0; q < PS; ++q) {
        Sr[q * NTH + tid] = v[q].x;
        Si[q * NTH + tid] = v[q].y;
      }
      __syncthreads();  // this strip's pivot rows (and M) complete; the buffer's last readers are two strips back
      const int sn = next(s + size);
      d4 nr[RT], ni[RT];
      if (sn >= 0) fetch(sn, v, nr, ni);
      // rows past n are multiplied too (their M is whatever LDS holds) and not stored: a
      // guard would keep the fragment reads from running ahead of the MFMAs
#pragma unroll
      for (int ks = 0; ks < KPI / 4; ++ks) {
        const int k = ks * 4 + kq;
        const double br = Sr[k * SC + m], bi = Si[k * SC + m];
        double ar[RT], ai[RT];
#pragma unroll
        for (int q = 0; q < RT; ++q) {
          ar[q] = Mr[mix(k, (wave + 4 * q) * 16 + m)];
          ai[q] = Mi[mix(k, (wave + 4 * q) * 16 + m)];
        }
#pragma unroll
        for (int q = 0; q < RT; ++q) cr[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[q], br, cr[q], 0, 0, 0);
#pragma unroll
        for (int q = 0; q < RT; ++q) ci[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[q], bi, ci[q], 0, 0, 0);
#pragma unroll
        for (int q = 0; q < RT; ++q) cr[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(-ai[q], bi, cr[q], 0, 0, 0);
#pragma unroll
        for (int q = 0; q < RT; ++q) ci[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai[q], br, ci[q], 0, 0, 0);
      }
#pragma unroll
      for (int q = 0; q < RT; ++q) {
        if ((wave + 4 * q) * 16 < n) {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            stgb(Wp + s * SC + (size_t)((wave + 4 * q) * 16 + 4 * r) * n, t_off, make_double2(cr[q][r], ci[q][r]));
        }
        cr[q] = nr[q];
        ci[q] = ni[q];
      }
      s = sn;
      buf ^= 1;
    }
    group_sync(n_);
  }
  // a group's barriers do not depend on the block: after a panel without a pivot the rest follow
  for (; k0 < n; k0 += KPI) group_sync(n_);
  if (!info) {
    late(n - KPI);
    for (int q = tid; q < n; q += NTH) pinv[piv[q]] = q;  // inverse permutation
  }
  group_sync(n_);
  // out(i, q) = W[piv[i]][pinv[q]], RB rows of out at a time: the source rows are read
  // whole into LDS and out is written in column segments of RB elements
  constexpr int RB = 16;
  static_assert(2 * RB * (NMAX + 1) <= L::OFF_S, "row block fits the panel area");
  const int ldr = n + 1;  // odd stride: the RB rows of one column sit in distinct banks
  ldsd* Lr = Mr;
  ldsd* Li = Mr + RB * ldr;
  for (int i0 = rank * RB; i0 < n; i0 += size * RB) {
    if (info) {
      for (int idx = tid; idx < RB * n; idx += NTH) out[(size_t)(i0 + idx % RB) + (size_t)(idx / RB) * n] = make_double2(0, 0);
      continue;
    }
    if (tid < n) {
      double2 v[RB];
#pragma unroll
      for (int rr = 0; rr < RB; ++rr) v[rr] = ldgb(Wp, 16u * (uint32_t)(piv[i0 + rr] * n + tid));
#pragma unroll
      for (int rr = 0; rr < RB; ++rr) {
        Lr[rr * ldr + tid] = v[rr].x;
        Li[rr * ldr + tid] = v[rr].y;
      }
    }
    __syncthreads();
    for (int idx = tid; idx < RB * n; idx += NTH) {
      const int rr = idx % RB, q = idx / RB;
      const int c = pinv[q];
      out[(size_t)(i0 + rr) + (size_t)q * n] = make_double2(Lr[rr * ldr + c], Li[rr * ldr + c]);
    }
    __syncthreads();
  }
  group_sync(n_);
  return info;
}

// ------------------------------------------------------ inverse, n > NTH
// The same Gauss-Jordan sweep for blocks larger than the workgroup (NMAX rows,
// RPT = NMAX / NTH panel rows per thread).  The swept panel M = F - E (n x KP,
// row-major) and the snapshot of the KP pivot rows (KP x n) do not fit in LDS at
// these sizes; they are kept in `out`, which is free until the final permutation
// copy, and staged per update tile through LDS (one K = KP panel of the tile's
// rows of M and columns of the snapshot), so the update of W is a K = 16 MFMA GEMM
// per tile accumulating onto the tile's old values as for n <= NTH.
template <int T, int NMAX>
struct InvBigLds {
  static constexpr int LDA = Cfg<T>::MR + PAD, LDB = Cfg<T>::MC + PAD;
  static constexpr int RB = 8;                                 // rows per step of the final copy
  static constexpr int PANELS = 2 * KP * LDA + 2 * KP * LDB;  // staged M rows and snapshot columns
  static constexpr int COPY = 2 * RB * (NMAX + 1);
  static constexpr int OFF_IDX = PANELS > COPY ? PANELS : COPY;  // piv, used after the larger area
  static constexpr int XCH = 2 * (4 * 2 * KP) + 2 * 8;          // pivot-row exchange, two parities
  static constexpr int DOUBLES = OFF_IDX + NMAX + XCH + 16;      // piv + used = 2 NMAX ints
};

__device__ __forceinline__ int wave_min_int(int v) {
  for (int off = 32; off > 0; off >>= 1) v = min(v, __shfl_xor(v, off, 64));
  return v;
}

template <int T, int NMAX>
__device__ __noinline__ int wg_inverse_big(int n, double2* W_, double2* out_, ldsd* lds) {
  using C = Cfg<T>;
  using L = InvBigLds<T, NMAX>;
  constexpr int NTH = C::NTH, RPT = (NMAX + NTH - 1) / NTH;
  constexpr int MR = C::MR, MC = C::MC, TA = C::TA, TB = C::TB, LDA = L::LDA, LDB = L::LDB;
  static_assert(RPT <= 8, "panel rows per thread");
  gd2* W = gw(W_);
  gd2* out = gw(out_);
  gd2* Mg = out;                       // M = F - E, row-major n x KP
  gd2* Sg = out + (size_t)n * KP;      // pivot-row snapshot, KP x n (row c at c * n)
  ldsd* Ar = lds;
  ldsd* Ai = Ar + KP * LDA;
  ldsd* Br = Ai + KP * LDA;
  ldsd* Bi = Br + KP * LDB;
  ldsi* piv = (ldsi*)(lds + L::OFF_IDX);
  ldsi* used = piv + NMAX;
  ldsd* xch = (ldsd*)(used + NMAX);  // [parity][wave][2 KP] rows, then [parity][8] values / rows
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int arow = (wave % C::WR) * 16 * TA, bcol = (wave / C::WR) * 16 * TB;
  for (int i = tid; i < n; i += NTH) used[i] = 0;
  __syncthreads();
  int info = 0;
  unsigned myused = 0;  // bit q: row tid + q * NTH has been a pivot
  for (int k0 = 0; k0 < n && !info; k0 += KP) {
    double2 rv[RPT][KP];
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
      const int r = tid + q * NTH;
#pragma unroll
      for (int c2 = 0; c2 < KP; ++c2) rv[q][c2] = r < n ? W[(size_t)r * n + k0 + c2] : make_double2(0, 0);
    }
    for (int c = 0; c < KP; ++c) {
      // the thread's candidate: first maximum of |Re| + |Im| over its unused rows
      double myv = -1.0;
      int myq = 0;
#pragma unroll
      for (int q = 0; q < RPT; ++q) {
        double2 cand = make_double2(0, 0);
#pragma unroll
        for (int c2 = 0; c2 < KP; ++c2)
          if (c2 == c) cand = rv[q][c2];
        const bool valid = (tid + q * NTH) < n && !((myused >> q) & 1u);
        const double v = valid ? fabs(cand.x) + fabs(cand.y) : -1.0;
        if (v > myv) { myv = v; myq = q; }
      }
      const int myrow = tid + myq * NTH;
      double best = wave_max(myv);
      int brow = wave_min_int((myv == best && myv >= 0.0) ? myrow : 0x7fffffff);
      ldsd* xrow = xch + (c & 1) * (4 * 2 * KP);
      ldsd* xval = xch + 2 * (4 * 2 * KP) + (c & 1) * 8;
      if (myrow == brow) {
#pragma unroll
        for (int q = 0; q < RPT; ++q)
          if (q == myq) {
#pragma unroll
            for (int c2 = 0; c2 < KP; ++c2) {
              xrow[wave * 2 * KP + 2 * c2] = rv[q][c2].x;
              xrow[wave * 2 * KP + 2 * c2 + 1] = rv[q][c2].y;
            }
          }
      }
      if (lane == 0) { xval[wave] = best; xval[4 + wave] = (double)brow; }
      __syncthreads();
      best = xval[0];
      int bw = 0;
      int bi = (int)xval[4];
      for (int w = 1; w < NTH / 64; ++w) {
        const double ov = xval[w];
        const int oi = (int)xval[4 + w];
        if (ov > best || (ov == best && oi < bi)) { best = ov; bi = oi; bw = w; }
      }
      if (!(best > 0.0)) { info = k0 + c + 1; break; }
      const int p = bi;
      const ldsd* prow = xrow + bw * 2 * KP;
      const double2 ainv = crecip(make_double2(prow[2 * c], prow[2 * c + 1]));
      double2 rp[KP];
#pragma unroll
      for (int c2 = 0; c2 < KP; ++c2)
        rp[c2] = (c2 == c) ? ainv : cmul(make_double2(prow[2 * c2], prow[2 * c2 + 1]), ainv);
#pragma unroll
      for (int q = 0; q < RPT; ++q) {
        const int r = tid + q * NTH;
        if (r == p) {
          myused |= 1u << q;
          used[p] = 1;
          piv[k0 + c] = p;
#pragma unroll
          for (int c2 = 0; c2 < KP; ++c2) rv[q][c2] = rp[c2];
        } else if (r < n) {
          double2 f = make_double2(0, 0);
#pragma unroll
          for (int c2 = 0; c2 < KP; ++c2)
            if (c2 == c) f = rv[q][c2];
#pragma unroll
          for (int c2 = 0; c2 < KP; ++c2) rv[q][c2] = csub((c2 == c) ? make_double2(0, 0) : rv[q][c2], cmul(f, rp[c2]));
        }
      }
    }
    if (info) break;
    __syncthreads();  // piv of this panel visible to every thread
    // M = F - E into out (row-major n x KP): a pivot row p = piv[k0 + c] has 1 subtracted at column c
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
      const int r = tid + q * NTH;
      if (r < n) {
#pragma unroll
        for (int c2 = 0; c2 < KP; ++c2) {
          double2 v = rv[q][c2];
          v.x -= (piv[k0 + c2] == r) ? 1.0 : 0.0;
          Mg[(size_t)r * KP + c2] = v;
        }
      }
    }
    // snapshot of the pivot rows before the update changes them, all loads of a thread in flight
    for (int j0 = 0; j0 < n; j0 += NTH) {
      const int j = j0 + tid;
      if (j < n) {
        double2 v[KP];
#pragma unroll
        for (int c2 = 0; c2 < KP; ++c2) v[c2] = W[(size_t)piv[k0 + c2] * n + j];
#pragma unroll
        for (int c2 = 0; c2 < KP; ++c2) Sg[(size_t)c2 * n + j] = v[c2];
      }
    }
    __syncthreads();
    const int ntr = n / MR, ntc = n / MC;
    const int m = lane & 15, kq = lane >> 4;
    const uint32_t t_off = 16u * (uint32_t)((arow + kq) * n + bcol + m);
    for (int tile = 0; tile < ntr * ntc; ++tile) {
      const int row0 = (tile % ntr) * MR, col0 = (tile / ntr) * MC;
      d4 cr[TA][TB], ci[TA][TB];
#pragma unroll
      for (int ti = 0; ti < TA; ++ti)
#pragma unroll
        for (int tj = 0; tj < TB; ++tj)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const double2 o = ldgb(W_ + (size_t)(row0 + ti * 16 + 4 * r) * n + col0 + tj * 16, t_off);
            cr[ti][tj][r] = o.x;
            ci[ti][tj][r] = o.y;
          }
      // stage M rows row0.. (k-major, [c][i]) and snapshot columns col0.. ([c][j])
      for (int idx = tid; idx < MR * KP; idx += NTH) {
        const int c2 = idx % KP, i = idx / KP;
        const double2 v = Mg[(size_t)(row0 + i) * KP + c2];
        Ar[c2 * LDA + i] = v.x;
        Ai[c2 * LDA + i] = v.y;
      }
      for (int idx = tid; idx < MC * KP; idx += NTH) {
        const int j = idx % MC, c2 = idx / MC;
        const double2 v = Sg[(size_t)c2 * n + col0 + j];
        Br[c2 * LDB + j] = v.x;
        Bi[c2 * LDB + j] = v.y;
      }
      __syncthreads();
      mma_steps<TA, TB, 1, KP / 4>(cr, ci, Ar, Ai, LDA, arow, Br, Bi, LDB, bcol);
      const bool panel = col0 <= k0 && k0 < col0 + MC;  // the panel's columns take F = M + E
      if (!panel) {
#pragma unroll
        for (int ti = 0; ti < TA; ++ti)
#pragma unroll
          for (int tj = 0; tj < TB; ++tj)
#pragma unroll
            for (int r = 0; r < 4; ++r)
              stgb(W_ + (size_t)(row0 + ti * 16 + 4 * r) * n + col0 + tj * 16, t_off,
                   make_double2(cr[ti][tj][r], ci[ti][tj][r]));
      } else {
#pragma unroll
        for (int ti = 0; ti < TA; ++ti)
#pragma unroll
          for (int tj = 0; tj < TB; ++tj)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int il = arow + ti * 16 + 4 * r + kq;  // row within the tile
              const int j = col0 + bcol + tj * 16 + m;
              const bool inp = j >= k0 && j < k0 + KP;
              const int c2 = inp ? j - k0 : 0;
              double2 f = make_double2(Ar[c2 * LDA + il], Ai[c2 * LDA + il]);
              f.x += (piv[k0 + c2] == row0 + il) ? 1.0 : 0.0;
              const double2 v = inp ? f : make_double2(cr[ti][tj][r], ci[ti][tj][r]);
              stgb(W_ + (size_t)(row0 + ti * 16 + 4 * r) * n + col0 + tj * 16, t_off, v);
            }
      }
      __syncthreads();  // the staged panels are overwritten by the next tile
    }
  }
  if (info) {
    __syncthreads();
    for (int idx = tid; idx < n * n; idx += NTH) out[idx] = make_double2(0, 0);
    __syncthreads();
    return info;
  }
  for (int q = tid; q < n; q += NTH) used[piv[q]] = q;  // inverse permutation
  __syncthreads();
  // out(i, q) = W[piv[i]][used[q]], RB rows at a time staged through LDS
  constexpr int RB = L::RB;
  const int ldr = n + 1;
  ldsd* Lr = lds;
  ldsd* Li = lds + RB * ldr;
  for (int i0 = 0; i0 < n; i0 += RB) {
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
      const int j = tid + q * NTH;
      if (j < n) {
        double2 v[RB];
#pragma unroll
        for (int rr = 0; rr < RB; ++rr) v[rr] = W[(size_t)piv[i0 + rr] * n + j];
#pragma unroll
        for (int rr = 0; rr < RB; ++rr) {
          Lr[rr * ldr + j] = v[rr].x;
          Li[rr * ldr + j] = v[rr].y;
        }
      }
    }
    __syncthreads();
    for (int idx = tid; idx < RB * n; idx += NTH) {
      const int rr = idx % RB, q = idx / RB;
      const int c = used[q];
      out[(size_t)(i0 + rr) + (size_t)q * n] = make_double2(Lr[rr * ldr + c], Li[rr * ldr + c]);
    }
    __syncthreads();
  }
  return 0;
}

// ------------------------------------------------ inverse, n = 32 or 64
// The whole matrix held in registers and swept by gj_sweep: at N = 64 lane l of wave w
// holds row l of columns 16 w .. 16 w + 15, at N = 32 each half wave holds the 32 rows
// of 4 columns.  `store` false: only the result's info.  No global memory between the load of W and the store of the inverse.
template <int T, int N>
struct InvRegLds {
  static constexpr int HV = N == 32 ? 2 : 1;
  static constexpr int LDO = N + 1;           // odd row stride of the output staging tile
  static constexpr int XCH = GjLds<1, N * N / 256, HV>::DOUBLES;
  static constexpr int OUT = 2 * N * LDO;     // re / im planes of the matrix for the final copy
  static constexpr int AREA = XCH > OUT ? XCH : OUT;
  static constexpr int DOUBLES = AREA + N + 8;  // + piv, pinv (2 N ints)
};

template <int T, int N>
__device__ __noinline__ int wg_inverse_reg(double2* W_, double2* out_, ldsd* lds, bool store = true) {
  using L = InvRegLds<T, N>;
  constexpr int NTH = Cfg<T>::NTH, C = N * N / NTH, LDO = L::LDO;
  static_assert(NTH == 256 && (N == 32 || N == 64), "register inverse: 256 threads, N = 32 or 64");
  gd2* W = gw(W_);
  gd2* out = gw(out_);
  ldsi* piv = (ldsi*)(lds + L::AREA);
  ldsi* pinv = piv + N;
  const int tid = threadIdx.x;
  const int i = tid % N, cb = tid / N;
  double2 m[1][C];
  double2(&a)[C] = m[0];
#pragma unroll
  for (int c = 0; c < C; ++c) a[c] = W[(size_t)i * N + cb * C + c];
  unsigned used = 0;
  const int info = gj_sweep<1, C, L::HV>(m, N, used, piv, lds);
  if (info) {
    for (int idx = tid; store && idx < N * N; idx += NTH) out[idx] = make_double2(0, 0);
    __syncthreads();
    return info;
  }
  __syncthreads();  // the last column's exchange reads are done before the staging tile is written
  ldsd* Lr = lds;
  ldsd* Li = lds + N * LDO;
#pragma unroll
  for (int c = 0; c < C; ++c) {
    Lr[i * LDO + cb * C + c] = a[c].x;
    Li[i * LDO + cb * C + c] = a[c].y;
  }
  for (int q = tid; q < N; q += NTH) pinv[piv[q]] = q;
  __syncthreads();
  // out(r, q) = W[piv[r]][pinv[q]], r fastest across the lanes: coalesced column-major stores
  for (int idx = tid; store && idx < N * N; idx += NTH) {
    const int r = idx % N, q = idx / N;
    const int src = piv[r] * LDO + pinv[q];
    out[idx] = make_double2(Lr[src], Li[src]);
  }
  __syncthreads();
  return 0;
}

template <int T, int NMAX>
struct InvLds {
  static constexpr int DOUBLES = NMAX <= 64    ? InvRegLds<T, NMAX>::DOUBLES
                                 : NMAX <= 128 ? InvStripLds<128>::DOUBLES
                                 : NMAX <= 256 ? InvStripLds<NMAX>::DOUBLES
                                               : InvBigLds<T, NMAX>::DOUBLES;
};

// Inverse of an n x n block (n <= NMAX): the whole matrix in registers at 32 and 64, the
// panel in LDS up to 256 rows, the panels staged through `out` above that.
template <int T, int NMAX>
__device__ __forceinline__ int wg_inverse(int n, double2* W, double2* out, ldsd* lds) {
  if constexpr (NMAX == 32 || NMAX == 64) {
    return wg_inverse_reg<T, NMAX>(W, out, lds);  // these variants are chosen for n = NMAX only
  } else if constexpr (NMAX <= 128) {
    return wg_inverse_strip<128>(n, W, out, lds);
  } else if constexpr (NMAX <= 256) {
    if constexpr (NMAX == 256) {
      if (n <= 192) return wg_inverse_strip<192>(n, W, out, lds);  // no wave multiplies rows past 192
    }
    return wg_inverse_strip<NMAX>(n, W, out, lds);
  } else {
    return wg_inverse_big<T, NMAX>(n, W, out, lds);
  }
}

}  // namespace rgf
