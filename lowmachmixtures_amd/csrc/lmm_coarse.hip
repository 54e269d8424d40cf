// Coarse levels of a V-cycle in one launch.
//
// Below a few tens of thousands of points a multigrid level is far too small
// to fill the GPU: each colour sweep, residual, restriction and prolongation
// becomes a launch of a few microseconds that does almost no work, and a
// V-cycle over eight levels spends most of its time in such launches.  Here
// one workgroup of 1024 threads runs the whole coarse part of the V-cycle --
// down-leg smoothing, residual and restriction on every coarse level, the
// bottom smoothing, then prolongation and up-leg smoothing -- with a
// workgroup barrier between dependent passes.  Every point is computed with the
// arithmetic of the one-launch-per-pass kernels, in the same
// order of passes, so the result is bit for bit that of the separate launches
// (and of the reference's stag_mg_solver / F_MG level loops).  For
// visc_type -1 and 1 a face component's operator reads only that component,
// so the staggered V-cycle runs one workgroup per component side by side
// (the serial chain of barriers a third as long); the coupled viscosities
// keep all components in one workgroup.
#include "lmm_kernels.h"
#include "lmm_points.h"

namespace lmm {

namespace {

constexpr int CTPB = 1024;
const char kStagCoarseName[] = "k_stag_coarse_lds";
const char kCCCoarseName[] = "k_cc_coarse_lds";

template <typename T>
struct SLevelDesc {
  Grid g;
  Ptr3<T> phi, rhs, res;
  StagCoef<T> K;
};

// visc: -1 or 1
template <typename T>
struct SCoarseArgs {
  SLevelDesc<T> L[COARSE_MAX_LEVELS];
  int m;                 // coarse levels held in L[0..m-1], finest first
  int visc, nd, nu, nb;  // visc_type, sweeps down / up / bottom
  T omega;
};

template <typename T>
__device__ void blk_fill(T *x, long n, T v) {
  for (long t = threadIdx.x; t < n; t += CTPB) x[t] = v;
}

// the colour loop is unrolled for each dimension so that the component a of
// every colour is a constant after inlining (no per-lane stack for the
// per-component pointer tables)
template <typename T, int DIM>
__device__ void blk_stag_smooth_d(const SLevelDesc<T> &L, int visc, T omega, int nsweeps) {
  const long half = (long)(L.g.n[0] >> 1) * L.g.n[1] * L.g.n[2];
  const T dxsqinv = (T)(1.0 / (L.g.dx * L.g.dx));
  for (int m = 0; m < nsweeps; m++) {
#pragma unroll
    for (int color = 1; color <= 2 * DIM; color++) {
      const int a = (color - 1) / 2, par = (color + 1) % 2;
      for (long t = threadIdx.x; t < half; t += CTPB)
        gs_colour_at<T>(L.g, DIM, visc, a, par, omega, dxsqinv, L.phi, L.K, L.rhs.c[a], t);
      __syncthreads();
    }
  }
}

template <typename T>
__device__ void blk_stag_smooth(const SLevelDesc<T> &L, int visc, T omega, int nsweeps) {
  if (L.g.dim == 3) blk_stag_smooth_d<T, 3>(L, visc, omega, nsweeps);
  else blk_stag_smooth_d<T, 2>(L, visc, omega, nsweeps);
}

template <typename T>
__device__ void blk_prolong(const SLevelDesc<T> &F, const SLevelDesc<T> &C) {
  const long N = F.g.N;
  if (F.g.dim == 2) {
    for (long t = threadIdx.x; t < N; t += CTPB) prolong_at<T, 2, 0>(F.g, C.g, F.phi.c[0], C.phi.c[0], t);
    for (long t = threadIdx.x; t < N; t += CTPB) prolong_at<T, 2, 1>(F.g, C.g, F.phi.c[1], C.phi.c[1], t);
  } else {
    for (long t = threadIdx.x; t < N; t += CTPB) prolong_at<T, 3, 0>(F.g, C.g, F.phi.c[0], C.phi.c[0], t);
    for (long t = threadIdx.x; t < N; t += CTPB) prolong_at<T, 3, 1>(F.g, C.g, F.phi.c[1], C.phi.c[1], t);
    for (long t = threadIdx.x; t < N; t += CTPB) prolong_at<T, 3, 2>(F.g, C.g, F.phi.c[2], C.phi.c[2], t);
  }
  __syncthreads();
}

// The staggered coarse V-cycle passing every field through memory, all
// components in one workgroup (visc_type -1 / 1 with coarse_split = 0 only: the
// form that the LDS kernels below are compared with).
template <typename T>
__global__ void __launch_bounds__(CTPB) k_stag_coarse_vcycle(SCoarseArgs<T> A) {
  const int m = A.m, dim = A.L[0].g.dim;
  for (int n = 0; n < m; n++)
    for (int d = 0; d < dim; d++) blk_fill<T>(A.L[n].phi.c[d], A.L[n].g.N, (T)0);
  __syncthreads();
  for (int n = 0; n < m - 1; n++) {
    const SLevelDesc<T> &L = A.L[n];
    blk_stag_smooth<T>(L, A.visc, A.omega, A.nd);
    const T dxsqinv = (T)(1.0 / (L.g.dx * L.g.dx));
    for (int a = 0; a < dim; a++)
      for (long t = threadIdx.x; t < L.g.N; t += CTPB) residual_at<T>(L.g, dim, A.visc, dxsqinv, L.phi, L.rhs, L.res, L.K, a, t);
    __syncthreads();
    const SLevelDesc<T> &Cn = A.L[n + 1];
    for (int a = 0; a < dim; a++)
      for (long t = threadIdx.x; t < Cn.g.N; t += CTPB) restrict_at<T>(Cn.g, L.g, 0, L.res, Cn.rhs, a, t);
    __syncthreads();
  }
  blk_stag_smooth<T>(A.L[m - 1], A.visc, A.omega, A.nb);
  for (int n = m - 2; n >= 0; n--) {
    blk_prolong<T>(A.L[n], A.L[n + 1]);
    blk_stag_smooth<T>(A.L[n], A.visc, A.omega, A.nu);
  }
}

// ---------------------------------------------------------------------------
// The coarse V-cycle with every level's phi in LDS.
//
// The form above takes each point's operands from memory in every pass, so a
// pass of at most 4096 points costs a memory round trip and an index decode
// (about 2.4 us) however few points it has, and a V-cycle over 16^3 .. 2^3 has
// 44 (one component) to 130 (three) dependent passes.  Here the phi of all
// coarse levels, the right-hand sides below the first and one residual field
// stay in LDS (at most 159 KB: 16^3 and below, three components, FP64), and a
// thread keeps the operator coefficients, the right-hand side and the
// neighbour offsets of its own points (NQ x-pairs: one point of each colour
// per pair) in registers for all sweeps of a level visit: a pass reads LDS
// only, does the update and meets one barrier.  What bounds it now is
// instruction issue on the first level (one compute unit works; about 0.5 us
// a pass of 16^3) and the chain of LDS read, update and barrier below (0.2 us).
// Each point's arithmetic and the order of passes are those of the form
// above, so the bits are the same (div_by has the range).  visc_type 3 in 3D and
// FP64 spills 31 registers at two pairs a thread, the cell-centred kernel one.  A whole coarse part over 16^3 .. 2^3,
// before and after: staggered FP64 100 -> 31 us, visc_type 2 (one workgroup)
// 315 -> 86 us, cell-centred 73 -> 28 us.
// ---------------------------------------------------------------------------

constexpr int LDS_BYTES = 160 * 1024;

// One level as the LDS kernels see it: extents, the reciprocals that turn the
// index divisions into multiplications (indices below 2^16), and where its
// arrays lie in LDS (elements).
struct LvShape {
  int nx, ny, nz, N;
  unsigned mhx, mx, my;  // ceil(2^32 / (nx/2)), / nx, / ny; 0 stands for 2^32
  int phi, rhs;          // LDS offsets; rhs of the first level lies in memory
};

__host__ inline unsigned magic32(int d) { return (unsigned)(((1ull << 32) + d - 1) / d); }

__device__ __forceinline__ int mdiv(int t, unsigned m) { return m ? (int)__umulhi((unsigned)t, m) : t; }

struct Ijk {
  int i, j, k;
};
__device__ __forceinline__ Ijk cell_of(const LvShape &L, int t) {
  const int r = mdiv(t, L.mx), k = mdiv(r, L.my);
  return {t - r * L.nx, r - k * L.ny, k};
}
// x-pair t: its first point (i even)
__device__ __forceinline__ Ijk pair_of(const LvShape &L, int t) {
  const int hx = L.nx >> 1, r = mdiv(t, L.mhx), k = mdiv(r, L.my);
  return {2 * (t - r * hx), r - k * L.ny, k};
}

// Element offsets of the wrapped neighbour of c along direction d.
__device__ __forceinline__ int shift(const LvShape &L, const Ijk &c, int d, bool plus) {
  const int x = d == 0 ? c.i : (d == 1 ? c.j : c.k), n = d == 0 ? L.nx : (d == 1 ? L.ny : L.nz);
  const int s = d == 0 ? 1 : (d == 1 ? L.nx : L.nx * L.ny);
  return plus ? (x == n - 1 ? -x * s : s) : (x == 0 ? (n - 1) * s : -s);
}

// Where a point and its wrapped neighbours lie in one array of its level.
// Wide: byte offsets into LDS of the level's phi, one register each.
// Otherwise element offsets within an array, 16 bits each.
template <typename T, int DIM, bool WIDE>
struct Nbr;
template <typename T, int DIM>
struct Nbr<T, DIM, true> {
  int p, o[2 * DIM];
  __device__ __forceinline__ void set(const LvShape &L, const Ijk &c) {
    const int e = c.i + L.nx * c.j + L.nx * L.ny * c.k;
    p = (L.phi + e) * (int)sizeof(T);
#pragma unroll
    for (int d = 0; d < DIM; d++) {
      o[2 * d] = p + shift(L, c, d, true) * (int)sizeof(T);
      o[2 * d + 1] = p + shift(L, c, d, false) * (int)sizeof(T);
    }
  }
  __device__ __forceinline__ Nbr fresh() const { return *this; }
  __device__ __forceinline__ int self(int) const { return p; }
  __device__ __forceinline__ int at(int, int d, bool plus) const { return o[2 * d + (plus ? 0 : 1)]; }
  __device__ __forceinline__ int elem(const LvShape &L) const { return p / (int)sizeof(T) - L.phi; }
};
template <typename T, int DIM>
struct Nbr<T, DIM, false> {
  unsigned p, w[DIM];
  __device__ __forceinline__ void set(const LvShape &L, const Ijk &c) {
    p = (unsigned)(c.i + L.nx * c.j + L.nx * L.ny * c.k);
#pragma unroll
    for (int d = 0; d < DIM; d++)
      w[d] = (p + (unsigned)shift(L, c, d, true)) | ((p + (unsigned)shift(L, c, d, false)) << 16);
  }
  // an opaque copy: keeps the compiler from unpacking the offsets of every
  // point ahead of a sweep loop, which would take several registers each
  __device__ __forceinline__ Nbr fresh() const {
    Nbr n = *this;
    asm volatile("" : "+v"(n.p), "+v"(n.w[0]), "+v"(n.w[1]));
    if (DIM == 3) asm volatile("" : "+v"(n.w[DIM - 1]));
    return n;
  }
  __device__ __forceinline__ int elem(int d, bool plus) const { return (int)(plus ? (w[d] & 0xffffu) : (w[d] >> 16)); }
  // byte offsets for an array at element offset base
  __device__ __forceinline__ int self(int base) const { return ((int)p + base) * (int)sizeof(T); }
  __device__ __forceinline__ int at(int base, int d, bool plus) const { return (elem(d, plus) + base) * (int)sizeof(T); }
  __device__ __forceinline__ int elem(const LvShape &) const { return (int)p; }
};

// x / d with r = rcp_of(d) taken once for many divisions by the same d.
// FP32: the multiplication of gs_div.  FP64: q = x r and two corrections by
// the exact remainder; the first brings q within an ulp, and with r the
// correctly rounded reciprocal the second is then the correctly rounded
// quotient (Markstein, IBM J. Res. Dev. 34, 1990), the same bits as x / d in
// 5 operations instead of about 14 as long as the remainders and 1 / d are
// normal numbers, that is for |x| above about 1e-289 and |d| between 1e-307 and
// 1e307; below, the last bit may differ, and a quotient of -0 comes out as +0,
// which changes nothing where it is added.  A quotient that is not finite is x r.
__device__ __forceinline__ double rcp_of(double d) { return 1.0 / d; }
__device__ __forceinline__ float rcp_of(float d) { return __builtin_amdgcn_rcpf(d); }
__device__ __forceinline__ float div_by(float x, float, float r) { return x * r; }
__device__ __forceinline__ double div_by(double x, double d, double r) {
  const double q = x * r;
  const double q1 = __builtin_fma(__builtin_fma(-d, q, x), r, q);
  const double q2 = __builtin_fma(__builtin_fma(-d, q1, x), r, q1);
  return __builtin_isfinite(q) ? q2 : q;
}

template <typename T>
__device__ __forceinline__ T &lds(T *sm, int byte) {
  return *reinterpret_cast<T *>(reinterpret_cast<char *>(sm) + byte);
}

template <typename T>
struct SLdsLevel {
  LvShape s;
  StagCoef<T> K;
  T dxsqinv;
};

template <typename T>
struct SLdsArgs {
  SLdsLevel<T> L[COARSE_MAX_LEVELS];
  Ptr3<T> phi0, rhs0;  // first level: solution out, right-hand side in
  int m, nd, nu, nb, res;  // res: LDS offset of the residual field
  T omega;
};

// What a point of one component needs besides phi: the multiplier dl of phi
// in L phi, the diagonal fac of the update (stag_point forms both in their
// own order) with its reciprocal, and the coefficients of the neighbours.
template <typename T>
struct PtCoef {
  T dl, fac, rcp, b0, b1, e10, e11, e20, e21, g0, gm;
};

// dl, fac and rcp from alpha and the neighbours' coefficients, as stag_point
// forms them (lmm_common.h).  b, cg: beta[0], gamma[0].
template <typename T, int DIM, int VISC>
__device__ __forceinline__ void finish_coef(PtCoef<T> &c, T av, T b, T cg, T dxsqinv) {
  const T fourthirds = (T)(4.0 / 3.0), onethird = (T)(1.0 / 3.0);
  if (VISC == 1) {
    c.dl = c.fac = av + (T)(2.0 * DIM) * b * dxsqinv;
  } else if (VISC == 2) {
    c.dl = c.fac = av + (T)(2.0 * DIM + 2.0) * b * dxsqinv;
  } else if (VISC == 3) {
    c.dl = av + ((T)(6.0 * DIM + 2.0) * b * onethird + (T)2.0 * cg) * dxsqinv;
    c.fac = av + ((T)((6.0 * DIM + 2.0) / 3.0) * b + (T)2.0 * cg) * dxsqinv;
  } else {
    T d0, d1;
    if (VISC == -1) d0 = c.b0 + c.b1;
    else if (VISC == -2) d0 = (T)2.0 * c.b0 + (T)2.0 * c.b1;
    else d0 = fourthirds * c.b0 + c.g0 + fourthirds * c.b1 + c.gm;
    if (DIM == 3) {
      d0 = d0 + c.e10 + c.e11 + c.e20 + c.e21;
      d1 = d0;
    } else {
      d1 = d0 + c.e10 + c.e11;
      d0 = d0 + c.e11 + c.e10;
    }
    c.dl = av + d0 * dxsqinv;
    c.fac = av + d1 * dxsqinv;
  }
  c.rcp = rcp_of(c.fac);
}

// directions across component a (t2 unused in 2D)
__device__ __forceinline__ constexpr int tdir1(int dim, int a) { return dim == 2 ? 1 - a : (a == 0 ? 1 : 0); }
__device__ __forceinline__ constexpr int tdir2(int dim, int a) { return dim == 2 ? 2 : (a == 2 ? 1 : 2); }

// The values of array f at the points (c, c + x) of an x-pair shifted along
// direction d: one vector load, or for d = 0 one load beside the pair's own.
template <typename T>
__device__ __forceinline__ void pair_at(const LvShape &L, const T *f, const Ijk &c, int p, int d, bool plus, T &v0,
                                        T &v1) {
  if (d != 0) {
    ld2(f, p + shift(L, c, d, plus), v0, v1);
    return;
  }
  T a, b;
  ld2(f, p, a, b);
  if (plus) {
    v0 = b;
    v1 = f[c.i + 1 == L.nx - 1 ? p - c.i : p + 2];
  } else {
    v0 = f[c.i == 0 ? p + L.nx - 1 : p - 1];
    v1 = a;
  }
}

// Coefficients of both points of an x-pair for component a.
template <typename T, int DIM, int VISC>
__device__ __forceinline__ void pair_coef(const SLdsLevel<T> &L, int a, const Ijk &c, int p, T b, T cg, PtCoef<T> &k0,
                                          PtCoef<T> &k1) {
  T a0, a1;
  ld2(L.K.alpha[a], (long)p, a0, a1);
  if (VISC < 0) {
    const int t1 = tdir1(DIM, a), t2 = tdir2(DIM, a);
    ld2(L.K.beta, (long)p, k0.b0, k1.b0);
    pair_at(L.s, L.K.beta, c, p, a, false, k0.b1, k1.b1);
    const T *E1 = L.K.bed[DIM == 2 ? 0 : edge_of(a, t1)];
    ld2(E1, (long)p, k0.e10, k1.e10);
    pair_at(L.s, E1, c, p, t1, true, k0.e11, k1.e11);
    if (DIM == 3) {
      const T *E2 = L.K.bed[edge_of(a, t2)];
      ld2(E2, (long)p, k0.e20, k1.e20);
      pair_at(L.s, E2, c, p, t2, true, k0.e21, k1.e21);
    }
    if (VISC == -3) {
      ld2(L.K.gamma, (long)p, k0.g0, k1.g0);
      pair_at(L.s, L.K.gamma, c, p, a, false, k0.gm, k1.gm);
    }
  }
  finish_coef<T, DIM, VISC>(k0, a0, b, cg, L.dxsqinv);
  finish_coef<T, DIM, VISC>(k1, a1, b, cg, L.dxsqinv);
}

// (theta*alpha - L) phi at a point of component a from LDS; f, g1, g2: the
// element offsets of the component and of those of t1 / t2 (|VISC| > 1 only).
template <typename T, int DIM, int VISC, bool WIDE>
__device__ __forceinline__ T lds_apply(T *sm, const PtCoef<T> &c, int f, int g1, int g2, int a,
                                       const Nbr<T, DIM, WIDE> &n, T b, T cg, T dxsqinv) {
  const int t1 = tdir1(DIM, a), t2 = tdir2(DIM, a);
  auto F = [&](int d, bool plus) -> T { return lds(sm, n.at(f, d, plus)); };
  const T F0 = lds(sm, n.self(f));
  if (VISC == 1) {
    T s;
    if (DIM == 3) s = F(0, true) + F(0, false) + F(1, true) + F(1, false) + F(2, true) + F(2, false);
    else s = F(a, true) + F(a, false) + F(t1, true) + F(t1, false);
    return F0 * c.dl - s * b * dxsqinv;
  }
  const T Fa = F(a, true), Fma = F(a, false), F1p = F(t1, true), F1m = F(t1, false);
  const T F2p = DIM == 3 ? F(t2, true) : (T)0, F2m = DIM == 3 ? F(t2, false) : (T)0;
  if (VISC == -1) {
    T off = Fa * c.b0 + Fma * c.b1 + F1p * c.e11 + F1m * c.e10;
    if (DIM == 3) off = off + F2p * c.e21 + F2m * c.e20;
    return F0 * c.dl - off * dxsqinv;
  }
  // the corner neighbours (-a, +t): the two shifts are independent
  const int s1 = g1 * (int)sizeof(T), s2 = g2 * (int)sizeof(T);
  const int p = n.self(0), pm = n.at(0, a, false), p1 = n.at(0, t1, true);
  const T g1a = lds(sm, s1 + p1), g1b = lds(sm, s1 + p), g1c = lds(sm, s1 + pm + p1 - p), g1d = lds(sm, s1 + pm);
  T g2a = (T)0, g2b = (T)0, g2c = (T)0, g2d = (T)0;
  if (DIM == 3) {
    const int p2 = n.at(0, t2, true);
    g2a = lds(sm, s2 + p2);
    g2b = lds(sm, s2 + p);
    g2c = lds(sm, s2 + pm + p2 - p);
    g2d = lds(sm, s2 + pm);
  }
  const T fourthirds = (T)(4.0 / 3.0), onethird = (T)(1.0 / 3.0), twothirds = (T)(2.0 / 3.0);
  if (VISC == 2) {
    T s = (T)2.0 * Fa + (T)2.0 * Fma + F1p + F1m;
    if (DIM == 3) s = s + F2p + F2m;
    s = s + g1a - g1b - g1c + g1d;
    if (DIM == 3) s = s + g2a - g2b - g2c + g2d;
    return F0 * c.dl - s * b * dxsqinv;
  }
  if (VISC == 3) {
    T cr = g1a - g1b - g1c + g1d, tr = F1p + F1m;
    if (DIM == 3) {
      cr = cr + g2a - g2b - g2c + g2d;
      tr = tr + F2p + F2m;
    }
    return F0 * c.dl - ((Fa + Fma) * (fourthirds * b + cg) + tr * b + cr * (onethird * b + cg)) * dxsqinv;
  }
  if (VISC == -2) {
    T off = (T)2.0 * Fa * c.b0 + (T)2.0 * Fma * c.b1 + F1p * c.e11 + F1m * c.e10;
    if (DIM == 3) off = off + F2p * c.e21 + F2m * c.e20;
    off = off + g1a * c.e11 - g1b * c.e10 - g1c * c.e11 + g1d * c.e10;
    if (DIM == 3) off = off + g2a * c.e21 - g2b * c.e20 - g2c * c.e21 + g2d * c.e20;
    return F0 * c.dl - off * dxsqinv;
  }
  T off = Fa * (fourthirds * c.b0 + c.g0) + Fma * (fourthirds * c.b1 + c.gm) + F1p * c.e11 + F1m * c.e10;
  if (DIM == 3) off = off + F2p * c.e21 + F2m * c.e20;
  off = off + g1a * (c.e11 - twothirds * c.b0 + c.g0) - g1b * (c.e10 - twothirds * c.b0 + c.g0) -
        g1c * (c.e11 - twothirds * c.b1 + c.gm) + g1d * (c.e10 - twothirds * c.b1 + c.gm);
  if (DIM == 3)
    off = off + g2a * (c.e21 - twothirds * c.b0 + c.g0) - g2b * (c.e20 - twothirds * c.b0 + c.g0) -
          g2c * (c.e21 - twothirds * c.b1 + c.gm) + g2d * (c.e20 - twothirds * c.b1 + c.gm);
  return F0 * c.dl - off * dxsqinv;
}

// Coefficients of one point of component a (the variable coupled viscosities,
// whose coefficients do not fit in registers between passes).
template <typename T, int DIM, int VISC>
__device__ __forceinline__ PtCoef<T> pt_coef(const SLdsLevel<T> &L, int a, const Nbr<T, DIM, false> &n) {
  PtCoef<T> c = {};
  const int p = (int)n.p, t1 = tdir1(DIM, a), t2 = tdir2(DIM, a), pma = n.elem(a, false);
  const T *E1 = L.K.bed[DIM == 2 ? 0 : edge_of(a, t1)];
  c.b0 = L.K.beta[p];
  c.b1 = L.K.beta[pma];
  c.e10 = E1[p];
  c.e11 = E1[n.elem(t1, true)];
  if (DIM == 3) {
    const T *E2 = L.K.bed[edge_of(a, t2)];
    c.e20 = E2[p];
    c.e21 = E2[n.elem(t2, true)];
  }
  if (VISC == -3) {
    c.g0 = L.K.gamma[p];
    c.gm = L.K.gamma[pma];
  }
  finish_coef<T, DIM, VISC>(c, L.K.alpha[a][p], (T)0, (T)0, L.dxsqinv);
  return c;
}

// The LDS form for one viscosity type.  visc_type -1 / 1: a workgroup per
// component (A0); else one workgroup for all (A0 = -1).  NQ: x-pairs a thread
// owns on the first level.  The coefficients of visc_type -2 / -3 are loaded
// again in each pass.
template <typename T, int DIM, int VISC, int NQ, int A0>
__device__ __forceinline__ void stag_coarse_lds(const SLdsArgs<T> &A, T *sm) {
  constexpr bool SPLIT = A0 >= 0, CACHED = VISC >= -1;
  constexpr int NC = SPLIT ? 1 : DIM;
  // one component: the offsets have registers of their own, unless the
  // coefficients of four FP64 points fill them
  constexpr bool WIDE = SPLIT && !(VISC == -1 && DIM == 3 && NQ == 2 && sizeof(T) == 8);
  using NB = Nbr<T, DIM, WIDE>;
  const int tid = threadIdx.x, nth = blockDim.x;
  auto comp = [&](int c) { return SPLIT ? A0 : c; };

  NB nb[2][NQ];
  PtCoef<T> pc[CACHED ? NC : 1][2][NQ];
  T rh[NC][2][NQ];

  int tot = 0;
  for (int n = 0; n < A.m; n++) tot += NC * A.L[n].s.N;
  for (int t = tid; t < tot; t += nth) sm[t] = (T)0;  // phi of every level lies first
  // One loop over the level visits (down to the last level and up again), so
  // that each phase is in the code once.
  const int last = A.m - 1;
  for (int v = 0; v <= 2 * last; v++) {
    const int n = v <= last ? v : 2 * last - v;
    const SLdsLevel<T> &L = A.L[n];
    const LvShape &F = L.s, &Cs = A.L[n < last ? n + 1 : n].s;
    const int half = F.N >> 1, phi = F.phi, Nn = F.N;
    const T dxsqinv = L.dxsqinv;
    const T b = VISC > 0 ? L.K.beta[0] : (T)0, cg = VISC == 3 ? L.K.gamma[0] : (T)0;
    // (theta*alpha - L) phi at this thread's point (par, q) of component c
    auto value = [&](int c, int par, int q, const NB &x, PtCoef<T> &k) -> T {
      const int a = comp(c);
      if constexpr (CACHED) k = pc[c][par][q];
      else k = pt_coef<T, DIM, VISC>(L, a, x);
      return lds_apply<T, DIM, VISC, WIDE>(sm, k, phi + c * Nn, phi + tdir1(DIM, a) * Nn,
                                           phi + (DIM == 3 ? tdir2(DIM, a) : 0) * Nn, a, x, b, cg, dxsqinv);
    };
    // this thread's pairs: offsets, coefficients, right-hand sides, and on
    // the way up the prolongation of the correction (red point first)
#pragma unroll
    for (int q = 0; q < NQ; q++) {
      const int t = tid + nth * q;
      if (t >= half) continue;
      const Ijk c0 = pair_of(F, t), c1 = {c0.i + 1, c0.j, c0.k};
      const bool odd_row = ((c0.j + c0.k) & 1) != 0;  // the pair's second point is red
      const int p = c0.i + F.nx * c0.j + F.nx * F.ny * c0.k;
      nb[0][q].set(F, odd_row ? c1 : c0);
      nb[1][q].set(F, odd_row ? c0 : c1);
#pragma unroll
      for (int c = 0; c < NC; c++) {
        const int a = comp(c);
        if constexpr (CACHED) {
          PtCoef<T> k0 = {}, k1 = {};
          pair_coef<T, DIM, VISC>(L, a, c0, p, b, cg, k0, k1);
          pc[c][0][q] = odd_row ? k1 : k0;
          pc[c][1][q] = odd_row ? k0 : k1;
        }
        T r0, r1;
        if (n == 0) {
          ld2(A.rhs0.c[a], (long)p, r0, r1);
        } else {
          r0 = sm[F.rhs + c * Nn + p];
          r1 = sm[F.rhs + c * Nn + p + 1];
        }
        rh[c][0][q] = odd_row ? r1 : r0;
        rh[c][1][q] = odd_row ? r0 : r1;
      }
      if (v > last) {
        const Ijk Q = {c0.i >> 1, c0.j >> 1, c0.k >> 1};
        const int q0 = Q.i + Cs.nx * Q.j + Cs.nx * Cs.ny * Q.k;
#pragma unroll
        for (int h = 0; h < 2; h++) {
          auto odd = [&](int d) -> bool { return d == 0 ? h == 1 : ((d == 1 ? c0.j : c0.k) & 1) != 0; };
#pragma unroll
          for (int c = 0; c < NC; c++) {
            const int a = comp(c), t1 = tdir1(DIM, a), t2 = tdir2(DIM, a);
            const T *cp = sm + Cs.phi + c * Cs.N + q0;
            const int da = shift(Cs, Q, a, true), d1 = shift(Cs, Q, t1, odd(t1));
            const int d2 = DIM == 3 ? shift(Cs, Q, t2, odd(t2)) : 0;
            T *w = sm + phi + c * Nn + p + h;
            *w = prolong_sum<T, DIM>(*w, !odd(a), [&](bool sa, bool s1, bool s2) -> T {
              return cp[(sa ? da : 0) + (s1 ? d1 : 0) + (s2 ? d2 : 0)];
            });
          }
        }
      }
    }
    __syncthreads();
    const int ns = v < last ? A.nd : (v == last ? A.nb : A.nu);
    for (int s = 0; s < ns; s++) {
#pragma unroll
      for (int c = 0; c < NC; c++)
#pragma unroll
        for (int par = 0; par < 2; par++) {
#pragma unroll
          for (int q = 0; q < NQ; q++)
            if (tid + nth * q < half) {
              PtCoef<T> k;
              const NB x = nb[par][q].fresh();
              const T Lp = value(c, par, q, x, k);
              T &f = lds(sm, x.self(phi + c * Nn));
              f = f + div_by(A.omega * (rh[c][par][q] - Lp), k.fac, k.rcp);
            }
          __syncthreads();
        }
    }
    if (v >= last) continue;
    const int sy = F.nx, sz = F.nx * F.ny;
#pragma unroll
    for (int c = 0; c < NC; c++) {
      const int a = comp(c);
#pragma unroll
      for (int par = 0; par < 2; par++)
#pragma unroll
        for (int q = 0; q < NQ; q++)
          if (tid + nth * q < half) {
            PtCoef<T> k;
            const NB x = nb[par][q].fresh();
            const T Lp = value(c, par, q, x, k);
            sm[A.res + x.elem(F)] = rh[c][par][q] - Lp;
          }
      __syncthreads();
      // 6-point (2D) / 12-point (3D) weights of restrict_at, in its order
      for (int t = tid; t < Cs.N; t += nth) {
        const Ijk C = cell_of(Cs, t);
        const T *f = sm + A.res + 2 * C.i + sy * 2 * C.j + sz * 2 * C.k;
        const int t1 = tdir1(DIM, a), t2 = tdir2(DIM, a);
        const int sa = a == 0 ? 1 : (a == 1 ? sy : sz), s1 = t1 == 0 ? 1 : sy, s2 = t2 == 1 ? sy : sz;
        const int am = shift(F, {2 * C.i, 2 * C.j, 2 * C.k}, a, false);
        T w;
        if (DIM == 2) {
          w = (T)0.25 * (f[0] + f[s1]) + (T)0.125 * (f[sa] + f[sa + s1] + f[am] + f[am + s1]);
        } else {
          const T v0 = f[0] + f[s1] + f[s2] + f[s1 + s2];
          const T vp = f[sa] + f[sa + s1] + f[sa + s2] + f[sa + s1 + s2];
          const T vm = f[am] + f[am + s1] + f[am + s2] + f[am + s1 + s2];
          w = (T)0.125 * v0 + (T)0.0625 * vp + (T)0.0625 * vm;
        }
        sm[Cs.rhs + c * Cs.N + t] = w;
      }
      __syncthreads();
    }
  }
  const int N0 = A.L[0].s.N;
#pragma unroll
  for (int c = 0; c < NC; c++)
    for (int t = tid; t < N0; t += nth) A.phi0.c[comp(c)][t] = sm[A.L[0].s.phi + c * N0 + t];
}

template <typename T, int DIM, int VISC, int NQ>
__global__ void __launch_bounds__(CTPB) k_stag_coarse_lds(SLdsArgs<T> A) {
  __shared__ T sm[LDS_BYTES / sizeof(T)];
  if constexpr (VISC == -1 || VISC == 1) {
    if (blockIdx.x == 0) stag_coarse_lds<T, DIM, VISC, NQ, 0>(A, sm);
    else if (DIM == 2 || blockIdx.x == 1) stag_coarse_lds<T, DIM, VISC, NQ, 1>(A, sm);
    else stag_coarse_lds<T, DIM, VISC, NQ, DIM == 3 ? 2 : 1>(A, sm);
  } else {
    stag_coarse_lds<T, DIM, VISC, NQ, -1>(A, sm);
  }
}

template <typename T>
struct CLdsLevel {
  LvShape s;
  Ptr3<T> a;
  T inv;
};
template <typename T>
struct CLdsArgs {
  CLdsLevel<T> L[COARSE_MAX_LEVELS];
  T *phi0;
  const T *rhs0;
  int m, nd, nu, nb, res;
};

// The cell-centred coarse V-cycle in LDS, as the staggered one.
template <typename T, int DIM, int NQ>
__global__ void __launch_bounds__(CTPB) k_cc_coarse_lds(CLdsArgs<T> A) {
  __shared__ T sm[LDS_BYTES / sizeof(T)];
  const int tid = threadIdx.x, nth = blockDim.x;
  // ten FP64 values for each of four points leave no room for wide offsets
  constexpr bool WIDE = NQ == 1 || sizeof(T) == 4;
  using NB = Nbr<T, DIM, WIDE>;
  struct Pc {
    T rhs, s, diag, rcp, l[DIM], h[DIM];
  };
  NB nb[2][NQ];
  Pc pc[2][NQ];
  int tot = 0;
  for (int n = 0; n < A.m; n++) tot += A.L[n].s.N;
  for (int t = tid; t < tot; t += nth) sm[t] = (T)0;
  const int last = A.m - 1;
  for (int v = 0; v <= 2 * last; v++) {
    const int n = v <= last ? v : 2 * last - v;
    const CLdsLevel<T> &L = A.L[n];
    const LvShape &F = L.s, &Cs = A.L[n < last ? n + 1 : n].s;
    const int half = F.N >> 1, phi = F.phi;
    const T inv = L.inv;
    // L phi at a point, as cc_apply forms it
    auto value = [&](const Pc &c, const NB &x) -> T {
      auto f = [&](int d, bool plus) -> T { return lds(sm, x.at(phi, d, plus)); };
      T off = c.l[0] * f(0, false) + c.h[0] * f(0, true) + c.l[1] * f(1, false) + c.h[1] * f(1, true);
      if (DIM == 3) off = off + c.l[DIM - 1] * f(DIM - 1, false) + c.h[DIM - 1] * f(DIM - 1, true);
      return (-c.s * lds(sm, x.self(phi)) + off) * inv;
    };
#pragma unroll
    for (int q = 0; q < NQ; q++) {
      const int t = tid + nth * q;
      if (t >= half) continue;
      const Ijk c0 = pair_of(F, t), c1 = {c0.i + 1, c0.j, c0.k};
      const bool odd_row = ((c0.j + c0.k) & 1) != 0;
      const int p = c0.i + F.nx * c0.j + F.nx * F.ny * c0.k;
      nb[0][q].set(F, odd_row ? c1 : c0);
      nb[1][q].set(F, odd_row ? c0 : c1);
      Pc k0 = {}, k1 = {};
#pragma unroll
      for (int d = 0; d < DIM; d++) {
        ld2(L.a.c[d], (long)p, k0.l[d], k1.l[d]);
        pair_at(F, L.a.c[d], c0, p, d, true, k0.h[d], k1.h[d]);
      }
      if (n == 0) {
        ld2(A.rhs0, (long)p, k0.rhs, k1.rhs);
      } else {
        k0.rhs = sm[F.rhs + p];
        k1.rhs = sm[F.rhs + p + 1];
      }
      auto finish = [&](Pc &k) {
        k.s = k.l[0] + k.h[0] + k.l[1] + k.h[1];
        if (DIM == 3) k.s = k.s + k.l[DIM - 1] + k.h[DIM - 1];
        k.diag = -k.s * inv;
        k.rcp = rcp_of(k.diag);
      };
      finish(k0);
      finish(k1);
      pc[0][q] = odd_row ? k1 : k0;
      pc[1][q] = odd_row ? k0 : k1;
      if (v > last) {
        const T e = sm[Cs.phi + (c0.i >> 1) + Cs.nx * (c0.j >> 1) + Cs.nx * Cs.ny * (c0.k >> 1)];
        sm[phi + p] = sm[phi + p] + e;
        sm[phi + p + 1] = sm[phi + p + 1] + e;
      }
    }
    __syncthreads();
    const int ns = v < last ? A.nd : (v == last ? A.nb : A.nu);
    for (int s = 0; s < ns; s++)
#pragma unroll
      for (int par = 0; par < 2; par++) {
#pragma unroll
        for (int q = 0; q < NQ; q++)
          if (tid + nth * q < half) {
            const NB x = nb[par][q].fresh();
            const Pc &c = pc[par][q];
            const T lp = value(c, x);
            T &f = lds(sm, x.self(phi));
            f = f + div_by(c.rhs - lp, c.diag, c.rcp);
          }
        __syncthreads();
      }
    if (v >= last) continue;
    const int sy = F.nx, sz = F.nx * F.ny;
#pragma unroll
    for (int par = 0; par < 2; par++)
#pragma unroll
      for (int q = 0; q < NQ; q++)
        if (tid + nth * q < half) {
          const NB x = nb[par][q].fresh();
          sm[A.res + x.elem(F)] = pc[par][q].rhs - value(pc[par][q], x);
        }
    __syncthreads();
    for (int t = tid; t < Cs.N; t += nth) {
      const Ijk C = cell_of(Cs, t);
      const T *f = sm + A.res + 2 * C.i + sy * 2 * C.j + sz * 2 * C.k;
      T w = f[0] + f[1] + f[sy] + f[1 + sy];
      if (DIM == 3) w = w + f[sz] + f[1 + sz] + f[sy + sz] + f[1 + sy + sz];
      sm[Cs.rhs + t] = (T)(DIM == 3 ? 0.125 : 0.25) * w;
    }
    __syncthreads();
  }
  for (int t = tid; t < A.L[0].s.N; t += nth) A.phi0[t] = sm[A.L[0].s.phi + t];
}

// Shapes and LDS offsets of levels lv[0..m-1] with nc components each: phi of
// every level, the right-hand sides below the first, one residual field of
// the first level's size.  Levels of at most COARSE_MAX_CELLS = 4096 cells and
// even extents always fit: the largest need is 16^3's, 159104 bytes with three
// FP64 components.  false: a level past that (also past the kernels' 16-bit
// offsets, colouring or two pairs a thread).
template <typename T, typename LV, typename OUT>
bool lds_plan(int m, const LV *lv, int nc, OUT *L, int &res) {
  long off = 0;
  for (int n = 0; n < m; n++) {
    const Grid &g = lv[n].g;
    LvShape &s = L[n].s;
    if (g.N > COARSE_MAX_CELLS || g.n[0] % 2 != 0) return false;
    s.nx = g.n[0];
    s.ny = g.n[1];
    s.nz = g.n[2];
    s.N = (int)g.N;
    s.mhx = magic32(s.nx / 2);
    s.mx = magic32(s.nx);
    s.my = magic32(s.ny);
    s.phi = (int)off;
    s.rhs = 0;
    off += (long)nc * g.N;
  }
  for (int n = 1; n < m; n++) {
    L[n].s.rhs = (int)off;
    off += (long)nc * L[n].s.N;
  }
  res = (int)off;
  if (m > 1) off += L[0].s.N;
  static_assert(COARSE_MAX_CELLS <= 4 * CTPB, "two pairs a thread");
  return off * (long)sizeof(T) <= LDS_BYTES;
}

// threads for `half` colour points at nq points a thread: whole waves
inline int lds_threads(int half, int nq) {
  const int t = ((half + nq - 1) / nq + 63) / 64 * 64;
  return t > CTPB ? CTPB : t;
}

template <typename T, int DIM, int VISC>
void launch_stag_lds(hipStream_t s, int m, const CoarseStagLevel<T> *lv, T omega, int nd, int nu, int nb) {
  constexpr int NC = (VISC == -1 || VISC == 1) ? 1 : DIM;
  SLdsArgs<T> A;
  if (!lds_plan<T>(m, lv, NC, A.L, A.res)) {
    report_error("launch_stag_coarse_vcycle: the levels do not fit LDS");
    return;
  }
  const int half = (int)(lv[0].g.N / 2), nq = half > CTPB ? 2 : 1;
  for (int n = 0; n < m; n++) {
    A.L[n].K = lv[n].K;
    A.L[n].dxsqinv = (T)(1.0 / (lv[n].g.dx * lv[n].g.dx));
  }
  A.phi0 = p3(lv[0].phi);
  A.rhs0 = p3(lv[0].rhs);
  A.m = m;
  A.nd = nd;
  A.nu = nu;
  A.nb = nb;
  A.omega = omega;
  const dim3 grid(NC == 1 ? DIM : 1), block(lds_threads(half, nq));
  if (nq == 1) hipLaunchKernelGGL((k_stag_coarse_lds<T, DIM, VISC, 1>), grid, block, 0, s, A);
  else hipLaunchKernelGGL((k_stag_coarse_lds<T, DIM, VISC, 2>), grid, block, 0, s, A);
  post_launch(s, kStagCoarseName);
}

template <typename T, int DIM>
void launch_stag_lds_visc(hipStream_t s, int m, const CoarseStagLevel<T> *lv, int visc, T omega, int nd, int nu,
                          int nb) {
  switch (visc) {
    case -1: launch_stag_lds<T, DIM, -1>(s, m, lv, omega, nd, nu, nb); break;
    case 1: launch_stag_lds<T, DIM, 1>(s, m, lv, omega, nd, nu, nb); break;
    case 2: launch_stag_lds<T, DIM, 2>(s, m, lv, omega, nd, nu, nb); break;
    case 3: launch_stag_lds<T, DIM, 3>(s, m, lv, omega, nd, nu, nb); break;
    case -2: launch_stag_lds<T, DIM, -2>(s, m, lv, omega, nd, nu, nb); break;
    default: launch_stag_lds<T, DIM, -3>(s, m, lv, omega, nd, nu, nb); break;
  }
}

template <typename T, int DIM>
void launch_cc_lds(hipStream_t s, int m, const CoarseCCLevel<T> *lv, int nd, int nu, int nb) {
  CLdsArgs<T> A;
  if (!lds_plan<T>(m, lv, 1, A.L, A.res)) {
    report_error("launch_cc_coarse_vcycle: the levels do not fit LDS");
    return;
  }
  const int half = (int)(lv[0].g.N / 2), nq = half > CTPB ? 2 : 1;
  for (int n = 0; n < m; n++) {
    A.L[n].a = p3(lv[n].a);
    A.L[n].inv = (T)(1.0 / (lv[n].g.dx * lv[n].g.dx));
  }
  A.phi0 = lv[0].phi;
  A.rhs0 = lv[0].rhs;
  A.m = m;
  A.nd = nd;
  A.nu = nu;
  A.nb = nb;
  const dim3 block(lds_threads(half, nq));
  if (nq == 1) hipLaunchKernelGGL((k_cc_coarse_lds<T, DIM, 1>), dim3(1), block, 0, s, A);
  else hipLaunchKernelGGL((k_cc_coarse_lds<T, DIM, 2>), dim3(1), block, 0, s, A);
  post_launch(s, kCCCoarseName);
}

}  // namespace

template <typename T>
void launch_stag_coarse_vcycle(hipStream_t s, int m, const CoarseStagLevel<T> *lv, int visc, T omega, int nd,
                               int nu, int nb) {
  // the LDS form was the faster one at every size measured, 4 to 4096 cells;
  // coarse_split = 0 asks for visc_type -1 / 1 in one workgroup
  if (tuning().coarse_split || (visc != -1 && visc != 1)) {
    if (lv[0].g.dim == 3) launch_stag_lds_visc<T, 3>(s, m, lv, visc, omega, nd, nu, nb);
    else launch_stag_lds_visc<T, 2>(s, m, lv, visc, omega, nd, nu, nb);
    return;
  }
  SCoarseArgs<T> A;
  A.m = m;
  A.visc = visc;
  A.nd = nd;
  A.nu = nu;
  A.nb = nb;
  A.omega = omega;
  for (int n = 0; n < m; n++) {
    A.L[n].g = lv[n].g;
    A.L[n].phi = p3(lv[n].phi);
    A.L[n].rhs = p3(lv[n].rhs);
    A.L[n].res = p3(lv[n].res);
    A.L[n].K = lv[n].K;
  }
  hipLaunchKernelGGL(k_stag_coarse_vcycle<T>, dim3(1), dim3(CTPB), 0, s, A);
  post_launch(s, "k_stag_coarse_vcycle");
}

template <typename T>
void launch_cc_coarse_vcycle(hipStream_t s, int m, const CoarseCCLevel<T> *lv, int nd, int nu, int nb) {
  if (lv[0].g.dim == 3) launch_cc_lds<T, 3>(s, m, lv, nd, nu, nb);
  else launch_cc_lds<T, 2>(s, m, lv, nd, nu, nb);
}

template void launch_stag_coarse_vcycle<double>(hipStream_t, int, const CoarseStagLevel<double> *, int, double,
                                                int, int, int);
template void launch_stag_coarse_vcycle<float>(hipStream_t, int, const CoarseStagLevel<float> *, int, float, int,
                                               int, int);
template void launch_cc_coarse_vcycle<double>(hipStream_t, int, const CoarseCCLevel<double> *, int, int, int);
template void launch_cc_coarse_vcycle<float>(hipStream_t, int, const CoarseCCLevel<float> *, int, int, int);

}  // namespace lmm
