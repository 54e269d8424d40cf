// Species mass-flux chain on gfx950 (declarations and layout in
// lmm_species.h).
//
// Every per-cell routine is a template on the species count NS (2..8; the
// face fluxes also take 1) so that the small dense matrices live in VGPRs
// with static indices.  The arithmetic follows the reference routine by
// routine, operation by operation (sums from 0.0 in ascending index order,
// the same association of products and quotients), so the FP64 results
// equal the CPU restatement bit for bit:
//   correct_rho_with_drho_local   mass_flux_utilities.f90:127-150
//   compute_molconc_rhotot_local  :279-313
//   mixture_properties_mass_local compute_mixture_properties.f90:165-233
//   compute_Gama_local            mass_flux_utilities.f90:562-599
//   compute_chi_local             :767-831 (+ Dbar2chi_iterative,
//                                 matrix_utilities.f90:21-156, or the
//                                 use_lapack form :833-927)
//   compute_rhoWchi_local         :1250-1273
//   compute_Lonsager_local        :1068-1118 (+ choldc, matrix_utilities.f90:160-239)
//   compute_baro_coef_2d          :1342-1369
//   diffusive_mass_flux           diffusive_mass_fluxdiv.f90:92-262
//   stochastic_mass_fluxdiv       stochastic_mass_fluxdiv.f90:32-154
//   correction_flux               correction_flux.f90:71-251
//
// Dbar2chi_iterative updates chi column by column: column j of iteration
// k+1 depends only on column j of iteration k, so running all iterations on
// one column before the next gives the same operations on every entry while
// holding one column instead of three matrices.
//
// compute_mass_fluxdiv.f90 runs as one cell pass (sp_chain_cell), which
// writes only what the faces need (mole fractions, rho W chi, Gama unless
// the mixture is ideal, zeta/T, the packed lower triangle of the Cholesky
// factor of L-Onsager) and restores rho, then one face pass computing both
// fluxes of every face (flux_total written once) and one pass for both
// divergences (sp_chain_face).  Giving each cell
// its upper faces too (recomputed, so the face arrays need not be stored)
// was tried: the two matrix-vector chains per face kept so many loads live
// that the kernel ran at one wave per SIMD with spills from 5 species up.
#include "lmm.h"
#include "lmm_kernels.h"
#include "lmm_points.h"
#include "lmm_species.h"

namespace lmm {
namespace {

constexpr int STPB = 256;

#define SLAUNCH(K, G, B, SHM, S, ...)                   \
  do {                                                  \
    hipLaunchKernelGGL(K, G, B, SHM, S, __VA_ARGS__);   \
    post_launch(S, #K);                                 \
  } while (0)

inline int sblk(long n) { return (int)((n + STPB - 1) / STPB); }

// strict lower triangle index of (r, c), r > c, in the Dbar / H_offdiag order
__host__ __device__ __forceinline__ int tri(int r, int c) { return r * (r - 1) / 2 + c; }
// packed lower triangle by columns: (r, c), r >= c
template <int NS>
__host__ __device__ __forceinline__ int lpk_index(int r, int c) {
  return c * NS - c * (c - 1) / 2 + (r - c);
}

// D_bar(i, j) from the constant knobs (mixture_properties_mass_local)
struct DParam {
  const SpParams &sp;
  __device__ double operator()(int i, int j) const {
    return i == j ? 0.0 : sp.Dbar[i > j ? tri(i, j) : tri(j, i)];
  }
};
// D_bar(i, j) from a field of ns*ns components
template <int NS>
struct DField {
  const double *p;
  long N, t;
  __device__ double operator()(int i, int j) const { return p[(long)(i + NS * j) * N + t]; }
};

template <int NS>
__device__ __forceinline__ void load(const double *f, long N, long t, double (&v)[NS]) {
#pragma unroll
  for (int q = 0; q < NS; q++) v[q] = f[(long)q * N + t];
}

template <int NS>
__device__ __forceinline__ void cell_correct(const SpParams &sp, double (&rho)[NS], double (&drho)[NS]) {
  double old[NS], tot = 0.0;
#pragma unroll
  for (int n = 0; n < NS; n++) {
    old[n] = rho[n];
    tot = tot + rho[n];
  }
  const double f = sp.ftol * tot;
#pragma unroll
  for (int n = 0; n < NS; n++) rho[n] = rho[n] > f ? rho[n] : f;
#pragma unroll
  for (int n = 0; n < NS; n++) drho[n] = rho[n] - old[n];
}

template <int NS>
__device__ __forceinline__ void cell_prim(const SpParams &sp, const double (&rho)[NS], double &tot,
                                          double (&x)[NS], double &mt) {
  tot = 0.0;
#pragma unroll
  for (int n = 0; n < NS; n++) tot = tot + rho[n];
  double W[NS], s = 0.0;
#pragma unroll
  for (int n = 0; n < NS; n++) {
    W[n] = rho[n] / tot;
    s = s + W[n] / sp.molmass[n];
  }
  mt = 1.0 / s;
#pragma unroll
  for (int n = 0; n < NS; n++) x[n] = mt * W[n] / sp.molmass[n];
}

// Gama(r, c) = delta_rc + sum_k X(r, k) H(k, c), X = diag(x) - x x^T
// (zero for an ideal mixture); H(k, c) from the callable.
template <int NS, class HF>
__device__ __forceinline__ double gama_entry(const SpParams &sp, const double (&x)[NS], int r, int c, HF H) {
  double acc = 0.0;
#pragma unroll
  for (int k = 0; k < NS; k++) {
    double X = 0.0;
    if (!sp.ideal) X = (k == r) ? x[r] - x[r] * x[r] : -(x[r] * x[k]);
    acc = acc + X * H(k, c);
  }
  return (r == c ? 1.0 : 0.0) + acc;
}

// Lambda(r, c), r != c, of compute_chi_local: the value set at (max, min)
template <int NS, class DF>
__device__ __forceinline__ double lambda_off(const double (&x)[NS], int r, int c, DF D) {
  const int hi = r > c ? r : c, lo = r > c ? c : r;
  return -(x[hi] * x[lo] / D(hi, lo));
}

// zeta_by_Temp of compute_chi_local (non-isothermal)
template <int NS, class DF>
__device__ __forceinline__ void cell_zeta(const double (&x)[NS], DF D, const double (&Dt)[NS], double T,
                                          double (&z)[NS]) {
#pragma unroll
  for (int r = 0; r < NS; r++) {
    double s = 0.0;
#pragma unroll
    for (int c = 0; c < NS; c++)
      if (c != r) s = s + lambda_off<NS>(x, r, c, D) * (Dt[r] - Dt[c]);
    z[r] = s / T;
  }
}

// Dbar2chi_iterative: hands each finished column j of chi to col(j, v).
template <int NS, class DF, class COL>
__device__ __forceinline__ void chi_iterative(const SpParams &sp, const double (&X)[NS], DF D, COL col) {
  double MW = 0.0, Y[NS], Mm[NS], Mi[NS], t1[NS];
#pragma unroll
  for (int i = 0; i < NS; i++) MW = MW + X[i] * sp.molmass[i];
#pragma unroll
  for (int i = 0; i < NS; i++) Y[i] = sp.molmass[i] / MW * X[i];
#pragma unroll
  for (int i = 0; i < NS; i++) {
    double t2 = 0.0;
#pragma unroll
    for (int j = 0; j < NS; j++)
      if (j != i) t2 = t2 + X[j] / D(i, j);
    const double Di = (1.0 - Y[i]) / t2;
    Mm[i] = X[i] / Di;
    Mi[i] = Di / X[i];
  }
#pragma unroll
  for (int i = 0; i < NS; i++) {
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < NS; k++)
      if (k != i) s = s + X[i] * X[k] / D(i, k);
    t1[i] = s;
  }
  auto P = [&](int i, int j) { return (i == j) ? -Y[j] + 1.0 : -Y[j]; };
  // Z = -Delta + diag(Mm); J = diag(Mi) Z; PJ = P J
  double PJ[NS * NS];
#pragma unroll
  for (int i = 0; i < NS; i++)
#pragma unroll
    for (int j = 0; j < NS; j++) {
      double acc = 0.0;
#pragma unroll
      for (int k = 0; k < NS; k++) {
        const double Z = (k == j) ? -t1[k] + Mm[k] : -(-(X[k] * X[j] / D(k, j)));
        acc = acc + P(i, k) * (Mi[k] * Z);
      }
      PJ[i + NS * j] = acc;
    }
#pragma unroll
  for (int j = 0; j < NS; j++) {
    double m2[NS], c[NS];
#pragma unroll
    for (int i = 0; i < NS; i++) {
      double scr = 0.0;
#pragma unroll
      for (int k = 0; k < NS; k++) scr = scr + P(i, k) * Mi[k] * P(j, k);
      m2[i] = scr;
      c[i] = scr;
    }
    for (int it = 0; it < sp.chi_iter; it++) {
      double nc[NS];
#pragma unroll
      for (int i = 0; i < NS; i++) {
        double scr = 0.0;
#pragma unroll
        for (int k = 0; k < NS; k++) scr = scr + PJ[i + NS * k] * c[k];
        nc[i] = scr + m2[i];
      }
#pragma unroll
      for (int i = 0; i < NS; i++) c[i] = nc[i];
    }
    col(j, c);
  }
}

// Gauss-Jordan inverse with partial pivoting (the result of LAPACK
// dgetrf + dgetri); row exchanges by static-index selects.
template <int NS>
__device__ __forceinline__ void invert(double (&A)[NS * NS]) {
  double B[NS * NS];
#pragma unroll
  for (int r = 0; r < NS; r++)
#pragma unroll
    for (int c = 0; c < NS; c++) B[r + NS * c] = (r == c) ? 1.0 : 0.0;
#pragma unroll
  for (int c = 0; c < NS; c++) {
    int p = c;
    double best = fabs(A[c + NS * c]);
#pragma unroll
    for (int r = c + 1; r < NS; r++)
      if (fabs(A[r + NS * c]) > best) {
        best = fabs(A[r + NS * c]);
        p = r;
      }
#pragma unroll
    for (int r = c + 1; r < NS; r++)
      if (r == p)
#pragma unroll
        for (int k = 0; k < NS; k++) {
          double t = A[c + NS * k];
          A[c + NS * k] = A[r + NS * k];
          A[r + NS * k] = t;
          t = B[c + NS * k];
          B[c + NS * k] = B[r + NS * k];
          B[r + NS * k] = t;
        }
    const double inv = 1.0 / A[c + NS * c];
#pragma unroll
    for (int k = 0; k < NS; k++) {
      A[c + NS * k] = A[c + NS * k] * inv;
      B[c + NS * k] = B[c + NS * k] * inv;
    }
#pragma unroll
    for (int r = 0; r < NS; r++) {
      if (r == c) continue;
      const double f = A[r + NS * c];
      if (f == 0.0) continue;
#pragma unroll
      for (int k = 0; k < NS; k++) {
        A[r + NS * k] = A[r + NS * k] - f * A[c + NS * k];
        B[r + NS * k] = B[r + NS * k] - f * B[c + NS * k];
      }
    }
  }
#pragma unroll
  for (int k = 0; k < NS * NS; k++) A[k] = B[k];
}

// Pseudo-inverse V diag(1/S) U^T by one-sided Jacobi (Hestenes), singular
// values at or below tol * sum(S) dropped (mass_flux_utilities.f90:905-915).
template <int NS>
__device__ __forceinline__ void pinv(const double (&A0)[NS * NS], double tol, double (&out)[NS * NS]) {
  double U[NS * NS], V[NS * NS];
#pragma unroll
  for (int k = 0; k < NS * NS; k++) U[k] = A0[k];
#pragma unroll
  for (int r = 0; r < NS; r++)
#pragma unroll
    for (int c = 0; c < NS; c++) V[r + NS * c] = (r == c) ? 1.0 : 0.0;
  for (int sweep = 0; sweep < 60; sweep++) {
    double off = 0.0;
#pragma unroll
    for (int p = 0; p < NS - 1; p++)
#pragma unroll
      for (int q = p + 1; q < NS; q++) {
        double a = 0.0, b = 0.0, g = 0.0;
#pragma unroll
        for (int k = 0; k < NS; k++) {
          a = a + U[k + NS * p] * U[k + NS * p];
          b = b + U[k + NS * q] * U[k + NS * q];
          g = g + U[k + NS * p] * U[k + NS * q];
        }
        if (g == 0.0) continue;
        const double rel = fabs(g) / sqrt(a * b);
        if (rel > off) off = rel;
        if (rel < 1e-15) continue;
        const double zeta = (b - a) / (2.0 * g);
        const double t = (zeta >= 0.0 ? 1.0 : -1.0) / (fabs(zeta) + sqrt(1.0 + zeta * zeta));
        const double cs = 1.0 / sqrt(1.0 + t * t), sn = cs * t;
#pragma unroll
        for (int k = 0; k < NS; k++) {
          const double up = U[k + NS * p], uq = U[k + NS * q];
          U[k + NS * p] = cs * up - sn * uq;
          U[k + NS * q] = sn * up + cs * uq;
          const double vp = V[k + NS * p], vq = V[k + NS * q];
          V[k + NS * p] = cs * vp - sn * vq;
          V[k + NS * q] = sn * vp + cs * vq;
        }
      }
    if (off < 1e-15) break;
  }
  double S[NS], ssum = 0.0;
#pragma unroll
  for (int c = 0; c < NS; c++) {
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < NS; k++) s = s + U[k + NS * c] * U[k + NS * c];
    S[c] = sqrt(s);
    ssum = ssum + S[c];
  }
#pragma unroll
  for (int k = 0; k < NS * NS; k++) out[k] = 0.0;
#pragma unroll
  for (int c = 0; c < NS; c++) {
    if (!(S[c] > tol * ssum)) continue;
    const double w = 1.0 / (S[c] * S[c]);
#pragma unroll
    for (int i = 0; i < NS; i++)
#pragma unroll
      for (int j = 0; j < NS; j++) out[i + NS * j] = out[i + NS * j] + V[i + NS * c] * w * U[j + NS * c];
  }
}

// compute_chi_lapack: hands the columns of chi to col(j, v).
template <int NS, class DF, class COL>
__device__ __forceinline__ void chi_lapack(const SpParams &sp, const double (&x)[NS], const double (&W)[NS], DF D,
                                           COL col) {
  double Lam[NS * NS];
#pragma unroll
  for (int r = 0; r < NS; r++)
#pragma unroll
    for (int c = 0; c < NS; c++) Lam[r + NS * c] = (r == c) ? 0.0 : lambda_off<NS>(x, r, c, D);
#pragma unroll
  for (int r = 0; r < NS; r++) {
    double s = 0.0;
#pragma unroll
    for (int c = 0; c < NS; c++)
      if (c != r) s = s - Lam[r + NS * c];
    Lam[r + NS * r] = s;
  }
  double alpha = 0.0;
#pragma unroll
  for (int r = 0; r < NS; r++) alpha = alpha + Lam[r + NS * r];
  double A[NS * NS];
#pragma unroll
  for (int r = 0; r < NS; r++)
#pragma unroll
    for (int c = 0; c < NS; c++) A[r + NS * c] = alpha * W[r] * W[c] + Lam[r + NS * c];
  double C[NS * NS];
  if (sp.inverse_type == 2) {
    pinv<NS>(A, sp.ftol, C);
  } else {
    invert<NS>(A);
#pragma unroll
    for (int k = 0; k < NS * NS; k++) C[k] = A[k];
  }
#pragma unroll
  for (int j = 0; j < NS; j++) {
    double v[NS];
#pragma unroll
    for (int i = 0; i < NS; i++) v[i] = C[i + NS * j] - 1.0 / alpha;
    col(j, v);
  }
}

template <int NS, bool LP, class DF, class COL>
__device__ __forceinline__ void cell_chi(const SpParams &sp, const double (&rho)[NS], double rhotot,
                                         const double (&x)[NS], DF D, COL col) {
  if (LP) {
    double W[NS];
#pragma unroll
    for (int r = 0; r < NS; r++) W[r] = rho[r] / rhotot;
    chi_lapack<NS>(sp, x, W, D, col);
  } else {
    chi_iterative<NS>(sp, x, D, col);
  }
}

// choldc (use_lapack = F) or the dpotrf factor with the reference's clean-up
// (use_lapack = T), in place on a full (NS, NS) matrix in registers.
template <int NS, bool LP>
__device__ __forceinline__ void cholesky(double (&a)[NS * NS]) {
  if (!LP) {
    double p[NS];
#pragma unroll
    for (int i = 0; i < NS; i++) {
      bool sing = false;
#pragma unroll
      for (int j = i; j < NS; j++) {
        double s = a[i + NS * j];
#pragma unroll
        for (int k = i - 1; k >= 0; k--) s = s - a[i + NS * k] * a[j + NS * k];
        if (i == j) {
          if (s <= 0.0) {
            p[i] = 0.0;
            sing = true;
          } else {
            p[i] = sqrt(s);
          }
        } else {
          a[j + NS * i] = sing ? 0.0 : s / p[i];
        }
      }
    }
#pragma unroll
    for (int i = 0; i < NS; i++) {
#pragma unroll
      for (int j = i + 1; j < NS; j++) a[i + NS * j] = 0.0;
      a[i + NS * i] = p[i];
    }
    return;
  }
  bool stop = false;
#pragma unroll
  for (int j = 0; j < NS; j++) {
    if (stop) break;
    double s = a[j + NS * j];
#pragma unroll
    for (int k = 0; k < j; k++) s = s - a[j + NS * k] * a[j + NS * k];
    if (!(s > 0.0)) {
      a[j + NS * j] = s;
      stop = true;
      continue;
    }
    const double d = sqrt(s);
    a[j + NS * j] = d;
    const double rinv = 1.0 / d;
#pragma unroll
    for (int i = j + 1; i < NS; i++) {
      double t = a[i + NS * j];
#pragma unroll
      for (int k = 0; k < j; k++) t = t - a[i + NS * k] * a[j + NS * k];
      a[i + NS * j] = t * rinv;
    }
  }
#pragma unroll
  for (int r = 0; r < NS; r++)
#pragma unroll
    for (int c = r + 1; c < NS; c++) a[r + NS * c] = 0.0;
  a[(NS - 1) + NS * (NS - 1)] = 0.0;
}

// ---------------- kernels: the reference routines one by one ----------------

template <int NS>
__global__ void __launch_bounds__(STPB) k_sp_correct(Grid g, SpParams sp, double *rho, double *drho) {
  const long t = xcd_block() * blockDim.x + threadIdx.x;
  if (t >= g.N) return;
  const long N = g.N;
  double r[NS], d[NS];
  load<NS>(rho, N, t, r);
  cell_correct<NS>(sp, r, d);
#pragma unroll
  for (int n = 0; n < NS; n++) {
    rho[(long)n * N + t] = r[n];
    drho[(long)n * N + t] = d[n];
  }
}

template <int NS>
__global__ void __launch_bounds__(STPB) k_sp_prim(Grid g, SpParams sp, const double *rho, double *rhotot, double *xm,
                                                   double *mt) {
  const long t = xcd_block() * blockDim.x + threadIdx.x;
  if (t >= g.N) return;
  const long N = g.N;
  double r[NS], x[NS], tot, m;
  load<NS>(rho, N, t, r);
  cell_prim<NS>(sp, r, tot, x, m);
  rhotot[t] = tot;
  mt[t] = m;
#pragma unroll
  for (int n = 0; n < NS; n++) xm[(long)n * N + t] = x[n];
}

template <int NS>
__global__ void __launch_bounds__(STPB) k_sp_mixture(Grid g, SpParams sp, double *D_bar, double *D_therm, double *H) {
  const long t = xcd_block() * blockDim.x + threadIdx.x;
  if (t >= g.N) return;
  const long N = g.N;
  const DParam D{sp};
#pragma unroll
  for (int r = 0; r < NS; r++) {
    D_therm[(long)r * N + t] = sp.Dtherm[r];
#pragma unroll
    for (int c = 0; c < NS; c++) {
      D_bar[(long)(r + NS * c) * N + t] = D(r, c);
      double h = 0.0;
      if (!sp.ideal) h = (r == c) ? sp.Hdiag[r] : sp.Hoff[r > c ? tri(r, c) : tri(c, r)];
      H[(long)(r + NS * c) * N + t] = h;
    }
  }
}

template <int NS>
__global__ void __launch_bounds__(STPB) k_sp_gama(Grid g, SpParams sp, const double *xm, const double *H,
                                                   double *Gama) {
  const long t = xcd_block() * blockDim.x + threadIdx.x;
  if (t >= g.N) return;
  const long N = g.N;
  double x[NS];
  load<NS>(xm, N, t, x);
  auto Hf = [&](int k, int c) { return H[(long)(k + NS * c) * N + t]; };
#pragma unroll
  for (int r = 0; r < NS; r++)
#pragma unroll
    for (int c = 0; c < NS; c++) Gama[(long)(r + NS * c) * N + t] = gama_entry<NS>(sp, x, r, c, Hf);
}

template <int NS, bool LP>
__global__ void __launch_bounds__(STPB) k_sp_chi(Grid g, SpParams sp, const double *rho, const double *rhotot,
                                                  const double *xm, const double *Dbar, const double *Dtherm,
                                                  const double *Temp, double *chi, double *zeta) {
  const long t = xcd_block() * blockDim.x + threadIdx.x;
  if (t >= g.N) return;
  const long N = g.N;
  double r[NS], x[NS];
  load<NS>(rho, N, t, r);
  load<NS>(xm, N, t, x);
  const DField<NS> D{Dbar, N, t};
  if (sp.noniso) {
    double Dt[NS], z[NS];
    load<NS>(Dtherm, N, t, Dt);
    cell_zeta<NS>(x, D, Dt, Temp[t], z);
#pragma unroll
    for (int n = 0; n < NS; n++) zeta[(long)n * N + t] = z[n];
  }
  cell_chi<NS, LP>(sp, r, rhotot[t], x, D, [&](int j, const double (&v)[NS]) {
#pragma unroll
    for (int i = 0; i < NS; i++) chi[(long)(i + NS * j) * N + t] = v[i];
  });
}

template <int NS>
__global__ void __launch_bounds__(STPB) k_sp_rhowchi(Grid g, const double *rho, const double *chi, double *rw) {
  const long t = xcd_block() * blockDim.x + threadIdx.x;
  if (t >= g.N) return;
  const long N = g.N;
  double r[NS];
  load<NS>(rho, N, t, r);
#pragma unroll
  for (int i = 0; i < NS; i++)
#pragma unroll
    for (int j = 0; j < NS; j++) {
      const long q = (long)(i + NS * j) * N + t;
      rw[q] = -(r[i] * chi[q]);
    }
}

template <int NS>
__device__ __forceinline__ double lonsager_entry(const SpParams &sp, double mt, double rt, const double (&W)[NS],
                                                 int r, int c, double chi_rc) {
  return mt * rt * W[r] * chi_rc * W[c] / sp.k_B;
}

template <int NS, bool LP>
__global__ void __launch_bounds__(STPB) k_sp_lonsager(Grid g, SpParams sp, const double *rho, const double *rhotot,
                                                       const double *molmtot, const double *chi, double *L) {
  const long t = xcd_block() * blockDim.x + threadIdx.x;
  if (t >= g.N) return;
  const long N = g.N;
  double r[NS], W[NS], a[NS * NS];
  load<NS>(rho, N, t, r);
  const double rt = rhotot[t], mt = molmtot[t];
#pragma unroll
  for (int n = 0; n < NS; n++) W[n] = r[n] / rt;
#pragma unroll
  for (int c = 0; c < NS; c++)
#pragma unroll
    for (int i = 0; i < NS; i++) a[i + NS * c] = lonsager_entry<NS>(sp, mt, rt, W, i, c, chi[(long)(i + NS * c) * N + t]);
  cholesky<NS, LP>(a);
#pragma unroll
  for (int k = 0; k < NS * NS; k++) L[(long)k * N + t] = a[k];
}

// ---------------- face fluxes ----------------

// acc[r] += sum_c 0.5 (M(r, c) at t + at m) v[c], c ascending; LOWER: r >= c.
// AHEAD: the loads of column c + 1 are issued before column c is summed, so a column's
// wait overlaps the one before it.  The empty asm makes the indices of later
// columns depend on the sums of earlier ones: scheduling fences alone let the
// compiler load the whole matrix of both cells first (eight species: 256
// registers and one wave per SIMD, 73 us at 384 x 320; now 121 and 61 us).
// Otherwise a column is loaded and summed in turn (diff_ahead).
template <int NS, bool LOWER, bool PACKED = false, bool AHEAD = true>
__device__ __forceinline__ void face_matvec(const double *M, long N, long t, long m, const double (&v)[NS],
                                            double (&acc)[NS]) {
  auto at = [&](int r, int c) { return (long)(PACKED ? lpk_index<NS>(r, c) : r + NS * c) * N; };
  if constexpr (!AHEAD) {
#pragma unroll
    for (int c = 0; c < NS; c++) {
#pragma unroll
      for (int r = 0; r < NS; r++)
        if (!LOWER || r >= c) acc[r] = acc[r] + 0.5 * (M[at(r, c) + t] + M[at(r, c) + m]) * v[c];
      __builtin_amdgcn_sched_barrier(0);
    }
    return;
  }
  double a[2][NS], b[2][NS];
#pragma unroll
  for (int c = 0; c <= NS; c++) {
    if (c < NS) {
#pragma unroll
      for (int r = 0; r < NS; r++)
        if (!LOWER || r >= c) {
          a[c & 1][r] = M[at(r, c) + t];
          b[c & 1][r] = M[at(r, c) + m];
        }
    }
    if (c > 0) {
#pragma unroll
      for (int r = 0; r < NS; r++)
        if (!LOWER || r >= c - 1) {
          acc[r] = acc[r] + 0.5 * (a[(c - 1) & 1][r] + b[(c - 1) & 1][r]) * v[c - 1];
          asm volatile("" : "+v"(t), "+v"(m), "+v"(acc[r]));
        }
    }
  }
}

template <int NS>
__device__ __forceinline__ void correct_flux(const SpParams &sp, double (&out)[NS]) {
  if (sp.correct && NS > 1) {
    double sum = 0.0;
#pragma unroll
    for (int s = 0; s < NS - 1; s++) sum = sum + out[s];
    out[NS - 1] = -sum;
  }
}

// Gama_face grad x + zeta_face grad T + baro_face gradp_baro of the face
// between cells t (above) and m (below): the vector that
// rhoWchi_face multiplies.  Gama null: identity.
template <int NS, bool AHEAD>
__device__ __forceinline__ void diff_drive(long N, double dxinv, long t, long m, const double *xm, const double *gama,
                                           const double *temp, const double *zeta, const double *baro, double gpb,
                                           double (&y)[NS]) {
  double x[NS];
#pragma unroll
  for (int s = 0; s < NS; s++) x[s] = (xm[(long)s * N + t] - xm[(long)s * N + m]) * dxinv;
  if (gama) {
#pragma unroll
    for (int r = 0; r < NS; r++) y[r] = 0.0;
    face_matvec<NS, false, false, AHEAD>(gama, N, t, m, x, y);
  } else {
    // Gama_face = I: the sum 0 + 0*x_0 + ... + 1*x_r + ... is 0 + x_r
#pragma unroll
    for (int r = 0; r < NS; r++) y[r] = 0.0 + x[r];
  }
  if (zeta) {
    const double gT = (temp[t] - temp[m]) * dxinv;
#pragma unroll
    for (int s = 0; s < NS; s++)
      y[s] = y[s] + 0.5 * (zeta[(long)s * N + t] + zeta[(long)s * N + m]) * gT;
  }
  if (baro) {
#pragma unroll
    for (int s = 0; s < NS; s++)
      y[s] = y[s] + 0.5 * (baro[(long)s * N + t] + baro[(long)s * N + m]) * gpb;
  }
}

// diffusive_mass_flux: rhoWchi_face times the above, correction_flux.
template <int NS, bool AHEAD = true>
__device__ __forceinline__ void diff_face(const SpParams &sp, long N, double dxinv, long t, long m, const double *xm,
                                          const double *rw, const double *gama, const double *temp, const double *zeta,
                                          const double *baro, double gpb, double (&out)[NS]) {
  // opaque copies of the indices: keeps the compiler from hoisting this face's
  // loads out of a caller's loop; no instruction is emitted
  asm volatile("" : "+v"(t), "+v"(m));
  double y[NS];
  diff_drive<NS, AHEAD>(N, dxinv, t, m, xm, gama, temp, zeta, baro, gpb, y);
#pragma unroll
  for (int r = 0; r < NS; r++) out[r] = 0.0;
  face_matvec<NS, false, false, AHEAD>(rw, N, t, m, y, out);
  correct_flux<NS>(sp, out);
}

// sum_r w_r W_r of the face of cell t in direction d; PAST: read past the caches
template <int NS, bool PAST = true>
__device__ __forceinline__ void face_noise(long N, long t, int d, int dim, const double *W, int n_rngs,
                                           const double *weights, double (&w)[NS]) {
#pragma unroll
  for (int s = 0; s < NS; s++) w[s] = 0.0;
  for (int r = 0; r < n_rngs; r++) {
    const double wr = weights[r];
#pragma unroll
    for (int s = 0; s < NS; s++) {
      const double *p = W + ((long)(r * dim + d) * NS + s) * N + t;
      w[s] = w[s] + wr * (PAST ? __builtin_nontemporal_load(p) : *p);
    }
  }
}

// stochastic flux on the face of cell t in direction d: variance *
// L_face (sum_r w_r W_r), L_face the face average of the cell factors
// (upper triangle zero, so only c <= r enters: adding 0*w leaves the sum's
// bits unchanged), then correction_flux.  Packed or full factors.
template <int NS, bool PACKED, bool PAST>
__device__ __forceinline__ void stoch_face(const SpParams &sp, long N, long t, long m, int d, int dim, const double *L,
                                           const double *W, int n_rngs, const double *weights, double variance,
                                           double (&out)[NS]) {
  asm volatile("" : "+v"(t), "+v"(m));
  double w[NS];
  face_noise<NS, PAST>(N, t, d, dim, W, n_rngs, weights, w);
#pragma unroll
  for (int r = 0; r < NS; r++) out[r] = 0.0;
  face_matvec<NS, true, PACKED>(L, N, t, m, w, out);
#pragma unroll
  for (int r = 0; r < NS; r++) out[r] = out[r] * variance;
  correct_flux<NS>(sp, out);
}

// flux_total: ft_zero set -> 0.0 + F (setval then add), else ft + F
template <int NS, bool AHEAD>
__global__ void __launch_bounds__(STPB) k_sp_diff_flux(Grid g, SpParams sp, const double *xm, const double *rw,
                                                        const double *gama, const double *temp, const double *zeta,
                                                        const double *baro, Ptr3<const double> gpb, double *flux,
                                                        Ptr3<double> ft, int ft_zero) {
  const long t = xcd_block() * blockDim.x + threadIdx.x;
  if (t >= g.N) return;
  int i, j, k;
  decode(g, t, i, j, k);
  const Pt P = make_pt(g, i, j, k);
  const long N = g.N;
  const double dxinv = 1.0 / g.dx;
  for (int d = 0; d < g.dim; d++) {
    const long m = at_sh(g, P, d, -1, -1, 0);
    double out[NS];
    diff_face<NS, AHEAD>(sp, N, dxinv, t, m, xm, rw, gama, temp, zeta, baro,
                         baro ? gpb.c[d][t] : 0.0, out);
    double *const f = ft.c[d];
#pragma unroll
    for (int s = 0; s < NS; s++) {
      flux[((long)d * NS + s) * N + t] = out[s];
      const long q = (long)s * N;
      f[q + t] = (ft_zero ? 0.0 : f[q + t]) + out[s];
    }
  }
}

template <int NS, bool PAST>
__global__ void __launch_bounds__(STPB) k_sp_stoch_flux(Grid g, SpParams sp, const double *L, const double *W,
                                                         int n_rngs, const double *weights, double variance,
                                                         double *flux, Ptr3<double> ft) {
  const long t = xcd_block() * blockDim.x + threadIdx.x;
  if (t >= g.N) return;
  int i, j, k;
  decode(g, t, i, j, k);
  const Pt P = make_pt(g, i, j, k);
  const long N = g.N;
  for (int d = 0; d < g.dim; d++) {
    const long m = at_sh(g, P, d, -1, -1, 0);
    double out[NS];
    stoch_face<NS, false, PAST>(sp, N, t, m, d, g.dim, L, W, n_rngs, weights, variance, out);
    double *const f = ft.c[d];
#pragma unroll
    for (int s = 0; s < NS; s++) {
      flux[((long)d * NS + s) * N + t] = out[s];
      f[(long)s * N + t] = f[(long)s * N + t] + out[s];
    }
  }
}

// compute_div of species face fluxes (div_and_grad.f90:304-455)
template <int NS>
__global__ void __launch_bounds__(STPB) k_sp_div(Grid g, const double *flux, double *div, int increment) {
  const long t = xcd_block() * blockDim.x + threadIdx.x;
  if (t >= g.N) return;
  int i, j, k;
  decode(g, t, i, j, k);
  const Pt P = make_pt(g, i, j, k);
  const long N = g.N;
  const double dxinv = 1.0 / g.dx;
  const long ip = at3(g, P, 1, 0, 0), jp = at3(g, P, 0, 1, 0), kp = at3(g, P, 0, 0, 1);
#pragma unroll
  for (int s = 0; s < NS; s++) {
    const double *fx = flux + (long)s * N, *fy = flux + (long)(NS + s) * N;
    double v = (fx[ip] - fx[t]) * dxinv;
    v = v + (fy[jp] - fy[t]) * dxinv;
    if (g.dim == 3) {
      const double *fz = flux + (long)(2 * NS + s) * N;
      v = v + (fz[kp] - fz[t]) * dxinv;
    }
    div[(long)s * N + t] = increment ? div[(long)s * N + t] + v : v;
  }
}

// compute_mass_fluxdiv's face pass: both fluxes of each cell's lower faces in
// one kernel, flux_total = (0 + F_diff) + F_stoch written once.
//
// A face needs the matrices of its two cells, NS^2 + NS (NS + 1) / 2 values
// and more each, so a thread that walks its faces one by one reads its own
// cell's once and its neighbours' per direction, long after they left the
// XCD's 4 MB of L2 (the cells in flight there hold five times that).  Here a
// workgroup owns a 32 x 8 tile of a plane and takes the matrices column by
// column: the column is loaded once per cell (and for the tile's lower x and y
// halo), passed through LDS, and applied to the faces of all directions; the
// cell below in z reads it from memory beside the cell's own, when it is in L2.
// The next column is loaded before the current one is applied.  128^3, four
// species, two noise stages: 595 us face by face, 427 to 471 here from run to
// run (1.6 GB that a face pass cannot do without, 3.4 to 3.7 TB/s; 64 x 4
// tiles, with a larger halo, 481 where these took 446); 384 x 320, eight
// species: 124 us in a pass and a divergence per flux, 49 for this and the
// common divergence.  The noise is read and flux_total written past the caches
// (427 against 447 us in one run); the two fluxes are not, the divergence reads
// them next.
constexpr int FTX = 32, FTY = 8;
constexpr int FHX = FTX + 1, FHY = FTY + 1;  // with the lower halo column and row
constexpr int FHALO = FTX + FTY;

template <int NS, int DIM>
struct FaceTile {
  static constexpr int NH = (FHALO * NS + STPB - 1) / STPB;
  struct Col {
    double own[NS], z[DIM == 3 ? NS : 1], halo[NH];
  };
  long N, t, mz;            // the thread's cell and the one below it in z
  int at;                   // its place in a tile
  long hc[NH];              // halo cells that the thread loads: cell,
  int hr[NH], hat[NH];      // component (NS and more: none) and place
  double (*tile)[NS][FHY * FHX];  // two columns

  // Loads from here on wait for v (no instruction): left alone, the compiler
  // loads whole matrices ahead of their columns, barriers or not.
  __device__ __forceinline__ void after(double &v) {
    asm volatile("" : "+v"(t), "+v"(mz), "+v"(v));
#pragma unroll
    for (int n = 0; n < NH; n++) asm volatile("" : "+v"(hc[n]), "+v"(v));
  }
  // component `index(r, c)` of M for r >= first(c)
  template <class IX>
  __device__ __forceinline__ void load(Col &a, const double *M, int lo, IX index) const {
#pragma unroll
    for (int r = 0; r < NS; r++)
      if (r >= lo) {
        a.own[r] = M[(long)index(r) * N + t];
        if constexpr (DIM == 3) a.z[r] = M[(long)index(r) * N + mz];
      }
#pragma unroll
    for (int n = 0; n < NH; n++)
      if (hr[n] >= lo && hr[n] < NS) a.halo[n] = M[(long)index(hr[n]) * N + hc[n]];
  }
  __device__ __forceinline__ void put(const Col &a, int lo, int half) const {
#pragma unroll
    for (int r = 0; r < NS; r++)
      if (r >= lo) tile[half][r][at] = a.own[r];
#pragma unroll
    for (int n = 0; n < NH; n++)
      if (hr[n] >= lo && hr[n] < NS) tile[half][hr[n]][hat[n]] = a.halo[n];
  }
  // the value of the cell below in direction d
  __device__ __forceinline__ double below(const Col &a, int d, int r, int half) const {
    if (DIM == 3 && d == 2) return a.z[DIM == 3 ? r : 0];
    return tile[half][r][d == 0 ? at - 1 : at - FHX];
  }
  // f(d, r, own, below), a reference to what it computed, of one vector
  template <class F>
  __device__ __forceinline__ void vec(const double *V, F f) {
    Col a;
    load(a, V, 0, [](int r) { return r; });
    __syncthreads();
    put(a, 0, 0);
    __syncthreads();
#pragma unroll
    for (int d = 0; d < DIM; d++)
#pragma unroll
      for (int r = 0; r < NS; r++) after(f(d, r, a.own[r], below(a, d, r, 0)));
  }
  // acc[d][r] += 0.5 (M(r, c) here + below) v[d][c], c ascending
  template <bool LOWER, class IX>
  __device__ __forceinline__ void matvec(const double *M, const double (&v)[DIM][NS], double (&acc)[DIM][NS],
                                         IX index) {
    Col a, b;
    load(a, M, 0, [&](int r) { return index(r, 0); });
    __syncthreads();  // the tiles' last readers are done
#pragma unroll
    for (int c = 0; c < NS; c++) {
      const int lo = LOWER ? c : 0;
      if (c + 1 < NS) load(b, M, LOWER ? c + 1 : 0, [&](int r) { return index(r, c + 1); });
      put(a, lo, c & 1);
      // one barrier a column: a tile is written again two columns on, past the
      // barrier that its readers reach after reading it
      __syncthreads();
#pragma unroll
      for (int d = 0; d < DIM; d++)
#pragma unroll
        for (int r = 0; r < NS; r++)
          if (r >= lo) {
            acc[d][r] = acc[d][r] + 0.5 * (a.own[r] + below(a, d, r, c & 1)) * v[d][c];
            after(acc[d][r]);
          }
      a = b;
    }
  }
};

template <int NS, int DIM>
__global__ void __launch_bounds__(STPB) k_sp_chain_flux(Grid g, SpParams sp, SpFaceIn in, int nbx, int nz, double *fd,
                                                         double *fs, Ptr3<double> ft) {
  using Tile = FaceTile<NS, DIM>;
  __shared__ double tile[2][NS][FHY * FHX];
  // tiles along x, then z, then y: the plane below is a few workgroups back
  const unsigned w = (unsigned)xcd_block(), bx = w % nbx, q = w / nbx, k = q % nz, by = q / nz;
  const int nx = g.n[0], ny = g.n[1];
  const long sy = g.s[1], sz = DIM == 3 ? g.s[2] : 0;
  const int lx = threadIdx.x % FTX, ly = threadIdx.x / FTX, i0 = bx * FTX, j0 = by * FTY;
  const bool inside = i0 + lx < nx && j0 + ly < ny;
  // cells of a tile that hangs over the box: periodic images, nothing stored
  const long plane = sz * k;
  auto cell = [&](int i, int j) { return wrap_any(i, nx) + sy * wrap_any(j, ny) + plane; };
  Tile T;
  T.N = g.N;
  T.t = cell(i0 + lx, j0 + ly);
  T.mz = DIM == 3 ? T.t - plane + sz * (k == 0 ? nz - 1 : k - 1) : T.t;
  T.at = (ly + 1) * FHX + lx + 1;
  T.tile = tile;
#pragma unroll
  for (int n = 0; n < Tile::NH; n++) {
    const int h = threadIdx.x + STPB * n, e = h % FHALO;  // e: the row below, then the column below
    const int hx = e < FTX ? e : -1, hy = e < FTX ? -1 : e - FTX;
    T.hr[n] = h / FHALO;
    T.hc[n] = cell(i0 + hx, j0 + hy);
    T.hat[n] = (hy + 1) * FHX + hx + 1;
  }
  const long N = g.N, t = T.t;
  const double dxinv = 1.0 / g.dx;
  auto full = [](int r, int c) { return r + NS * c; };
  double x[DIM][NS], y[DIM][NS];
  T.vec(in.xm, [&](int d, int r, double a, double b) -> double & { return x[d][r] = (a - b) * dxinv; });
  if (in.gama) {
#pragma unroll
    for (int d = 0; d < DIM; d++)
#pragma unroll
      for (int r = 0; r < NS; r++) y[d][r] = 0.0;
    T.template matvec<false>(in.gama, x, y, full);
  } else {
    // Gama_face = I: the sum 0 + 0*x_0 + ... + 1*x_r + ... is 0 + x_r
#pragma unroll
    for (int d = 0; d < DIM; d++)
#pragma unroll
      for (int r = 0; r < NS; r++) y[d][r] = 0.0 + x[d][r];
  }
  long m[DIM];
#pragma unroll
  for (int d = 0; d < DIM; d++)
    m[d] = d == 0 ? cell(i0 + lx - 1, j0 + ly) : (d == 1 ? cell(i0 + lx, j0 + ly - 1) : T.mz);
  if (in.zeta) {
    double gT[DIM];
#pragma unroll
    for (int d = 0; d < DIM; d++) gT[d] = (in.temp[t] - in.temp[m[d]]) * dxinv;
    T.vec(in.zeta, [&](int d, int r, double a, double b) -> double & {
      return y[d][r] = y[d][r] + 0.5 * (a + b) * gT[d];
    });
  }
  if (in.baro) {
    double gp[DIM];
#pragma unroll
    for (int d = 0; d < DIM; d++) gp[d] = in.gpb[d][t];
    T.vec(in.baro, [&](int d, int r, double a, double b) -> double & {
      return y[d][r] = y[d][r] + 0.5 * (a + b) * gp[d];
    });
  }
  double od[DIM][NS], os[DIM][NS];
#pragma unroll
  for (int d = 0; d < DIM; d++)
#pragma unroll
    for (int r = 0; r < NS; r++) od[d][r] = os[d][r] = 0.0;
  T.template matvec<false>(in.rw, y, od, full);
  double wn[DIM][NS];
#pragma unroll
  for (int d = 0; d < DIM; d++) {
    correct_flux<NS>(sp, od[d]);
    face_noise<NS>(N, T.t, d, DIM, in.W, in.n_rngs, in.weights, wn[d]);
  }
  T.template matvec<true>(in.lpk, wn, os, [](int r, int c) { return lpk_index<NS>(r, c); });
  if (!inside) return;
#pragma unroll
  for (int d = 0; d < DIM; d++) {
#pragma unroll
    for (int r = 0; r < NS; r++) os[d][r] = os[d][r] * in.variance;
    correct_flux<NS>(sp, os[d]);
#pragma unroll
    for (int s = 0; s < NS; s++) {
      const long q = ((long)d * NS + s) * N + t;
      fd[q] = od[d][s];
      fs[q] = os[d][s];
      __builtin_nontemporal_store((0.0 + od[d][s]) + os[d][s], ft.c[d] + (long)s * N + t);
    }
  }
}

// The same face by face, both fluxes of each lower face in one thread: for
// boxes that would leave most of every tile empty (face_tiles).
template <int NS, bool PAST>
__global__ void __launch_bounds__(STPB) k_sp_face_flux(Grid g, SpParams sp, SpFaceIn in, double *fd, double *fs,
                                                        Ptr3<double> ft) {
  const long t = xcd_block() * blockDim.x + threadIdx.x;
  if (t >= g.N) return;
  int i, j, k;
  decode(g, t, i, j, k);
  const Pt P = make_pt(g, i, j, k);
  const long N = g.N;
  const double dxinv = 1.0 / g.dx;
  for (int d = 0; d < g.dim; d++) {
    const long m = at_sh(g, P, d, -1, -1, 0);
    double od[NS], os[NS];
    diff_face<NS>(sp, N, dxinv, t, m, in.xm, in.rw, in.gama, in.temp, in.zeta, in.baro,
                  in.baro ? in.gpb[d][t] : 0.0, od);
    stoch_face<NS, true, PAST>(sp, N, t, m, d, g.dim, in.lpk, in.W, in.n_rngs, in.weights, in.variance, os);
    double *const f = ft.c[d];
#pragma unroll
    for (int s = 0; s < NS; s++) {
      const long q = ((long)d * NS + s) * N + t;
      fd[q] = od[s];
      fs[q] = os[s];
      f[(long)s * N + t] = (0.0 + od[s]) + os[s];
    }
  }
}

// compute_div of two species face-flux sets in one pass
template <int NS>
__global__ void __launch_bounds__(STPB) k_sp_div2(Grid g, const double *fa, double *da, const double *fb,
                                                   double *db) {
  const long t = xcd_block() * blockDim.x + threadIdx.x;
  if (t >= g.N) return;
  int i, j, k;
  decode(g, t, i, j, k);
  const Pt P = make_pt(g, i, j, k);
  const long N = g.N;
  const double dxinv = 1.0 / g.dx;
  const long ip = at3(g, P, 1, 0, 0), jp = at3(g, P, 0, 1, 0), kp = at3(g, P, 0, 0, 1);
  for (int w = 0; w < 2; w++) {
    const double *flux = w ? fb : fa;
    double *div = w ? db : da;
#pragma unroll
    for (int s = 0; s < NS; s++) {
      const double *fx = flux + (long)s * N, *fy = flux + (long)(NS + s) * N;
      double v = (fx[ip] - fx[t]) * dxinv;
      v = v + (fy[jp] - fy[t]) * dxinv;
      if (g.dim == 3) {
        const double *fz = flux + (long)(2 * NS + s) * N;
        v = v + (fz[kp] - fz[t]) * dxinv;
      }
      div[(long)s * N + t] = v;
    }
  }
}

// ---------------- compute_mass_fluxdiv, fused ----------------

template <int NS, bool LP>
__global__ void __launch_bounds__(STPB) k_sp_chain_cell(Grid g, SpParams sp, const double *temp, SpCellOut o) {
  const long t = xcd_block() * blockDim.x + threadIdx.x;
  if (t >= g.N) return;
  const long N = g.N;
  double r[NS], dr[NS], x[NS], rt, mt;
  load<NS>(o.rho, N, t, r);
  cell_correct<NS>(sp, r, dr);
  cell_prim<NS>(sp, r, rt, x, mt);
#pragma unroll
  for (int n = 0; n < NS; n++) o.xm[(long)n * N + t] = x[n];
  const DParam D{sp};
  if (o.gama) {
    auto Hf = [&](int kk, int c) {
      return (kk == c) ? sp.Hdiag[kk] : sp.Hoff[kk > c ? tri(kk, c) : tri(c, kk)];
    };
#pragma unroll
    for (int i = 0; i < NS; i++)
#pragma unroll
      for (int c = 0; c < NS; c++) o.gama[(long)(i + NS * c) * N + t] = gama_entry<NS>(sp, x, i, c, Hf);
  }
  if (o.zeta) {
    double Dt[NS], z[NS];
#pragma unroll
    for (int n = 0; n < NS; n++) Dt[n] = sp.Dtherm[n];
    cell_zeta<NS>(x, D, Dt, temp[t], z);
#pragma unroll
    for (int n = 0; n < NS; n++) o.zeta[(long)n * N + t] = z[n];
  }
  if (o.baro) {
    double nn = 0.0;
#pragma unroll
    for (int c = 0; c < NS; c++) nn = nn + r[c] / sp.molmass[c];
#pragma unroll
    for (int c = 0; c < NS; c++) o.baro[(long)c * N + t] = r[c] / sp.rhobar[c] / (nn * sp.k_B * temp[t]);
  }
  double W[NS];
#pragma unroll
  for (int n = 0; n < NS; n++) W[n] = r[n] / rt;
  const bool want_l = o.lpk != nullptr;
  double a[NS * NS];
  cell_chi<NS, LP>(sp, r, rt, x, D, [&](int jc, const double (&v)[NS]) {
#pragma unroll
    for (int i = 0; i < NS; i++) {
      o.rw[(long)(i + NS * jc) * N + t] = -(r[i] * v[i]);
      a[i + NS * jc] = lonsager_entry<NS>(sp, mt, rt, W, i, jc, v[i]);
    }
  });
  if (want_l) {
    cholesky<NS, LP>(a);
#pragma unroll
    for (int c = 0; c < NS; c++)
#pragma unroll
      for (int i = c; i < NS; i++) o.lpk[(long)lpk_index<NS>(i, c) * N + t] = a[i + NS * c];
  }
#pragma unroll
  for (int n = 0; n < NS; n++) o.rho[(long)n * N + t] = r[n] + -1.0 * dr[n];
}

template <typename T>
Ptr3<const T> cp3(const T *const a[3]) {
  Ptr3<const T> r;
  for (int d = 0; d < 3; d++) r.c[d] = a ? a[d] : nullptr;
  return r;
}

// Dispatch on the species count.
template <template <int> class F, class... A>
int dispatch(int ns, A &&...args) {
  switch (ns) {
    case 1: return F<1>::run(args...);
    case 2: return F<2>::run(args...);
    case 3: return F<3>::run(args...);
    case 4: return F<4>::run(args...);
    case 5: return F<5>::run(args...);
    case 6: return F<6>::run(args...);
    case 7: return F<7>::run(args...);
    case 8: return F<8>::run(args...);
    default: return LMM_ERR_UNSUPPORTED;
  }
}

// NS = 1 has no chi (Dbar2chi divides by an empty sum): those routines
// reject it; the face fluxes take it.
#define SP_NEEDS2 \
  if (NS < 2) return LMM_ERR_UNSUPPORTED

template <int NS>
struct RunCorrect {
  static int run(hipStream_t s, const Grid &g, const SpParams &sp, double *rho, double *drho) {
    SP_NEEDS2;
    SLAUNCH(k_sp_correct<NS>, dim3(sblk(g.N)), dim3(STPB), 0, s, g, sp, rho, drho);
    return 0;
  }
};
template <int NS>
struct RunPrim {
  static int run(hipStream_t s, const Grid &g, const SpParams &sp, const double *rho, double *rt, double *xm,
                 double *mt) {
    SP_NEEDS2;
    SLAUNCH(k_sp_prim<NS>, dim3(sblk(g.N)), dim3(STPB), 0, s, g, sp, rho, rt, xm, mt);
    return 0;
  }
};
template <int NS>
struct RunMixture {
  static int run(hipStream_t s, const Grid &g, const SpParams &sp, double *Db, double *Dt, double *H) {
    SP_NEEDS2;
    SLAUNCH(k_sp_mixture<NS>, dim3(sblk(g.N)), dim3(STPB), 0, s, g, sp, Db, Dt, H);
    return 0;
  }
};
template <int NS>
struct RunGama {
  static int run(hipStream_t s, const Grid &g, const SpParams &sp, const double *xm, const double *H, double *G) {
    SP_NEEDS2;
    SLAUNCH(k_sp_gama<NS>, dim3(sblk(g.N)), dim3(STPB), 0, s, g, sp, xm, H, G);
    return 0;
  }
};
template <int NS>
struct RunChi {
  static int run(hipStream_t s, const Grid &g, const SpParams &sp, const double *rho, const double *rt,
                 const double *xm, const double *Db, const double *Dt, const double *T, double *chi, double *z) {
    SP_NEEDS2;
    if (sp.lapack)
      SLAUNCH((k_sp_chi<NS, true>), dim3(sblk(g.N)), dim3(STPB), 0, s, g, sp, rho, rt, xm, Db, Dt, T, chi, z);
    else
      SLAUNCH((k_sp_chi<NS, false>), dim3(sblk(g.N)), dim3(STPB), 0, s, g, sp, rho, rt, xm, Db, Dt, T, chi, z);
    return 0;
  }
};
template <int NS>
struct RunRhoWchi {
  static int run(hipStream_t s, const Grid &g, const double *rho, const double *chi, double *rw) {
    SP_NEEDS2;
    SLAUNCH(k_sp_rhowchi<NS>, dim3(sblk(g.N)), dim3(STPB), 0, s, g, rho, chi, rw);
    return 0;
  }
};
template <int NS>
struct RunLonsager {
  static int run(hipStream_t s, const Grid &g, const SpParams &sp, const double *rho, const double *rt,
                 const double *mt, const double *chi, double *L) {
    SP_NEEDS2;
    if (sp.lapack)
      SLAUNCH((k_sp_lonsager<NS, true>), dim3(sblk(g.N)), dim3(STPB), 0, s, g, sp, rho, rt, mt, chi, L);
    else
      SLAUNCH((k_sp_lonsager<NS, false>), dim3(sblk(g.N)), dim3(STPB), 0, s, g, sp, rho, rt, mt, chi, L);
    return 0;
  }
};
// Whether the diffusive face pass loads a column ahead: not for 5 and 6 species
// whose matrices exceed the 256 MB of the last-level cache, which gain nothing
// from it (128^3, diffusive_mass_fluxdiv in us, ahead / in turn: 5 species 708 /
// 681, 6 974 / 948, 8 species at 96^3 694 / 832; 512^2, in the cache: 5 species
// 67 / 69, 6 84 / 89, 8 129 / 151; at 2 to 4 no difference).
template <int NS>
inline bool diff_ahead(const Grid &g) {
  return (NS != 5 && NS != 6) || (double)NS * NS * g.N * sizeof(double) <= 256e6;
}
template <int NS>
inline auto diff_kernel(const Grid &g) {
  auto k = k_sp_diff_flux<NS, true>;
  if constexpr (NS == 5 || NS == 6)
    if (!diff_ahead<NS>(g)) k = k_sp_diff_flux<NS, false>;
  return k;
}
// Whether a face-by-face pass reads the noise past the caches: of which it
// uses every value once, but below about 55 MB it finds the noise in them
// (stochastic_mass_fluxdiv in us, past / through, two stages: 128^3 two species,
// 201 MB, 181 / 200; 512^2 two, 17 MB, 44.5 / 43.3, four, 34 MB, 60.5 / 59.0; 8 x
// 256 x 256 two, 50 MB, 64.9 / 60.2, four, 101 MB, 114 / 129).  From 6 species on
// the pass is the faster past them at any size (64 x 48 x 32 six, 28 MB, 66.7 /
// 69.7, eight 82.7 / 86.7).
template <int NS>
inline bool noise_past(const Grid &g, int n_rngs) {
  return NS >= 6 || (double)n_rngs * g.dim * NS * g.N * sizeof(double) > 55e6;
}

template <int NS>
struct RunDiffusive {
  static int run(hipStream_t s, const Grid &g, const SpParams &sp, const double *xm, const double *rw,
                 const double *G, const double *T, const double *z, const double *baro, const double *const gpb[3],
                 double *flux, double *const ft[3], double *div) {
    SLAUNCH(diff_kernel<NS>(g), dim3(sblk(g.N)), dim3(STPB), 0, s, g, sp, xm, rw, G, T, z, baro, cp3(gpb), flux,
            p3(ft), 0);
    SLAUNCH(k_sp_div<NS>, dim3(sblk(g.N)), dim3(STPB), 0, s, g, flux, div, 0);
    return 0;
  }
};
template <int NS>
struct RunBaro {
  static int run(hipStream_t s, const Grid &g, const SpParams &sp, const double *rho, const double *T, double *baro);
};
template <int NS>
struct RunStochastic {
  static int run(hipStream_t s, const Grid &g, const SpParams &sp, const double *L, const double *W, int nr,
                 const double *w, double var, double *flux, double *const ft[3], double *div, int inc) {
    auto kern = k_sp_stoch_flux<NS, true>;
    if constexpr (NS < 6)
      if (!noise_past<NS>(g, nr)) kern = k_sp_stoch_flux<NS, false>;
    SLAUNCH(kern, dim3(sblk(g.N)), dim3(STPB), 0, s, g, sp, L, W, nr, w, var, flux, p3(ft));
    SLAUNCH(k_sp_div<NS>, dim3(sblk(g.N)), dim3(STPB), 0, s, g, flux, div, inc);
    return 0;
  }
};
template <int NS>
struct RunChainCell {
  static int run(hipStream_t s, const Grid &g, const SpParams &sp, const double *T, const SpCellOut &o) {
    SP_NEEDS2;
    if (sp.lapack)
      SLAUNCH((k_sp_chain_cell<NS, true>), dim3(sblk(g.N)), dim3(STPB), 0, s, g, sp, T, o);
    else
      SLAUNCH((k_sp_chain_cell<NS, false>), dim3(sblk(g.N)), dim3(STPB), 0, s, g, sp, T, o);
    return 0;
  }
};
// Whether compute_mass_fluxdiv's face pass goes in tiles: not in 3D boxes of
// fewer than 12 cells in x, unless the tiles are so few that neither form fills
// the GPU.  The whole call in us, face by face / in tiles: 4 x 256 x 256 two
// species 68 / 113, four 136 / 250, eight 534 / 1014; 8 x 256 x 256 four
// 275 / 341; 10 x 160 x 160 four 136 / 147; 12 x 160 x 160 four 179 / 163 (two
// 75 / 78); 8 x 8 x 512 (512 tiles) four 56 / 50.  Thin in y (256 x 4 x 256 four
// species 138 / 123) and in 2D (4 x 8192 four 52 / 50) the tiles win.
inline bool face_tiles(const Grid &g, int ntiles) { return g.dim == 2 || g.n[0] >= 12 || ntiles <= 1024; }

template <int NS>
struct RunChainFace {
  static int run(hipStream_t s, const Grid &g, const SpParams &sp, const SpFaceIn &in, double *flux, double *dd,
                 double *sd, double *const ft[3]) {
    SP_NEEDS2;
    if (in.W) {  // flux holds 2 * dim * ns * N: the diffusive then the stochastic face fluxes
      double *fs = flux + (long)g.dim * NS * g.N;
      const int nbx = (g.n[0] + FTX - 1) / FTX, nby = (g.n[1] + FTY - 1) / FTY, nz = g.dim == 3 ? g.n[2] : 1;
      const dim3 nb(nbx * nby * nz);
      auto face = k_sp_face_flux<NS, true>;
      if constexpr (NS < 6)
        if (!noise_past<NS>(g, in.n_rngs)) face = k_sp_face_flux<NS, false>;
      if (!face_tiles(g, nbx * nby * nz))
        SLAUNCH(face, dim3(sblk(g.N)), dim3(STPB), 0, s, g, sp, in, flux, fs, p3(ft));
      else if (g.dim == 3)
        SLAUNCH((k_sp_chain_flux<NS, 3>), nb, dim3(STPB), 0, s, g, sp, in, nbx, nz, flux, fs, p3(ft));
      else
        SLAUNCH((k_sp_chain_flux<NS, 2>), nb, dim3(STPB), 0, s, g, sp, in, nbx, nz, flux, fs, p3(ft));
      SLAUNCH(k_sp_div2<NS>, dim3(sblk(g.N)), dim3(STPB), 0, s, g, flux, dd, fs, sd);
      return 0;
    }
    SLAUNCH(diff_kernel<NS>(g), dim3(sblk(g.N)), dim3(STPB), 0, s, g, sp, in.xm, in.rw, in.gama, in.temp, in.zeta,
            in.baro, cp3(in.baro ? in.gpb : nullptr), flux, p3(ft), 1);
    SLAUNCH(k_sp_div<NS>, dim3(sblk(g.N)), dim3(STPB), 0, s, g, flux, dd, 0);
    return 0;
  }
};

// compute_baro_coef on cells (the diffusive entry computes it from rho)
template <int NS>
__global__ void __launch_bounds__(STPB) k_sp_baro(Grid g, SpParams sp, const double *rho, const double *temp,
                                                   double *baro) {
  const long t = xcd_block() * blockDim.x + threadIdx.x;
  if (t >= g.N) return;
  const long N = g.N;
  double r[NS];
  load<NS>(rho, N, t, r);
  double nn = 0.0;
#pragma unroll
  for (int c = 0; c < NS; c++) nn = nn + r[c] / sp.molmass[c];
#pragma unroll
  for (int c = 0; c < NS; c++) baro[(long)c * N + t] = r[c] / sp.rhobar[c] / (nn * sp.k_B * temp[t]);
}

template <int NS>
int RunBaro<NS>::run(hipStream_t s, const Grid &g, const SpParams &sp, const double *rho, const double *T,
                     double *baro) {
  SLAUNCH(k_sp_baro<NS>, dim3(sblk(g.N)), dim3(STPB), 0, s, g, sp, rho, T, baro);
  return 0;
}

}  // namespace

int sp_correct_rho(hipStream_t s, const Grid &g, const SpParams &sp, double *rho, double *drho) {
  return dispatch<RunCorrect>(sp.ns, s, g, sp, rho, drho);
}
int sp_cons_to_prim(hipStream_t s, const Grid &g, const SpParams &sp, const double *rho, double *rhotot,
                    double *molarconc, double *molmtot) {
  return dispatch<RunPrim>(sp.ns, s, g, sp, rho, rhotot, molarconc, molmtot);
}
int sp_mixture(hipStream_t s, const Grid &g, const SpParams &sp, double *D_bar, double *D_therm, double *H) {
  return dispatch<RunMixture>(sp.ns, s, g, sp, D_bar, D_therm, H);
}
int sp_gama(hipStream_t s, const Grid &g, const SpParams &sp, const double *molarconc, const double *H,
            double *Gama) {
  return dispatch<RunGama>(sp.ns, s, g, sp, molarconc, H, Gama);
}
int sp_chi(hipStream_t s, const Grid &g, const SpParams &sp, const double *rho, const double *rhotot,
           const double *molarconc, const double *D_bar, const double *D_therm, const double *Temp, double *chi,
           double *zeta) {
  return dispatch<RunChi>(sp.ns, s, g, sp, rho, rhotot, molarconc, D_bar, D_therm, Temp, chi, zeta);
}
int sp_rhowchi(hipStream_t s, const Grid &g, const SpParams &sp, const double *rho, const double *chi,
               double *rhoWchi) {
  return dispatch<RunRhoWchi>(sp.ns, s, g, rho, chi, rhoWchi);
}
int sp_lonsager(hipStream_t s, const Grid &g, const SpParams &sp, const double *rho, const double *rhotot,
                const double *molmtot, const double *chi, double *L) {
  return dispatch<RunLonsager>(sp.ns, s, g, sp, rho, rhotot, molmtot, chi, L);
}
int sp_diffusive(hipStream_t s, const Grid &g, const SpParams &sp, const double *rho, const double *molarconc,
                 const double *rhoWchi, const double *Gama, const double *Temp, const double *zeta,
                 const double *const gpb[3], double *baro, double *flux, double *const flux_total[3], double *div) {
  if (gpb) {
    if (int rc = dispatch<RunBaro>(sp.ns, s, g, sp, rho, Temp, baro)) return rc;
  } else {
    baro = nullptr;
  }
  return dispatch<RunDiffusive>(sp.ns, s, g, sp, molarconc, rhoWchi, Gama, Temp, zeta, baro, gpb, flux, flux_total,
                                div);
}
int sp_stochastic(hipStream_t s, const Grid &g, const SpParams &sp, const double *L, const double *W, int n_rngs,
                  const double *weights, double variance, double *flux, double *const flux_total[3], double *div,
                  int increment) {
  return dispatch<RunStochastic>(sp.ns, s, g, sp, L, W, n_rngs, weights, variance, flux, flux_total, div, increment);
}
int sp_chain_cell(hipStream_t s, const Grid &g, const SpParams &sp, const double *Temp, const SpCellOut &o) {
  return dispatch<RunChainCell>(sp.ns, s, g, sp, Temp, o);
}
int sp_chain_face(hipStream_t s, const Grid &g, const SpParams &sp, const SpFaceIn &in, double *flux,
                  double *diff_div, double *stoch_div, double *const flux_total[3]) {
  return dispatch<RunChainFace>(sp.ns, s, g, sp, in, flux, diff_div, stoch_div, flux_total);
}

}  // namespace lmm
