// assemble.hip -- symbolic pattern, geometry pass, host side of the numeric
// volume assembly, and Neumann traction kernels for tensor-product B-spline
// patches on gfx950.
//
// Numeric assembly is row-owned ("owner computes"): the geometry pass writes
// a record per (element, Gauss point), then line kernels (lines.hpp,
// lines_direct.hpp) form the rows of node lines.  Every K entry is written
// exactly once, coalesced, without atomics, and the summation order is
// fixed, so results are bitwise reproducible.
//
// This replaces the reference's element loop with colour groups and the
// per-entry std::find scatter (src/ASM/ASMs3D.C:2071-2335,
// src/LinAlg/SparseMatrix.C:614-688); the per-GP arithmetic follows
// utl::Jacobian (src/Utility/CoordinateMapping.C:24-63) and the integrands
// of Integrand::evalInt.
#include <hip/hip_runtime.h>

#include <type_traits>

#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

#include "asmargs.hpp"
#include "devutil.hpp"
#include "internal.hpp"
#include "lines_launch.hpp"

namespace ifem {

// ---------------------------------------------------------------------------
// Gauss-Legendre rule by Newton iteration on the Legendre polynomial in long
// double (same nodes/weights as the reference tables G1..G10,
// src/Utility/GaussQuadrature.C:17-60, to the last bit or one ulp).
static void gauss_rule(int n, double* xi, double* w)
{
  const long double pi = 3.141592653589793238462643383279502884L;
  for (int i = 0; i < n; i++) {
    long double x = cosl(pi * (i + 0.75L) / (n + 0.5L));
    long double dp = 0.0L;
    for (int it = 0; it < 100; it++) {
      long double p0 = 1.0L, p1 = x;
      for (int k = 1; k < n; k++) {
        long double p2 = ((2 * k + 1) * x * p1 - k * p0) / (k + 1);
        p0 = p1;
        p1 = p2;
      }
      dp = n * (x * p1 - p0) / (x * x - 1.0L);
      long double dx = p1 / dp;
      x -= dx;
      if (fabsl(dx) < 1e-30L) break;
    }
    if (2 * i + 1 == n) x = 0.0L;
    long double p0 = 1.0L, p1 = x;
    for (int k = 1; k < n; k++) {
      long double p2 = ((2 * k + 1) * x * p1 - k * p0) / (k + 1);
      p0 = p1;
      p1 = p2;
    }
    dp = n * (x * p1 - p0) / (x * x - 1.0L);
    xi[n - 1 - i] = (double)x;
    w[n - 1 - i] = (double)(2.0L / ((1.0L - x * x) * dp * dp));
  }
}

// ---------------------------------------------------------------------------
// 1D B-spline values and first derivatives on span s (Cox-de Boor,
// Piegl & Tiller A2.2/A2.3), the per-direction factor of GoTools'
// SplineVolume::computeBasisGrid (src/ASM/ASMs3D.C:4114-4143).
template <int P>
__device__ inline void bspline_1d(const double* __restrict__ t, int s, double u, double* N,
                                  double* dN)
{
  double left[P + 1], right[P + 1], ndu[P + 1][P + 1];
  ndu[0][0] = 1.0;
#pragma unroll
  for (int j = 1; j <= P; j++) {
    left[j] = u - t[s + 1 - j];
    right[j] = t[s + j] - u;
    double saved = 0.0;
#pragma unroll
    for (int r = 0; r < j; r++) {
      ndu[j][r] = right[r + 1] + left[j - r];
      double temp = ndu[r][j - 1] / ndu[j][r];
      ndu[r][j] = saved + right[r + 1] * temp;
      saved = left[j - r] * temp;
    }
    ndu[j][j] = saved;
  }
#pragma unroll
  for (int r = 0; r <= P; r++) {
    N[r] = ndu[r][P];
    double d = 0.0;
    if (r >= 1) d += ndu[r - 1][P - 1] / ndu[P][r - 1];
    if (r <= P - 1) d -= ndu[r][P - 1] / ndu[P][r];
    dN[r] = P * d;
  }
}

struct GaussArgs {
  double xi[kMaxNG];
  double w[kMaxNG];
};

// Tables per direction: for element e and Gauss point g, N and dN/du of the
// p+1 nonzero functions, plus the span length.
template <int P>
__global__ void k_basis_tables(const double* __restrict__ t, int nel, int ng, GaussArgs ga,
                               double* __restrict__ tabN, double* __restrict__ tabD,
                               double* __restrict__ span)
{
  const int id = blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= nel * ng) return;
  const int e = id / ng, g = id % ng;
  const int s = e + P;
  const double u0 = t[s], u1 = t[s + 1];
  const double u = 0.5 * ((u1 - u0) * ga.xi[g] + u1 + u0); // SplineUtils.C:217
  double N[P + 1], dN[P + 1];
  bspline_1d<P>(t, s, u, N, dN);
#pragma unroll
  for (int a = 0; a <= P; a++) {
    tabN[id * (P + 1) + a] = N[a];
    tabD[id * (P + 1) + a] = dN[a];
  }
  if (g == 0) span[e] = u1 - u0;
}

// ---------------------------------------------------------------------------
// cos(x) for the Fourier fields: Cody-Waite argument reduction modulo pi
// (W. J. Cody and W. Waite, Software Manual for the Elementary Functions,
// 1980: pi split into three doubles, each product subtracted by a fused
// multiply-add; the first difference is exact), cos x = (-1)^n cos r with
// |r| <= pi/2, and the Taylor series of cos to degree 20 (truncation below
// 2e-17 at |r| = pi/2).  Absolute error below 1.3 ulp(1) and within 2 ulp of
// the C library's cos where |cos x| > 1/2, for |x| <= 1e9 (2e7 samples per
// range, also next to multiples of pi/2 and pi); larger |x| goes to the
// library routine, kept out of line so that its registers do not count
// against the callers.  The 128-mode log-normal conductivity spends most of
// the geometry pass in this function.
__device__ __noinline__ double cos_library(double x)
{
  return cos(x);
}

__device__ __noinline__ double sin_library(double x)
{
  return sin(x);
}

// Reduction modulo pi: x = n pi + r, |r| <= pi/2; returns n, r^2 in s.
__device__ inline double reduce_pi(double x, double& s)
{
  const double n = rint(x * 0x1.45f306dc9c883p-2); // x / pi
  double r = fma(-n, 0x1.921fb54442d18p+1, x);     // pi, three parts
  r = fma(-n, 0x1.1a62633145c07p-53, r);
  r = fma(-n, -0x1.f1976b7ed8fbcp-109, r);
  s = r * r;
  return n;
}

// Taylor coefficients of cos in r^2, highest first: 1/20!, -1/18!, ..., 1.
__device__ constexpr double kCosTaylor[11] = {
    1.0 / 2432902008176640000.0, -1.0 / 6402373705728000.0, 1.0 / 20922789888000.0,
    -1.0 / 87178291200.0,        1.0 / 479001600.0,         -1.0 / 3628800.0,
    1.0 / 40320.0,               -1.0 / 720.0,              1.0 / 24.0,
    -0.5,                        1.0};

// |x| <= 2^30 (no check)
__device__ inline double cos_reduced(double x)
{
  double s;
  const double n = reduce_pi(x, s);
  double c = kCosTaylor[0];
#pragma unroll
  for (int k = 1; k < 11; k++) c = fma(c, s, kCosTaylor[k]);
  return ((int)n & 1) ? -c : c;
}

__device__ inline double cos_cw(double x)
{
  return fabs(x) <= 0x1p30 ? cos_reduced(x) : cos_library(x);
}

// Mode tables are read through the constant address space: where the table
// pointer is the same for the whole wave the compiler loads the modes with
// scalar loads (no vector registers, no per-lane memory instructions).
typedef const __attribute__((address_space(4))) double* ConstModes;

// sum_m a_m cos(k_m.x + phi_m), four modes at a time, summed in mode order.
// FAST: every argument is known to be within 2^30 (no library fallback, so
// no call in the loop); the four cosines run the operations of cos_reduced
// with their polynomial steps interleaved (four independent chains).
template <bool FAST>
__device__ inline double fourier_sum(const DevFunction& f, double x, double y, double z)
{
  double acc = 0.0;
  ConstModes md = (ConstModes)f.modes;
  int m = 0;
  for (; m + 4 <= f.nmodes; m += 4, md += 20) {
    double c[4];
    if (FAST) {
      double n[4], s[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const double arg = md[5 * u] * x + md[5 * u + 1] * y + md[5 * u + 2] * z + md[5 * u + 3];
        n[u] = reduce_pi(arg, s[u]);
        c[u] = kCosTaylor[0];
      }
#pragma unroll
      for (int k = 1; k < 11; k++)
#pragma unroll
        for (int u = 0; u < 4; u++) c[u] = fma(c[u], s[u], kCosTaylor[k]);
#pragma unroll
      for (int u = 0; u < 4; u++) c[u] = ((int)n[u] & 1) ? -c[u] : c[u];
    } else {
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const double arg = md[5 * u] * x + md[5 * u + 1] * y + md[5 * u + 2] * z + md[5 * u + 3];
        c[u] = cos_cw(arg);
      }
    }
#pragma unroll
    for (int u = 0; u < 4; u++) acc += md[5 * u + 4] * c[u];
  }
  for (; m < f.nmodes; m++, md += 5) {
    const double arg = md[0] * x + md[1] * y + md[2] * z + md[3];
    acc += md[4] * (FAST ? cos_reduced(arg) : cos_cw(arg));
  }
  return acc;
}

// Scalar fields evaluated at Gauss points (same definitions as the oracle).
__device__ inline double eval_field(const DevFunction& f, double x, double y, double z)
{
  switch (f.type) {
  case IFEM_GPU_FN_CONST:
    return f.scale;
  case IFEM_GPU_FN_SINPROD:
    return f.scale * sin_library(M_PI * x) * sin_library(M_PI * y) * sin_library(M_PI * z);
  case IFEM_GPU_FN_FOURIER:
  case IFEM_GPU_FN_EXP_FOURIER: {
    // the bound (with a margin for rounding) decides once per point
    const double xm = fmax(fabs(x), fmax(fabs(y), fabs(z)));
    const double s = f.kbound * xm + f.pbound <= 0x1p29 ? fourier_sum<true>(f, x, y, z)
                                                        : fourier_sum<false>(f, x, y, z);
    const double g = f.mean + f.scale * s;
    return f.type == IFEM_GPU_FN_EXP_FOURIER ? exp(g) : g;
  }
  default:
    return 0.0;
  }
}

// Geometry pre-pass: one thread per (element, Gauss point) computes, once
// per element, what the line kernels would otherwise recompute in each of the
// (p+1)^2 lines touching the element: J = X dN/du with the reference's
// cofactor det/inverse (utl::Jacobian, src/Utility/CoordinateMapping.C:24-63,
// src/LinAlg/matrix.h:791-862, |detJ| <= 1e-12 drops the point),
// detJxW = detJ*dV*w_i*w_j*w_k (src/ASM/ASMs3D.C:2145,2285), and for scalar
// problems the material kappa(X) and source f(X) at X = sum_b N_b x_b
// (src/ASM/ASMs3D.C:2303), folded into the record GeoRec.
__device__ inline bool field_varies(const DevFunction& f)
{
  return f.type == IFEM_GPU_FN_SINPROD ||
         ((f.type == IFEM_GPU_FN_FOURIER || f.type == IFEM_GPU_FN_EXP_FOURIER) && f.nmodes > 0);
}

__device__ inline DevFunction load_function(const __attribute__((address_space(4))) DevFunction& f)
{
  DevFunction d;
  d.type = f.type;
  d.nmodes = f.nmodes;
  d.scale = f.scale;
  d.mean = f.mean;
  d.modes = f.modes;
  d.kbound = f.kbound;
  d.pbound = f.pbound;
  return d;
}

template <int P, bool VEC = false>
__device__ inline void gp_geometry_at(ConstArgs& a, int64_t id, bool want_rhs)
{
  constexpr int P1 = P + 1;
  const int ng = a.ng;
  const int gp3 = ng * ng * ng;
  const int64_t e = id / gp3;
  const int q = (int)(id - e * gp3);
  const int q1 = q % ng, q2 = (q / ng) % ng, q3 = q / (ng * ng);
  const int e1 = (int)(e % a.nel1), e2 = (int)((e / a.nel1) % a.nel2),
            e3 = (int)(e / ((int64_t)a.nel1 * a.nel2));
  double J[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  double X[3] = {0.0, 0.0, 0.0};
#pragma unroll 1
  for (int b3 = 0; b3 < P1; b3++)
#pragma unroll 1
    for (int b2 = 0; b2 < P1; b2++)
#pragma unroll
      for (int b1 = 0; b1 < P1; b1++) {
        const double n1 = a.tabN1[(e1 * ng + q1) * P1 + b1], d1 = a.tabD1[(e1 * ng + q1) * P1 + b1];
        const double n2 = a.tabN2[(e2 * ng + q2) * P1 + b2], d2 = a.tabD2[(e2 * ng + q2) * P1 + b2];
        const double n3 = a.tabN3[(e3 * ng + q3) * P1 + b3], d3 = a.tabD3[(e3 * ng + q3) * P1 + b3];
        const double g0 = d1 * n2 * n3, g1 = n1 * d2 * n3, g2 = n1 * n2 * d3;
        const double nv = n1 * n2 * n3;
        const int64_t node =
            (int64_t)(e1 + b1) + (int64_t)a.n1 * ((e2 + b2) + (int64_t)a.n2 * (e3 + b3));
#pragma unroll
        for (int i = 0; i < 3; i++) {
          const double xi = a.coefs[3 * node + i];
          J[3 * i + 0] += xi * g0;
          J[3 * i + 1] += xi * g1;
          J[3 * i + 2] += xi * g2;
          X[i] += xi * nv;
        }
      }
  const double det = J[0] * (J[4] * J[8] - J[7] * J[5]) - J[1] * (J[3] * J[8] - J[6] * J[5]) +
                     J[2] * (J[3] * J[7] - J[6] * J[4]);
  double Ji[9];
  double wdet;
  if (det <= 1e-12 && det >= -1e-12) {
#pragma unroll
    for (int m = 0; m < 9; m++) Ji[m] = 0.0;
    wdet = 0.0;
  } else {
    Ji[0] = (J[4] * J[8] - J[7] * J[5]) / det;
    Ji[3] = -(J[3] * J[8] - J[6] * J[5]) / det;
    Ji[6] = (J[3] * J[7] - J[6] * J[4]) / det;
    Ji[1] = -(J[1] * J[8] - J[7] * J[2]) / det;
    Ji[4] = (J[0] * J[8] - J[6] * J[2]) / det;
    Ji[7] = -(J[0] * J[7] - J[6] * J[1]) / det;
    Ji[2] = (J[1] * J[5] - J[4] * J[2]) / det;
    Ji[5] = -(J[0] * J[5] - J[3] * J[2]) / det;
    Ji[8] = (J[0] * J[4] - J[3] * J[1]) / det;
    const double dV = 0.125 * (a.span1[e1] * a.span2[e2] * a.span3[e3]);
    wdet = det * (dV * a.gw[q1] * a.gw[q2] * a.gw[q3]);
  }
  if ((VEC || a.ncomp == 3) && a.geo_pairs) {
    double2* out = reinterpret_cast<double2*>(a.gp_geo) + e * gp3 * (GeoRec<3>::N / 2) + q;
#pragma unroll
    for (int k = 0; k < 4; k++) out[k * gp3] = make_double2(Ji[2 * k], Ji[2 * k + 1]);
    out[4 * gp3] = make_double2(Ji[8], wdet);
    return;
  }
  if (VEC || a.ncomp == 3) {
    double* out = a.gp_geo + e * gp3 * GeoRec<3>::N + q;
#pragma unroll
    for (int k = 0; k < 9; k++) out[k * gp3] = Ji[k];
    out[9 * gp3] = wdet;
    return;
  }
  const DevFunction kf = load_function(a.kappa), sf = load_function(a.source);
  const double kap = field_varies(kf) ? eval_field(kf, X[0], X[1], X[2]) : a.kappa_c;
  const double sk = wdet * kap;
  double* out = a.gp_geo + e * gp3 * GeoRec<1>::N + q;
  out[0] = sk * (Ji[0] * Ji[0] + Ji[1] * Ji[1] + Ji[2] * Ji[2]);
  out[gp3] = sk * (Ji[0] * Ji[3] + Ji[1] * Ji[4] + Ji[2] * Ji[5]);
  out[2 * gp3] = sk * (Ji[0] * Ji[6] + Ji[1] * Ji[7] + Ji[2] * Ji[8]);
  out[3 * gp3] = sk * (Ji[3] * Ji[3] + Ji[4] * Ji[4] + Ji[5] * Ji[5]);
  out[4 * gp3] = sk * (Ji[3] * Ji[6] + Ji[4] * Ji[7] + Ji[5] * Ji[8]);
  out[5 * gp3] = sk * (Ji[6] * Ji[6] + Ji[7] * Ji[7] + Ji[8] * Ji[8]);
  if (want_rhs)
    out[6 * gp3] = wdet * (field_varies(sf) ? eval_field(sf, X[0], X[1], X[2]) : a.source_c);
}

// Scalar problems: built for four waves per SIMD (at most 128 registers):
// the Fourier-mode loop is latency-bound, and more waves hide more of it
// (measured: 4 waves beat 2, 3, 5, 6 and 8 on the 256-patch diffusion batch;
// beyond 4 the geometry part spills).  Vector problems (no fields): their
// own instance without the field code, built for five waves per SIMD (64^3
// elasticity: 0.34 ms against 0.48 ms with the shared instance).
template <int P>
__global__ __launch_bounds__(256, 4) __attribute__((flatten)) void k_gp_geometry(
    const AsmArgs* __restrict__ args, int64_t total, int want_rhs)
{
  ConstArgs& a = *const_args(args);
  for (int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; id < total;
       id += (int64_t)gridDim.x * blockDim.x)
    gp_geometry_at<P>(a, id, want_rhs != 0);
}

template <int P>
__global__ __launch_bounds__(256, 5) void k_gp_geometry_vec(const AsmArgs* __restrict__ args,
                                                            int64_t total)
{
  ConstArgs& a = *const_args(args);
  for (int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; id < total;
       id += (int64_t)gridDim.x * blockDim.x)
    gp_geometry_at<P, true>(a, id, false);
}

// The value of the wave's first active lane (64-bit).
__device__ __forceinline__ int64_t readfirstlane64(int64_t v)
{
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)((uint64_t)v >> 32));
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

// Batch, one launch per degree P: the patches of that degree are
// plist[0..np), patch plist[i] holding points [gq0[i], gq0[i+1]) of the
// launch's total.  The point function is inlined (flatten: no call, so no
// register saves to scratch per point; the library fallbacks stay calls).
template <int P>
__global__ __launch_bounds__(256, 4) __attribute__((flatten)) void k_gp_geometry_batch(
    const AsmArgs* __restrict__ args, const int* __restrict__ plist,
    const int64_t* __restrict__ gq0, int np, int64_t total, int want_rhs)
{
  for (int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; id < total;
       id += (int64_t)gridDim.x * blockDim.x) {
    // The wave's first point (its lowest index) picks a patch by a
    // wave-uniform search; a wave whose points all lie in that patch (all
    // but the waves that straddle a patch boundary) runs with the patch index
    // as a wave-uniform value, so that the patch's arguments and mode tables
    // come through scalar loads.
    const int64_t idw = readfirstlane64(id);
    int lw = 0, hw = np - 1;
    while (lw < hw) {
      const int mid = (lw + hw + 1) >> 1;
      if (gq0[mid] <= idw) lw = mid;
      else hw = mid - 1;
    }
    const int64_t wend = lw + 1 < np ? gq0[lw + 1] : total;
    if (__ballot(id >= wend) == 0) {
      const int pl = __builtin_amdgcn_readfirstlane(plist[lw]);
      gp_geometry_at<P>(const_args(args)[pl], id - readfirstlane64(gq0[lw]), want_rhs != 0);
    } else {
      int lo = 0, hi = np - 1;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (gq0[mid] <= id) lo = mid;
        else hi = mid - 1;
      }
      gp_geometry_at<P>(const_args(args)[plist[lo]], id - gq0[lo], want_rhs != 0);
    }
  }
}

// Value of a constant field (kappa of type ZERO means 1).
static double const_value(const ifem_gpu_function& f, double zero_value)
{
  switch (f.type) {
  case IFEM_GPU_FN_CONST: return f.scale;
  case IFEM_GPU_FN_FOURIER: return f.mean;
  case IFEM_GPU_FN_EXP_FOURIER: return std::exp(f.mean);
  case IFEM_GPU_FN_ZERO: return zero_value;
  default: return 0.0;
  }
}

static int grid_for(int64_t total)
{
  const int64_t g = (total + 255) / 256;
  return (int)(g < 1 ? 1 : (g > 65536 ? 65536 : g));
}

// ---------------------------------------------------------------------------
// Symbolic pattern: row lengths, scan, columns.  Two nodes couple when their
// index boxes are within p in every direction (open knots, simple interior
// knots); eliminated DOFs are dropped.  Column order = DOF order =
// equation order (the SAM numbering is monotone), i.e. sorted.
__global__ void k_row_lengths(int n1, int n2, int n3, int p, int nc, const int* __restrict__ eq,
                              int64_t* __restrict__ rowlen, int ndof)
{
  const int d = blockIdx.x * blockDim.x + threadIdx.x;
  if (d >= ndof) return;
  const int r = eq[d];
  if (r < 0) return;
  const int node = d / nc;
  const int i = node % n1, j = (node / n1) % n2, k = node / (n1 * n2);
  int64_t cnt = 0;
  for (int kk = max(0, k - p); kk <= min(n3 - 1, k + p); kk++)
    for (int jj = max(0, j - p); jj <= min(n2 - 1, j + p); jj++)
      for (int ii = max(0, i - p); ii <= min(n1 - 1, i + p); ii++) {
        const int64_t nn = (int64_t)ii + (int64_t)n1 * (jj + (int64_t)n2 * kk);
        for (int c = 0; c < nc; c++) cnt += eq[nn * nc + c] >= 0;
      }
  rowlen[r] = cnt;
}

// One wave per row DOF; lanes write consecutive columns (ballot compaction).
__global__ void k_fill_columns(int n1, int n2, int n3, int p, int nc, const int* __restrict__ eq,
                               const int64_t* __restrict__ rowptr, int32_t* __restrict__ colind,
                               int ndof)
{
  const int d = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (d >= ndof) return;
  const int r = eq[d];
  if (r < 0) return;
  const int node = d / nc;
  const int i = node % n1, j = (node / n1) % n2, k = node / (n1 * n2);
  const int W1 = 2 * p + 1;
  const int total = W1 * W1 * W1 * nc;
  int64_t pos = rowptr[r];
  for (int t0 = 0; t0 < total; t0 += 64) {
    const int t = t0 + lane;
    bool valid = false;
    int col = 0;
    if (t < total) {
      const int nbr = t / nc, cc = t % nc;
      const int ii = i + nbr % W1 - p, jj = j + (nbr / W1) % W1 - p, kk = k + nbr / (W1 * W1) - p;
      if (ii >= 0 && ii < n1 && jj >= 0 && jj < n2 && kk >= 0 && kk < n3) {
        const int64_t nn = (int64_t)ii + (int64_t)n1 * (jj + (int64_t)n2 * kk);
        col = eq[nn * nc + cc];
        valid = col >= 0;
      }
    }
    const unsigned long long m = __ballot(valid);
    if (valid) colind[pos + __popcll(m & ((1ull << lane) - 1ull))] = col;
    pos += __popcll(m);
  }
}

// Exclusive scan of int64 (block-local scan, scan of block sums, add).
constexpr int kScanBlock = 1024;

__global__ void k_scan_local(const int64_t* __restrict__ in, int64_t* __restrict__ out,
                             int64_t* __restrict__ bsum, int n)
{
  __shared__ int64_t s[kScanBlock];
  const int i = blockIdx.x * kScanBlock + threadIdx.x;
  s[threadIdx.x] = i < n ? in[i] : 0;
  __syncthreads();
  for (int off = 1; off < kScanBlock; off <<= 1) {
    int64_t v = threadIdx.x >= off ? s[threadIdx.x - off] : 0;
    __syncthreads();
    s[threadIdx.x] += v;
    __syncthreads();
  }
  if (i < n) out[i + 1] = s[threadIdx.x]; // inclusive into out[1..]
  if (threadIdx.x == kScanBlock - 1) bsum[blockIdx.x] = s[threadIdx.x];
}

__global__ void k_scan_sums(int64_t* __restrict__ bsum, int nb)
{
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    int64_t run = 0;
    for (int b = 0; b < nb; b++) {
      const int64_t v = bsum[b];
      bsum[b] = run;
      run += v;
    }
  }
}

__global__ void k_scan_add(int64_t* __restrict__ out, const int64_t* __restrict__ bsum, int n)
{
  const int i = blockIdx.x * kScanBlock + threadIdx.x;
  if (i < n) out[i + 1] += bsum[blockIdx.x];
  if (i == 0) out[0] = 0;
}

// Several patches: the global pattern is the union of the patches' node
// couplings (nodes within +-p in every direction of one patch), built on the
// host (SAM::getDofCouplings over all patches, src/LinAlg/SAM.C:377-427).
int host_union_pattern(const Context& c, const std::vector<SubPatch>& subs, int neq,
                       std::vector<int64_t>& rowptr, std::vector<int32_t>& colind)
{
  const int nc = c.ncomp;
  std::vector<std::vector<int>> cols(neq > 0 ? neq : 1);
  for (const SubPatch& sp : subs) {
    const PatchRec& P = c.patches[sp.patch];
    const int p = P.p[0], n1 = P.n[0], n2 = P.n[1], n3 = P.n[2];
    for (int k = 0; k < n3; k++)
      for (int j = 0; j < n2; j++)
        for (int i = 0; i < n1; i++) {
          const int node = i + n1 * (j + n2 * k);
          for (int ci = 0; ci < nc; ci++) {
            const int r = sp.h_leq[node * nc + ci];
            if (r < 0) continue;
            std::vector<int>& row = cols[r];
            for (int kk = std::max(0, k - p); kk <= std::min(n3 - 1, k + p); kk++)
              for (int jj = std::max(0, j - p); jj <= std::min(n2 - 1, j + p); jj++)
                for (int ii = std::max(0, i - p); ii <= std::min(n1 - 1, i + p); ii++) {
                  const int nb = ii + n1 * (jj + n2 * kk);
                  for (int cj = 0; cj < nc; cj++) {
                    const int e = sp.h_leq[nb * nc + cj];
                    if (e >= 0) row.push_back(e);
                  }
                }
          }
        }
  }
  rowptr.assign(neq + 1, 0);
  for (int r = 0; r < neq; r++) {
    std::vector<int>& row = cols[r];
    std::sort(row.begin(), row.end());
    row.erase(std::unique(row.begin(), row.end()), row.end());
    rowptr[r + 1] = rowptr[r] + (int64_t)row.size();
  }
  const int64_t nnz = rowptr[neq];
  colind.assign(nnz > 0 ? nnz : 1, 0);
  for (int r = 0; r < neq; r++)
    std::copy(cols[r].begin(), cols[r].end(), colind.begin() + rowptr[r]);
  return IFEM_GPU_OK;
}

// Positions of every (local row, valid window column) of each patch in the
// shared CSR, in the order the line kernels visit them (window offsets
// (dk, dj, di) ascending, components minor), found once by binary search.
int sub_position_maps(Context& c, std::vector<SubPatch>& subs, const std::vector<int64_t>& rowptr,
                      const std::vector<int32_t>& colind)
{
  const int nc = c.ncomp;
  for (SubPatch& sp : subs) {
    const PatchRec& P = c.patches[sp.patch];
    const int p = P.p[0], n1 = P.n[0], n2 = P.n[1], n3 = P.n[2];
    const int64_t nd = (int64_t)n1 * n2 * n3 * nc;
    std::vector<int64_t> pptr(nd + 1, 0), pmap;
    for (int k = 0; k < n3; k++)
      for (int j = 0; j < n2; j++)
        for (int i = 0; i < n1; i++) {
          const int node = i + n1 * (j + n2 * k);
          for (int ci = 0; ci < nc; ci++) {
            const int64_t d = (int64_t)node * nc + ci;
            const int r = sp.h_leq[d];
            if (r >= 0) {
              const int32_t* rb = colind.data() + rowptr[r];
              const int32_t* re = colind.data() + rowptr[r + 1];
              for (int kk = k - p; kk <= k + p; kk++)
                for (int jj = j - p; jj <= j + p; jj++)
                  for (int ii = i - p; ii <= i + p; ii++) {
                    if (ii < 0 || ii >= n1 || jj < 0 || jj >= n2 || kk < 0 || kk >= n3) continue;
                    const int nb = ii + n1 * (jj + n2 * kk);
                    for (int cj = 0; cj < nc; cj++) {
                      const int e = sp.h_leq[(int64_t)nb * nc + cj];
                      if (e < 0) continue;
                      const int32_t* f = std::lower_bound(rb, re, e);
                      if (f == re || *f != e)
                        return fail(IFEM_GPU_EINVAL, "pattern: column missing from the union row");
                      pmap.push_back(rowptr[r] + (f - rb));
                    }
                  }
            }
            pptr[d + 1] = (int64_t)pmap.size();
          }
        }
    hipFree(sp.d_pmap);
    hipFree(sp.d_pptr);
    sp.d_pmap = sp.d_pptr = nullptr;
    IFEM_HIP(hipMalloc(&sp.d_pptr, sizeof(int64_t) * pptr.size()));
    IFEM_HIP(hipMemcpy(sp.d_pptr, pptr.data(), sizeof(int64_t) * pptr.size(), hipMemcpyHostToDevice));
    IFEM_HIP(hipMalloc(&sp.d_pmap, sizeof(int64_t) * (pmap.empty() ? 1 : pmap.size())));
    if (!pmap.empty())
      IFEM_HIP(hipMemcpy(sp.d_pmap, pmap.data(), sizeof(int64_t) * pmap.size(), hipMemcpyHostToDevice));
  }
  return IFEM_GPU_OK;
}

int device_union_pattern(Context& c, std::vector<SubPatch>& subs, int neq, int64_t** rowptr_out,
                         int32_t** colind_out, int64_t* nnz_out);

// Several patches sharing nodes: the union pattern and the per-patch
// position maps are built on the device (pattern.hip).
static int build_pattern_multi(Context& c)
{
  const int neq = c.neq;
  int64_t* rowptr = nullptr;
  int32_t* colind = nullptr;
  int64_t nnz = 0;
  int rc0 = device_union_pattern(c, c.multi, neq, &rowptr, &colind, &nnz);
  if (rc0) return rc0;
  hipFree(c.d_rowptr);
  hipFree(c.d_colind);
  hipFree(c.d_val);
  hipFree(c.d_val32);
  hipFree(c.d_rhs);
  c.d_rowptr = rowptr;
  c.d_colind = colind;
  c.d_val = nullptr;
  c.d_val32 = nullptr;
  c.d_rhs = nullptr;
  c.fp64_ready = c.fp32_ready = false;
  c.nnz = nnz;
  IFEM_HIP(hipMalloc(&c.d_val, sizeof(double) * (nnz > 0 ? nnz : 1)));
  IFEM_HIP(hipMalloc(&c.d_rhs, sizeof(double) * (neq > 0 ? neq : 1)));
  IFEM_HIP(hipMemsetAsync(c.d_rhs, 0, sizeof(double) * (neq > 0 ? neq : 1), c.stream));
  IFEM_HIP(hipStreamSynchronize(c.stream));
  c.pattern_ready = true;
  return solver_setup(c);
}

int build_pattern(Context& c)
{
  if (c.mpc) return mpc_build_pattern(c);
  if (!c.multi.empty()) return build_pattern_multi(c);
  const PatchRec& P = c.patches[c.patch];
  if (P.p[0] != P.p[1] || P.p[0] != P.p[2])
    return fail(IFEM_GPU_EUNSUPPORTED, "init_assembly: the GPU path needs equal degrees in all directions");
  const int p = P.p[0];
  hipFree(c.d_rowptr);
  hipFree(c.d_colind);
  hipFree(c.d_val);
  hipFree(c.d_val32);
  hipFree(c.d_rhs);
  c.d_rowptr = nullptr;
  c.d_colind = nullptr;
  c.d_val = nullptr;
  c.d_val32 = nullptr;
  c.d_rhs = nullptr;
  c.fp64_ready = c.fp32_ready = false;
  const int neq = c.neq;
  int64_t* rowlen = nullptr;
  int64_t* bsum = nullptr;
  const int nb = (neq + kScanBlock - 1) / kScanBlock;
  IFEM_HIP(hipMalloc(&c.d_rowptr, sizeof(int64_t) * (neq + 1)));
  IFEM_HIP(hipMalloc(&rowlen, sizeof(int64_t) * (neq > 0 ? neq : 1)));
  IFEM_HIP(hipMalloc(&bsum, sizeof(int64_t) * (nb > 0 ? nb : 1)));
  IFEM_HIP(hipMemsetAsync(c.d_rowptr, 0, sizeof(int64_t) * (neq + 1), c.stream));
  if (neq > 0) {
    k_row_lengths<<<(c.ndof + 255) / 256, 256, 0, c.stream>>>(P.n[0], P.n[1], P.n[2], p, c.ncomp,
                                                              c.d_eq, rowlen, c.ndof);
    k_scan_local<<<nb, kScanBlock, 0, c.stream>>>(rowlen, c.d_rowptr, bsum, neq);
    k_scan_sums<<<1, 64, 0, c.stream>>>(bsum, nb);
    k_scan_add<<<nb, kScanBlock, 0, c.stream>>>(c.d_rowptr, bsum, neq);
  }
  IFEM_HIP(hipGetLastError());
  int64_t nnz = 0;
  IFEM_HIP(hipMemcpyAsync(&nnz, c.d_rowptr + neq, sizeof(int64_t), hipMemcpyDeviceToHost, c.stream));
  IFEM_HIP(hipStreamSynchronize(c.stream));
  hipFree(rowlen);
  hipFree(bsum);
  c.nnz = nnz;
  IFEM_HIP(hipMalloc(&c.d_colind, sizeof(int32_t) * (nnz > 0 ? nnz : 1)));
  if (neq > 0) {
    const int waves = 4;
    k_fill_columns<<<(c.ndof + waves - 1) / waves, 64 * waves, 0, c.stream>>>(
        P.n[0], P.n[1], P.n[2], p, c.ncomp, c.d_eq, c.d_rowptr, c.d_colind, c.ndof);
  }
  IFEM_HIP(hipGetLastError());
  IFEM_HIP(hipMalloc(&c.d_val, sizeof(double) * (nnz > 0 ? nnz : 1)));
  IFEM_HIP(hipMalloc(&c.d_rhs, sizeof(double) * (neq > 0 ? neq : 1)));
  IFEM_HIP(hipMemsetAsync(c.d_rhs, 0, sizeof(double) * (neq > 0 ? neq : 1), c.stream));
  IFEM_HIP(hipStreamSynchronize(c.stream));
  c.pattern_ready = true;
  return solver_setup(c);
}

// ---------------------------------------------------------------------------
// Host dispatch of the numeric assembly.
// Basis tables of patch Pt for ng Gauss points per direction (owned by the
// context's cache; built by k_basis_tables on first use).
using Tables = Context::BasisTables;

template <int P>
static int make_tables(Context& c, const PatchRec& Pt, int ng, Tables& tb, GaussArgs& ga)
{
  for (const Tables& t : c.basis_cache)
    if (t.knots0 == Pt.d_knots[0] && t.ng == ng) {
      tb = t;
      return IFEM_GPU_OK;
    }
  Tables t;
  t.knots0 = Pt.d_knots[0];
  t.ng = ng;
  for (int d = 0; d < 3; d++) {
    const size_t cnt = (size_t)Pt.nel[d] * ng * (P + 1);
    if (hipMalloc(&t.tabN[d], sizeof(double) * cnt) != hipSuccess ||
        hipMalloc(&t.tabD[d], sizeof(double) * cnt) != hipSuccess ||
        hipMalloc(&t.span[d], sizeof(double) * Pt.nel[d]) != hipSuccess) {
      for (int e = 0; e <= d; e++) {
        hipFree(t.tabN[e]);
        hipFree(t.tabD[e]);
        hipFree(t.span[e]);
      }
      return fail(IFEM_GPU_EDEVICE, "assemble: out of device memory for the basis tables");
    }
  }
  for (int d = 0; d < 3; d++) {
    const int tot = Pt.nel[d] * ng;
    k_basis_tables<P><<<(tot + 127) / 128, 128, 0, c.stream>>>(Pt.d_knots[d], Pt.nel[d], ng, ga,
                                                              t.tabN[d], t.tabD[d], t.span[d]);
  }
  c.basis_cache.push_back(t);
  tb = t;
  IFEM_HIP(hipGetLastError());
  return IFEM_GPU_OK;
}

// slot: 0 conductivity, 1 source, 2 exact solution (one device buffer each,
// reused by later calls on the same stream)
static int upload_function(Context& c, const ifem_gpu_function& f, DevFunction& df, int slot)
{
  df.type = f.type;
  df.nmodes = f.nmodes;
  df.scale = f.scale;
  df.mean = f.mean;
  df.modes = nullptr;
  if (f.type < 0 || f.type > IFEM_GPU_FN_EXP_FOURIER)
    return fail(IFEM_GPU_EINVAL, "assemble: unknown field type");
  if ((f.type == IFEM_GPU_FN_FOURIER || f.type == IFEM_GPU_FN_EXP_FOURIER) && f.nmodes > 0) {
    if (!f.modes) return fail(IFEM_GPU_EINVAL, "assemble: null mode table");
    const size_t need = (size_t)5 * f.nmodes;
    if (c.modes_cap[slot] < need) {
      hipFree(c.d_modes[slot]);
      c.d_modes[slot] = nullptr;
      c.modes_cap[slot] = 0;
      IFEM_HIP(hipMalloc(&c.d_modes[slot], sizeof(double) * need));
      c.modes_cap[slot] = need;
    }
    double* d = c.d_modes[slot];
    IFEM_HIP(hipMemcpyAsync(d, f.modes, sizeof(double) * need, hipMemcpyHostToDevice, c.stream));
    df.modes = d;
    mode_bounds(f.modes, f.nmodes, df.kbound, df.pbound);
  } else {
    df.nmodes = 0;
  }
  return IFEM_GPU_OK;
}

// Work-split variant of the line kernels for (p, ng, ncomp, precision): the
// tuned (or set) choice if ifem_gpu_autotune_assembly or
// ifem_gpu_set_assembly_variant ran, else -1 (the built-in choice).
int& asm_half_slot(Context& c, int p, int ng, int nc, bool fp32)
{
  return c.asm_half[p][ng > p + 1 ? 1 : 0][nc == 3 ? 1 : 0][fp32 ? 1 : 0];
}

// Vector problems that the direct line kernels assemble (lines2.hip, lines3.hip).
static bool direct_lines(int p, int ng, bool fp32)
{
  return p == 3 || (p == 2 && (ng == 4 || fp32));
}

// The line kernels of degree p with ng Gauss points per direction
// (lines1.hip .. lines3.hip).
static int launch_lines(Context& c, const AsmArgs& args, int p, int ng, bool fp32, bool has_rhs)
{
  if (ng != p + 1 && ng != p + 2)
    return fail(IFEM_GPU_EUNSUPPORTED, "assemble: the GPU path supports ng = p+1 or p+2");
  const int v = asm_half_slot(c, p, ng, c.ncomp, fp32);
  switch (p) {
  case 1: return launch_lines1(c, args, ng, fp32, has_rhs, v);
  case 2: return launch_lines2(c, args, ng, fp32, has_rhs, v);
  default: return launch_lines3(c, args, ng, fp32, has_rhs, v);
  }
}

// The undivided-line variant exists for p <= 2 with at most 3x3x3 points.
static inline bool whole_variant_ok(int p, int ng) { return p <= 2 && ng * ng * ng <= 27; }

// One patch: Pt with eq (local DOF -> equation or -1) and gval (local DOF
// -> prescribed value, or nullptr).  accum: the system holds several
// patches; values and right-hand side are added (zeroed by the caller).
template <int P>
static int assemble_p(Context& c, const SysView& sv, const PatchRec& Pt, const int* eq,
                      const double* gval, int accum, const int64_t* pmap, const int64_t* pptr,
                      const ifem_gpu_integrand& itg, int ng, int precision)
{
  GaussArgs ga{};
  gauss_rule(ng, ga.xi, ga.w);
  Tables tb;
  int rc = make_tables<P>(c, Pt, ng, tb, ga);
  if (rc) return rc;
  AsmArgs a{};
  a.n1 = Pt.n[0];
  a.n2 = Pt.n[1];
  a.n3 = Pt.n[2];
  a.nel1 = Pt.nel[0];
  a.nel2 = Pt.nel[1];
  a.nel3 = Pt.nel[2];
  a.coefs = Pt.d_coefs;
  a.tabN1 = tb.tabN[0]; a.tabD1 = tb.tabD[0]; a.span1 = tb.span[0];
  a.tabN2 = tb.tabN[1]; a.tabD2 = tb.tabD[1]; a.span2 = tb.span[1];
  a.tabN3 = tb.tabN[2]; a.tabD3 = tb.tabD[2]; a.span3 = tb.span[2];
  for (int g = 0; g < kMaxNG; g++) a.gw[g] = ga.w[g];
  a.eq = eq;
  a.rowptr = sv.rowptr;
  a.colind = sv.colind;
  a.accum = accum;
  a.pmap = accum ? pmap : nullptr;
  a.pptr = accum ? pptr : nullptr;
  const bool fp32 = precision == IFEM_GPU_FP32;
  if (fp32) {
    a.val32 = sv.val32;
    a.val64 = nullptr;
    a.rhs = nullptr;
  } else {
    a.val64 = sv.val;
    a.val32 = nullptr;
    a.rhs = sv.rhs;
    a.gval = gval;
  }
  rc = upload_function(c, itg.kappa, a.kappa, 0);
  if (!rc) rc = upload_function(c, itg.source, a.source, 1);
  if (rc) return rc;
  for (int i = 0; i < 3; i++) a.body[i] = itg.body[i];
  if (itg.kind == IFEM_GPU_ELASTICITY) {
    a.lam = itg.E * itg.nu / ((1.0 + itg.nu) * (1.0 - 2.0 * itg.nu));
    a.mu = itg.E / (2.0 * (1.0 + itg.nu));
  }
  bool has_rhs = false;
  if (!fp32) {
    if (c.ncomp == 1) has_rhs = itg.source.type != IFEM_GPU_FN_ZERO;
    else has_rhs = itg.body[0] != 0.0 || itg.body[1] != 0.0 || itg.body[2] != 0.0;
    if (!accum)
      IFEM_HIP(hipMemsetAsync(sv.rhs, 0, sizeof(double) * (sv.neq > 0 ? sv.neq : 1), c.stream));
  }
  // geometry records of all (element, Gauss point) pairs, then the lines
  a.ng = ng;
  a.ncomp = c.ncomp;
  a.kappa_c = const_value(itg.kappa, 1.0);
  a.source_c = const_value(itg.source, 0.0);
  const int64_t ngp = (int64_t)Pt.nel[0] * Pt.nel[1] * Pt.nel[2] * ng * ng * ng;
  const size_t need = (size_t)(ngp > 0 ? ngp : 1) * (c.ncomp == 3 ? GeoRec<3>::N : GeoRec<1>::N);
  if (c.gpgeo_cap < need) {
    hipFree(c.d_gpgeo);
    c.d_gpgeo = nullptr;
    c.gpgeo_cap = 0;
    IFEM_HIP(hipMalloc(&c.d_gpgeo, sizeof(double) * need));
    c.gpgeo_cap = need;
  }
  a.gp_geo = c.d_gpgeo;
  a.geo_pairs = c.ncomp == 3 && direct_lines(P, ng, fp32);
  if (!c.d_asmargs) IFEM_HIP(hipMalloc(&c.d_asmargs, sizeof(AsmArgs)));
  IFEM_HIP(hipMemcpyAsync(c.d_asmargs, &a, sizeof(AsmArgs), hipMemcpyHostToDevice, c.stream));
  IFEM_HIP(hipEventRecord(c.ev0, c.stream));
  if (ngp > 0 && c.ncomp == 3)
    k_gp_geometry_vec<P><<<grid_for(ngp), 256, 0, c.stream>>>(
        static_cast<const AsmArgs*>(c.d_asmargs), ngp);
  else if (ngp > 0)
    k_gp_geometry<P><<<grid_for(ngp), 256, 0, c.stream>>>(static_cast<const AsmArgs*>(c.d_asmargs),
                                                         ngp, has_rhs ? 1 : 0);
  IFEM_HIP(hipEventRecord(c.ev_mid, c.stream));
  rc = launch_lines(c, a, P, ng, fp32, has_rhs);
  if (rc) return rc;
  IFEM_HIP(hipEventRecord(c.ev1, c.stream));
  IFEM_HIP(hipEventSynchronize(c.ev1));
  float ms = 0.f, ms_geo = 0.f;
  IFEM_HIP(hipEventElapsedTime(&ms, c.ev0, c.ev1));
  IFEM_HIP(hipEventElapsedTime(&ms_geo, c.ev0, c.ev_mid));
  c.last_assemble_ms = ms;
  c.last_geometry_ms = ms_geo;
  c.last_lines_ms = ms - ms_geo;
  return IFEM_GPU_OK;
}

int set_assembly_variant(Context& c, int p, int ng, int nc, bool fp32, int variant)
{
  if (variant < -1 || variant > 2 || (variant == 2 && !whole_variant_ok(p, ng)))
    return fail(IFEM_GPU_EUNSUPPORTED, "set_assembly_variant: no such variant for this degree and rule");
  asm_half_slot(c, p, ng, nc, fp32) = variant;
  return IFEM_GPU_OK;
}

// Times the work splits of the line kernels on this system and keeps the
// fastest for (p, ng, ncomp, precision); the system is left assembled with
// the chosen variant.
int autotune_assembly(Context& c, const ifem_gpu_integrand& itg, const int ng[3], int precision,
                      int* half_out)
{
  const PatchRec& Pt = c.patches[c.patch];
  const bool fp32 = precision == IFEM_GPU_FP32;
  if (ng[0] < 1 || ng[0] > kMaxNG) return fail(IFEM_GPU_EUNSUPPORTED, "autotune: ng out of range");
  int& slot = asm_half_slot(c, Pt.p[0], ng[0], c.ncomp, fp32);
  double best = 1e300;
  int best_h = 0;
  const int hmax = whole_variant_ok(Pt.p[0], ng[0]) ? 2 : 1;
  for (int h = 0; h <= hmax; h++) {
    slot = h;
    double t = 1e300;
    for (int rep = 0; rep < 3; rep++) {
      int rc = assemble_volume(c, itg, ng, precision);
      if (rc) return rc;
      t = std::fmin(t, c.last_assemble_ms);
    }
    if (t < best) {
      best = t;
      best_h = h;
    }
  }
  slot = best_h;
  if (half_out) *half_out = best_h;
  return assemble_volume(c, itg, ng, precision);
}

static int assemble_one(Context& c, const SysView& sv, const PatchRec& Pt, const int* eq,
                        const double* gval, int accum, const ifem_gpu_integrand& itg, int ng,
                        int precision, const int64_t* pmap = nullptr,
                        const int64_t* pptr = nullptr)
{
  switch (Pt.p[0]) {
  case 1: return assemble_p<1>(c, sv, Pt, eq, gval, accum, pmap, pptr, itg, ng, precision);
  case 2: return assemble_p<2>(c, sv, Pt, eq, gval, accum, pmap, pptr, itg, ng, precision);
  case 3: return assemble_p<3>(c, sv, Pt, eq, gval, accum, pmap, pptr, itg, ng, precision);
  default: return fail(IFEM_GPU_EUNSUPPORTED, "assemble: degree out of range");
  }
}

// Patches added one after the other into the zeroed system sv.
static int assemble_sum(Context& c, SysView& sv, const std::vector<SubPatch>& subs,
                        const ifem_gpu_integrand& itg, int ng, int precision)
{
  const bool fp32 = precision == IFEM_GPU_FP32;
  const size_t nz = (size_t)(sv.nnz > 0 ? sv.nnz : 1);
  if (fp32) {
    IFEM_HIP(hipMemsetAsync(sv.val32, 0, sizeof(float) * nz, c.stream));
  } else {
    IFEM_HIP(hipMemsetAsync(sv.val, 0, sizeof(double) * nz, c.stream));
    IFEM_HIP(hipMemsetAsync(sv.rhs, 0, sizeof(double) * (sv.neq > 0 ? sv.neq : 1), c.stream));
  }
  double tot = 0.0, geo = 0.0;
  for (const SubPatch& sp : subs) {
    int rc = assemble_one(c, sv, c.patches[sp.patch], sp.d_leq, sp.d_lgval, 1, itg, ng, precision,
                          sp.d_pmap, sp.d_pptr);
    if (rc) return rc;
    tot += c.last_assemble_ms;
    geo += c.last_geometry_ms;
  }
  c.last_assemble_ms = tot;
  c.last_geometry_ms = geo;
  c.last_lines_ms = tot - geo;
  return IFEM_GPU_OK;
}

int assemble_volume(Context& c, const ifem_gpu_integrand& itg, const int ng[3], int precision)
{
  if (ng[0] != ng[1] || ng[0] != ng[2])
    return fail(IFEM_GPU_EUNSUPPORTED, "assemble: the GPU path needs equal Gauss counts per direction");
  if (ng[0] < 1 || ng[0] > kMaxNG) return fail(IFEM_GPU_EUNSUPPORTED, "assemble: ng out of range");
  const bool fp32 = precision == IFEM_GPU_FP32;
  if (fp32 && !c.d_val32)
    IFEM_HIP(hipMalloc(&c.d_val32, sizeof(float) * (c.nnz > 0 ? c.nnz : 1)));
  SysView sv{c.d_rowptr, c.d_colind, c.d_val, c.d_val32, c.d_rhs, c.nnz, c.neq};
  if (c.mpc) {
    // constraint equations with masters: the extended system (slaves as
    // unknowns) is assembled, then condensed to the free equations
    MpcSystem& x = *c.mpc;
    if (fp32 && !x.d_val32)
      IFEM_HIP(hipMalloc(&x.d_val32, sizeof(float) * (x.nnz > 0 ? x.nnz : 1)));
    SysView xv{x.d_rowptr, x.d_colind, x.d_val, x.d_val32, x.d_rhs, x.nnz, x.ne};
    // a shallow copy: x.ext owns the device arrays (SubPatch frees nothing)
    std::vector<SubPatch> subs(1, x.ext);
    int rc = assemble_sum(c, xv, subs, itg, ng[0], precision);
    if (rc) return rc;
    rc = mpc_condense(c, fp32, false);
    if (rc) return rc;
  } else if (c.multi.empty()) {
    int rc = assemble_one(c, sv, c.patches[c.patch], c.d_eq, c.d_gval, 0, itg, ng[0], precision);
    if (rc) return rc;
  } else {
    int rc = assemble_sum(c, sv, c.multi, itg, ng[0], precision);
    if (rc) return rc;
  }
  if (fp32) c.fp32_ready = true;
  else c.fp64_ready = true;
  return IFEM_GPU_OK;
}

// ---------------------------------------------------------------------------
// Neumann traction on one face: one thread per (face node, component); sums
// over the face elements holding the node and their ng x ng Gauss points in
// fixed order (src/ASM/ASMs3D.C:2547-2812; face utl::Jacobian,
// src/Utility/CoordinateMapping.C:90-133: dS = |J_t1 x J_t2|, zero if J is
// singular; detJxW = dS * dA * w_i * w_j with dA = 0.25 * area).
// Pass 1: one thread per (face element, Gauss point): w = dS * dA * w_i * w_j
// (0 where J is singular), face element (ea, eb) along the tangent
// directions, w[((eb*nel_ta + ea)*ng + gb)*ng + ga].
template <int P>
__global__ void k_traction_w(int n1, int n2, int n3, int nel1, int nel2, int nel3,
                             const double* __restrict__ coefs, const double* k1,
                             const double* k2, const double* k3, int face, int ng, GaussArgs ga,
                             double* __restrict__ wout)
{
  constexpr int P1 = P + 1;
  const int dn = face / 2, side = face % 2;
  const int n[3] = {n1, n2, n3}, nel[3] = {nel1, nel2, nel3};
  const double* kn[3] = {k1, k2, k3};
  const int ta = dn == 0 ? 1 : 0, tb = dn == 2 ? 1 : 2; // tangent directions, ascending
  const int id = blockIdx.x * blockDim.x + threadIdx.x;
  const int ntot = nel[ta] * nel[tb] * ng * ng;
  if (id >= ntot) return;
  const int gA = id % ng, gb = (id / ng) % ng, fe = id / (ng * ng);
  const int ea = fe % nel[ta], eb = fe / nel[ta];
  // faceDir = +-(dn+1): t1 = 1 + |faceDir| % 3, t2 = 1 + t1 % 3 (1-based)
  const int T1 = (dn + 1) % 3, T2 = (T1 + 1) % 3;
  int e[3];
  e[dn] = side ? nel[dn] - 1 : 0;
  e[ta] = ea;
  e[tb] = eb;
  double spn[3];
  for (int d = 0; d < 3; d++) spn[d] = kn[d][e[d] + P + 1] - kn[d][e[d] + P];
  const double dA = 0.25 * (spn[ta] * spn[tb]);
  double Nd[3][P1], dNd[3][P1];
  for (int d = 0; d < 3; d++) {
    const int s = e[d] + P;
    const double* kt = kn[d];
    double u;
    if (d == dn) u = side ? kt[n[d]] : kt[P];
    else {
      const double xi = ga.xi[d == ta ? gA : gb];
      u = 0.5 * ((kt[s + 1] - kt[s]) * xi + kt[s + 1] + kt[s]);
    }
    bspline_1d<P>(kt, s, u, Nd[d], dNd[d]);
  }
  double J[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  for (int b3 = 0; b3 < P1; b3++)
    for (int b2 = 0; b2 < P1; b2++)
      for (int b1 = 0; b1 < P1; b1++) {
        const int64_t nb = (int64_t)(e[0] + b1) + (int64_t)n1 * ((e[1] + b2) + (int64_t)n2 * (e[2] + b3));
        const double g0 = dNd[0][b1] * Nd[1][b2] * Nd[2][b3];
        const double g1 = Nd[0][b1] * dNd[1][b2] * Nd[2][b3];
        const double g2 = Nd[0][b1] * Nd[1][b2] * dNd[2][b3];
        for (int i = 0; i < 3; i++) {
          const double x = coefs[3 * nb + i];
          J[3 * i + 0] += x * g0;
          J[3 * i + 1] += x * g1;
          J[3 * i + 2] += x * g2;
        }
      }
  const double v1[3] = {J[T1], J[3 + T1], J[6 + T1]};
  const double v2[3] = {J[T2], J[3 + T2], J[6 + T2]};
  const double nx = v1[1] * v2[2] - v1[2] * v2[1];
  const double ny = v1[2] * v2[0] - v1[0] * v2[2];
  const double nz = v1[0] * v2[1] - v1[1] * v2[0];
  double dS = sqrt(nx * nx + ny * ny + nz * nz);
  const double det = J[0] * (J[4] * J[8] - J[7] * J[5]) - J[1] * (J[3] * J[8] - J[6] * J[5]) +
                     J[2] * (J[3] * J[7] - J[6] * J[4]);
  if (det <= 1e-12 && det >= -1e-12) dS = 0.0;
  wout[id] = dS == 0.0 ? 0.0 : dS * (dA * ga.w[gA] * ga.w[gb]);
}

// Pass 2: one thread per face node sums w * N_a over the face elements and
// Gauss points holding it (fixed order), then adds t_c times the sum to the
// node's free components.
template <int P>
__global__ void k_traction_sum(int n1, int n2, int n3, int nel1, int nel2, int nel3,
                               const double* k1, const double* k2, const double* k3, int face,
                               int ng, GaussArgs ga, const double* __restrict__ wf, double t0,
                               double t1, double t2, int nc, const int* __restrict__ eq,
                               double* __restrict__ rhs)
{
  constexpr int P1 = P + 1;
  const int dn = face / 2, side = face % 2;
  const int n[3] = {n1, n2, n3}, nel[3] = {nel1, nel2, nel3};
  const double* kn[3] = {k1, k2, k3};
  const int ta = dn == 0 ? 1 : 0, tb = dn == 2 ? 1 : 2;
  const int id = blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= n[ta] * n[tb]) return;
  const int ia = id % n[ta], ib = id / n[ta];
  int idx[3];
  idx[dn] = side ? n[dn] - 1 : 0;
  idx[ta] = ia;
  idx[tb] = ib;
  const int64_t node = (int64_t)idx[0] + (int64_t)n1 * (idx[1] + (int64_t)n2 * idx[2]);
  // basis value of the node in the normal direction on the face
  const int en = side ? nel[dn] - 1 : 0;
  double Nn[P1], dNn[P1];
  {
    const double* kt = kn[dn];
    bspline_1d<P>(kt, en + P, side ? kt[n[dn]] : kt[P], Nn, dNn);
  }
  const double nface = Nn[idx[dn] - en];
  double sum = 0.0;
  for (int eb = max(0, ib - P); eb <= min(nel[tb] - 1, ib); eb++)
    for (int ea = max(0, ia - P); ea <= min(nel[ta] - 1, ia); ea++) {
      const double* w = wf + (int64_t)(eb * nel[ta] + ea) * ng * ng;
      for (int gb = 0; gb < ng; gb++) {
        double Nb[P1], dNb[P1];
        const double* kb = kn[tb];
        const int sb = eb + P;
        bspline_1d<P>(kb, sb, 0.5 * ((kb[sb + 1] - kb[sb]) * ga.xi[gb] + kb[sb + 1] + kb[sb]), Nb,
                      dNb);
        for (int gA = 0; gA < ng; gA++) {
          const double wg = w[gb * ng + gA];
          if (wg == 0.0) continue;
          double Na[P1], dNa[P1];
          const double* ka = kn[ta];
          const int sa = ea + P;
          bspline_1d<P>(ka, sa, 0.5 * ((ka[sa + 1] - ka[sa]) * ga.xi[gA] + ka[sa + 1] + ka[sa]),
                        Na, dNa);
          sum += wg * (Na[ia - ea] * Nb[ib - eb] * nface);
        }
      }
    }
  const double tv[3] = {t0, t1, t2};
  for (int c = 0; c < nc; c++) {
    const int r = eq[node * nc + c];
    if (r >= 0) rhs[r] += tv[c] * sum;
  }
}

int assemble_traction(Context& c, int index, int face0, const double* t, int ng)
{
  if (index < 0 || index >= (c.multi.empty() ? 1 : (int)c.multi.size()))
    return fail(IFEM_GPU_EINVAL, "traction: patch index out of range");
  const PatchRec& Pt = c.patches[c.multi.empty() ? c.patch : c.multi[index].patch];
  const int* eqmap = c.multi.empty() ? c.d_eq : c.multi[index].d_leq;
  double* rhs = c.d_rhs;
  if (c.mpc) { // into the extended right-hand side, condensed below
    if (!c.fp64_ready)
      return fail(IFEM_GPU_EINVAL,
                  "assemble_neumann: constraints with masters need the FP64 system first");
    eqmap = c.mpc->ext.d_leq;
    rhs = c.mpc->d_rhs;
  }
  GaussArgs ga{};
  gauss_rule(ng, ga.xi, ga.w);
  const int dn = face0 / 2;
  const int ta = dn == 0 ? 1 : 0, tb = dn == 2 ? 1 : 2;
  const int nfn = Pt.n[ta] * Pt.n[tb];
  const int nw = Pt.nel[ta] * Pt.nel[tb] * ng * ng;
  const double t1 = c.ncomp > 1 ? t[1] : 0.0, t2 = c.ncomp > 2 ? t[2] : 0.0;
  if (c.facew_cap < (size_t)nw) {
    hipFree(c.d_facew);
    c.d_facew = nullptr;
    c.facew_cap = 0;
    IFEM_HIP(hipMalloc(&c.d_facew, sizeof(double) * (nw > 0 ? nw : 1)));
    c.facew_cap = nw;
  }
#define LAUNCH_TR(PP)                                                                          \
  k_traction_w<PP><<<(nw + 255) / 256, 256, 0, c.stream>>>(                                     \
      Pt.n[0], Pt.n[1], Pt.n[2], Pt.nel[0], Pt.nel[1], Pt.nel[2], Pt.d_coefs, Pt.d_knots[0],    \
      Pt.d_knots[1], Pt.d_knots[2], face0, ng, ga, c.d_facew);                                  \
  k_traction_sum<PP><<<(nfn + 127) / 128, 128, 0, c.stream>>>(                                  \
      Pt.n[0], Pt.n[1], Pt.n[2], Pt.nel[0], Pt.nel[1], Pt.nel[2], Pt.d_knots[0], Pt.d_knots[1], \
      Pt.d_knots[2], face0, ng, ga, c.d_facew, t[0], t1, t2, c.ncomp, eqmap, rhs)
  switch (Pt.p[0]) {
  case 1: LAUNCH_TR(1); break;
  case 2: LAUNCH_TR(2); break;
  case 3: LAUNCH_TR(3); break;
  default: return fail(IFEM_GPU_EUNSUPPORTED, "traction: degree out of range");
  }
#undef LAUNCH_TR
  IFEM_HIP(hipGetLastError());
  if (c.mpc) {
    int rc = mpc_condense(c, false, true);
    if (rc) return rc;
  }
  IFEM_HIP(hipStreamSynchronize(c.stream));
  return IFEM_GPU_OK;
}

// ---------------------------------------------------------------------------
// Batch of independent scalar patches (block-diagonal global system).  Each
// patch is integrated as SIMbase::assembleSystem does per patch
// (src/SIM/SIMbase.C:1229-1400), but every patch has its own equations and
// all patches go through one persistent launch.

static int batch_tables(Context& c, const PatchRec& Pt, BatchPatch& bp)
{
  GaussArgs ga{};
  gauss_rule(bp.ng, ga.xi, ga.w);
  for (int d = 0; d < 3; d++) {
    const size_t cnt = (size_t)Pt.nel[d] * bp.ng * (bp.p + 1);
    IFEM_HIP(hipMalloc(&bp.tabN[d], sizeof(double) * cnt));
    IFEM_HIP(hipMalloc(&bp.tabD[d], sizeof(double) * cnt));
    IFEM_HIP(hipMalloc(&bp.span[d], sizeof(double) * Pt.nel[d]));
    const int tot = Pt.nel[d] * bp.ng;
    const dim3 g((tot + 127) / 128), b(128);
    switch (bp.p) {
    case 1: k_basis_tables<1><<<g, b, 0, c.stream>>>(Pt.d_knots[d], Pt.nel[d], bp.ng, ga, bp.tabN[d], bp.tabD[d], bp.span[d]); break;
    case 2: k_basis_tables<2><<<g, b, 0, c.stream>>>(Pt.d_knots[d], Pt.nel[d], bp.ng, ga, bp.tabN[d], bp.tabD[d], bp.span[d]); break;
    default: k_basis_tables<3><<<g, b, 0, c.stream>>>(Pt.d_knots[d], Pt.nel[d], bp.ng, ga, bp.tabN[d], bp.tabD[d], bp.span[d]); break;
    }
  }
  IFEM_HIP(hipGetLastError());
  return IFEM_GPU_OK;
}

static DevFunction batch_function(const ifem_gpu_function& f, const double* d_modes)
{
  DevFunction df;
  df.type = f.type;
  df.nmodes = d_modes ? f.nmodes : 0;
  df.scale = f.scale;
  df.mean = f.mean;
  df.modes = d_modes;
  if (d_modes && f.modes) mode_bounds(f.modes, f.nmodes, df.kbound, df.pbound);
  else df.kbound = df.pbound = 1e300; // unknown: the checked loop
  return df;
}

// Per-patch assembly arguments for both precisions.
int batch_upload_args(Context& c)
{
  Batch& B = *c.batch;
  const int np = (int)B.pp.size();
  std::vector<AsmArgs> a64(np), a32(np);
  for (int q = 0; q < np; q++) {
    const BatchPatch& bp = B.pp[q];
    const PatchRec& Pt = c.patches[bp.patch];
    AsmArgs a{};
    a.n1 = Pt.n[0];
    a.n2 = Pt.n[1];
    a.n3 = Pt.n[2];
    a.nel1 = Pt.nel[0];
    a.nel2 = Pt.nel[1];
    a.nel3 = Pt.nel[2];
    a.coefs = Pt.d_coefs;
    a.tabN1 = bp.tabN[0]; a.tabD1 = bp.tabD[0]; a.span1 = bp.span[0];
    a.tabN2 = bp.tabN[1]; a.tabD2 = bp.tabD[1]; a.span2 = bp.span[1];
    a.tabN3 = bp.tabN[2]; a.tabD3 = bp.tabD[2]; a.span3 = bp.span[2];
    GaussArgs ga{};
    gauss_rule(bp.ng, ga.xi, ga.w);
    for (int g = 0; g < kMaxNG; g++) a.gw[g] = ga.w[g];
    a.eq = bp.d_eq;
    a.rowptr = B.d_rowptr;
    a.kappa = batch_function(bp.itg.kappa, bp.d_kmodes);
    a.source = batch_function(bp.itg.source, bp.d_smodes);
    a.ng = bp.ng;
    a.ncomp = 1;
    const int64_t g0 = B.h_gp0.empty() ? 0 : B.h_gp0[q];
    a.gp_geo = B.d_geo + g0 * GeoRec<1>::N;
    a.kappa_c = const_value(bp.itg.kappa, 1.0);
    a.source_c = const_value(bp.itg.source, 0.0);
    a.val64 = B.d_val;
    a.val32 = nullptr;
    a.rhs = B.d_rhs;
    a64[q] = a;
    a.val64 = nullptr;
    a.val32 = B.d_val32;
    a.rhs = nullptr;
    a32[q] = a;
  }
  if (!B.d_args64) IFEM_HIP(hipMalloc(&B.d_args64, sizeof(AsmArgs) * (np > 0 ? np : 1)));
  if (!B.d_args32) IFEM_HIP(hipMalloc(&B.d_args32, sizeof(AsmArgs) * (np > 0 ? np : 1)));
  IFEM_HIP(hipMemcpy(B.d_args64, a64.data(), sizeof(AsmArgs) * np, hipMemcpyHostToDevice));
  IFEM_HIP(hipMemcpy(B.d_args32, a32.data(), sizeof(AsmArgs) * np, hipMemcpyHostToDevice));
  return IFEM_GPU_OK;
}

// Work list of the line kernels: items are groups of neighbouring lines with a
// segment of their rows (degree 3: whole lines), split so that every degree has
// a few items per workgroup that the chip holds, largest first.  The second
// list (half) has segments of half the length at degrees 1 and 2; it is built
// when the tuner first asks for it.
static int batch_items(Context& c, int half)
{
  Batch& B = *c.batch;
  const int np = (int)B.pp.size();
  struct Item { double cost; LineItem it; };
  std::vector<LineItem> hi;
  for (int p = half ? 2 : 3; p >= 1; p--) {
    const int most = batch_lines_per_item(p);
    int64_t groups = 0;
    for (const BatchPatch& bp : B.pp) {
      const PatchRec& Pt = c.patches[bp.patch];
      if (bp.p == p && bp.neq > 0) groups += (int64_t)((Pt.n[1] + most - 1) / most) * Pt.n[2];
    }
    const int64_t want = groups > 0 ? (4 * B.ncu + groups - 1) / groups : 1; // segments per line
    std::vector<Item> items;
    for (int q = 0; q < np; q++) {
      const BatchPatch& bp = B.pp[q];
      if (bp.p != p || bp.neq == 0) continue;
      const PatchRec& Pt = c.patches[bp.patch];
      const int ngj = (Pt.n[1] + most - 1) / most;
      int nseg = (int)std::min<int64_t>(want, std::max(1, Pt.n[0] / (4 * p)));
      // few groups: down to one row each while every item has a compute
      // unit (8 quadratic patches of 4 to 8 elements, FP32: 75 -> 55 us)
      nseg = std::max(nseg, (int)std::min<int64_t>(Pt.n[0], B.ncu / groups));
      if (half) nseg = std::min(2 * nseg, Pt.n[0]);
      if (p == 3) nseg = 1; // whole lines (direct kernels)
      for (int k = 0; k < Pt.n[2]; k++) {
        const int c3 = std::min(k, Pt.nel[2] - 1) - std::max(0, k - p) + 1;
        for (int g = 0; g < ngj; g++)
          for (int sg = 0; sg < nseg; sg++) {
            const int j0 = (int)((int64_t)Pt.n[1] * g / ngj), j1 = (int)((int64_t)Pt.n[1] * (g + 1) / ngj);
            const int i0 = (int)((int64_t)Pt.n[0] * sg / nseg), i1 = (int)((int64_t)Pt.n[0] * (sg + 1) / nseg);
            const int layers = std::min(i1, Pt.nel[0]) - std::max(0, i0 - p);
            const int c2 = p == 3 ? std::min(j0, Pt.nel[1] - 1) - std::max(0, j0 - p) + 1 : 1;
            items.push_back({(double)layers * c3 * c2, LineItem{q, j0, j1 - j0, k, i0, i1}});
          }
      }
    }
    std::stable_sort(items.begin(), items.end(),
                     [](const Item& x, const Item& y) { return x.cost > y.cost; });
    B.item0[half][p] = (int)hi.size();
    for (const Item& it : items) hi.push_back(it.it);
    B.item1[half][p] = (int)hi.size();
  }
  IFEM_HIP(hipMalloc(&B.d_items[half], sizeof(LineItem) * (hi.empty() ? 1 : hi.size())));
  if (!hi.empty())
    IFEM_HIP(hipMemcpy(B.d_items[half], hi.data(), sizeof(LineItem) * hi.size(), hipMemcpyHostToDevice));
  return IFEM_GPU_OK;
}

// Symbolic phase of the batch: per-patch basis tables, global CSR pattern
// (patch q's rows and columns are its equations shifted by eq0), and the
// (patch, line) work list sorted by decreasing estimated cost.
int batch_symbolic(Context& c)
{
  Batch& B = *c.batch;
  const int np = (int)B.pp.size();
  int eq0 = 0;
  for (BatchPatch& bp : B.pp) {
    bp.eq0 = eq0;
    eq0 += bp.neq;
  }
  B.neq = eq0;
  const int neq = B.neq;
  IFEM_HIP(hipEventRecord(c.ev0, c.stream));
  for (BatchPatch& bp : B.pp) {
    int rc = batch_tables(c, c.patches[bp.patch], bp);
    if (rc) return rc;
  }
  int64_t* rowlen = nullptr;
  int64_t* bsum = nullptr;
  const int nb = (neq + kScanBlock - 1) / kScanBlock;
  IFEM_HIP(hipMalloc(&B.d_rowptr, sizeof(int64_t) * (neq + 1)));
  IFEM_HIP(hipMalloc(&rowlen, sizeof(int64_t) * (neq > 0 ? neq : 1)));
  IFEM_HIP(hipMalloc(&bsum, sizeof(int64_t) * (nb > 0 ? nb : 1)));
  IFEM_HIP(hipMemsetAsync(B.d_rowptr, 0, sizeof(int64_t) * (neq + 1), c.stream));
  for (BatchPatch& bp : B.pp) {
    const PatchRec& Pt = c.patches[bp.patch];
    if (bp.neq > 0)
      k_row_lengths<<<(bp.nnod + 255) / 256, 256, 0, c.stream>>>(Pt.n[0], Pt.n[1], Pt.n[2], bp.p, 1,
                                                                   bp.d_eq, rowlen, bp.nnod);
  }
  if (neq > 0) {
    k_scan_local<<<nb, kScanBlock, 0, c.stream>>>(rowlen, B.d_rowptr, bsum, neq);
    k_scan_sums<<<1, 64, 0, c.stream>>>(bsum, nb);
    k_scan_add<<<nb, kScanBlock, 0, c.stream>>>(B.d_rowptr, bsum, neq);
  }
  IFEM_HIP(hipGetLastError());
  int64_t nnz = 0;
  IFEM_HIP(hipMemcpyAsync(&nnz, B.d_rowptr + neq, sizeof(int64_t), hipMemcpyDeviceToHost, c.stream));
  IFEM_HIP(hipStreamSynchronize(c.stream));
  hipFree(rowlen);
  hipFree(bsum);
  B.nnz = nnz;
  IFEM_HIP(hipMalloc(&B.d_colind, sizeof(int32_t) * (nnz > 0 ? nnz : 1)));
  for (BatchPatch& bp : B.pp) {
    const PatchRec& Pt = c.patches[bp.patch];
    if (bp.neq > 0)
      k_fill_columns<<<(bp.nnod + 3) / 4, 256, 0, c.stream>>>(Pt.n[0], Pt.n[1], Pt.n[2], bp.p, 1,
                                                              bp.d_eq, B.d_rowptr, B.d_colind, bp.nnod);
  }
  IFEM_HIP(hipGetLastError());
  IFEM_HIP(hipMalloc(&B.d_val, sizeof(double) * (nnz > 0 ? nnz : 1)));
  IFEM_HIP(hipMalloc(&B.d_val32, sizeof(float) * (nnz > 0 ? nnz : 1)));
  IFEM_HIP(hipMalloc(&B.d_rhs, sizeof(double) * (neq > 0 ? neq : 1)));
  IFEM_HIP(hipMemsetAsync(B.d_rhs, 0, sizeof(double) * (neq > 0 ? neq : 1), c.stream));

  // geometry records of every patch's (element, Gauss point) pairs
  B.h_gp0.assign(np, 0);
  int64_t ngp = 0;
  for (int q = 0; q < np; q++) {
    const BatchPatch& bp = B.pp[q];
    const PatchRec& Pt = c.patches[bp.patch];
    B.h_gp0[q] = ngp;
    ngp += (int64_t)Pt.nel[0] * Pt.nel[1] * Pt.nel[2] * bp.ng * bp.ng * bp.ng;
  }
  B.ngp = ngp;
  IFEM_HIP(hipMalloc(&B.d_geo, sizeof(double) * GeoRec<1>::N * (ngp > 0 ? ngp : 1)));
  // per degree: its patches and the first point of each among that degree's
  // points (one geometry launch per degree)
  std::vector<int> glist;
  std::vector<int64_t> gq0;
  for (int p = 1; p <= 3; p++) {
    B.gdeg_off[p] = (int)glist.size();
    int64_t t = 0;
    for (int q = 0; q < np; q++) {
      const BatchPatch& bp = B.pp[q];
      if (bp.p != p) continue;
      const PatchRec& Pt = c.patches[bp.patch];
      glist.push_back(q);
      gq0.push_back(t);
      t += (int64_t)Pt.nel[0] * Pt.nel[1] * Pt.nel[2] * bp.ng * bp.ng * bp.ng;
    }
    B.gdeg_n[p] = (int)glist.size() - B.gdeg_off[p];
    B.gdeg_total[p] = t;
  }
  IFEM_HIP(hipMalloc(&B.d_glist, sizeof(int) * (np > 0 ? np : 1)));
  IFEM_HIP(hipMalloc(&B.d_gq0, sizeof(int64_t) * (np > 0 ? np : 1)));
  IFEM_HIP(hipMemcpy(B.d_glist, glist.data(), sizeof(int) * glist.size(), hipMemcpyHostToDevice));
  IFEM_HIP(hipMemcpy(B.d_gq0, gq0.data(), sizeof(int64_t) * gq0.size(), hipMemcpyHostToDevice));

  hipDeviceProp_t prop;
  IFEM_HIP(hipGetDeviceProperties(&prop, c.device));
  B.ncu = prop.multiProcessorCount;
  int rc = batch_items(c, 0);
  if (rc) return rc;
  IFEM_HIP(hipMalloc(&B.d_queue, sizeof(int) * 4));
  rc = batch_upload_args(c);
  if (rc) return rc;
  IFEM_HIP(hipEventRecord(c.ev1, c.stream));
  IFEM_HIP(hipEventSynchronize(c.ev1));
  float ms = 0.f;
  IFEM_HIP(hipEventElapsedTime(&ms, c.ev0, c.ev1));
  B.symbolic_ms = ms;
  return IFEM_GPU_OK;
}

// Numeric assembly of every patch of the batch, one persistent launch per
// degree: FP64 writes K and b, FP32 writes the FP32 copy of K.  Returns the
// device time in *ms.
int batch_assemble(Context& c, int precision, double* ms_out)
{
  Batch& B = *c.batch;
  const bool fp32 = precision == IFEM_GPU_FP32;
  if ((B.tune[1].half || B.tune[2].half) && !B.d_items[1]) {
    const int rc = batch_items(c, 1);
    if (rc) return rc;
  }
  k_fill<int><<<1, 64, 0, c.stream>>>(4, B.d_queue, 0);
  IFEM_HIP(hipEventRecord(c.ev0, c.stream));
  // geometry pass: always for FP64 (the full assembly); an FP32 assembly
  // reuses the records of an earlier assembly of the same batch (the
  // material part of the records is the same in both precisions)
  if (B.ngp > 0 && !(fp32 && B.geo_valid)) {
    const AsmArgs* ga = static_cast<const AsmArgs*>(fp32 ? B.d_args32 : B.d_args64);
    for (int p = 3; p >= 1; p--) {
      const int64_t tot = B.gdeg_total[p];
      if (tot <= 0) continue;
      const int* pl = B.d_glist + B.gdeg_off[p];
      const int64_t* q0 = B.d_gq0 + B.gdeg_off[p];
      if (p == 3)
        k_gp_geometry_batch<3><<<grid_for(tot), 256, 0, c.stream>>>(ga, pl, q0, B.gdeg_n[p], tot, fp32 ? 0 : 1);
      else if (p == 2)
        k_gp_geometry_batch<2><<<grid_for(tot), 256, 0, c.stream>>>(ga, pl, q0, B.gdeg_n[p], tot, fp32 ? 0 : 1);
      else
        k_gp_geometry_batch<1><<<grid_for(tot), 256, 0, c.stream>>>(ga, pl, q0, B.gdeg_n[p], tot, fp32 ? 0 : 1);
    }
  }
  for (int p = 3; p >= 1; p--) {
    const int half = p < 3 && B.tune[p].half ? 1 : 0;
    const int n = B.item1[half][p] - B.item0[half][p];
    if (n <= 0) continue;
    const LineItem* items = static_cast<const LineItem*>(B.d_items[half]) + B.item0[half][p];
    const AsmArgs* args = static_cast<const AsmArgs*>(fp32 ? B.d_args32 : B.d_args64);
    const int rc = p == 3   ? launch_lines_batch3(c, args, items, n, B.d_queue + p, B.ncu, fp32)
                   : p == 2 ? launch_lines_batch2(c, args, items, n, B.d_queue + p, B.ncu, fp32)
                            : launch_lines_batch1(c, args, items, n, B.d_queue + p, B.ncu, fp32);
    if (rc) return rc;
  }
  IFEM_HIP(hipGetLastError());
  IFEM_HIP(hipEventRecord(c.ev1, c.stream));
  IFEM_HIP(hipEventSynchronize(c.ev1));
  float ms = 0.f;
  IFEM_HIP(hipEventElapsedTime(&ms, c.ev0, c.ev1));
  if (ms_out) *ms_out = ms;
  if (fp32) B.fp32_ready = true;
  else B.fp64_ready = true;
  B.geo_valid = true;
  return IFEM_GPU_OK;
}

// ---------------------------------------------------------------------------
// Norms of the current solution, NormBase / ElmNorm / GlbNorm with the SQRT
// final operation (src/ASM/IntegrandBase.h:378-530, src/ASM/GlbNorm.C:33-79):
// one thread per (element, Gauss point) evaluates u_h = sum_b N_b u_b and
// grad u_h = J^-T sum_b u_b grad_ref N_b with the volume loop's quadrature,
// Jacobian and singular-point rule, and accumulates
//   [0] |u_h|^2, [1] energy density of u_h (kappa |grad u_h|^2, or
//   eps:C:eps), and with an exact scalar solution u: [2] u^2, [3] kappa
//   |grad u|^2, [4] (u - u_h)^2, [5] kappa |grad(u - u_h)|^2
// times detJxW, reduced per block in fixed order.
__device__ inline void eval_field_grad(const DevFunction& f, double x, double y, double z,
                                       double* g)
{
  g[0] = g[1] = g[2] = 0.0;
  switch (f.type) {
  case IFEM_GPU_FN_SINPROD: {
    const double s0 = sin(M_PI * x), s1 = sin(M_PI * y), s2 = sin(M_PI * z);
    const double c0 = cos(M_PI * x), c1 = cos(M_PI * y), c2 = cos(M_PI * z);
    g[0] = f.scale * M_PI * c0 * s1 * s2;
    g[1] = f.scale * M_PI * s0 * c1 * s2;
    g[2] = f.scale * M_PI * s0 * s1 * c2;
    return;
  }
  case IFEM_GPU_FN_FOURIER:
  case IFEM_GPU_FN_EXP_FOURIER: {
    double s = 0.0;
    for (int m = 0; m < f.nmodes; m++) {
      const double* md = f.modes + 5 * m;
      const double arg = md[0] * x + md[1] * y + md[2] * z + md[3];
      s += md[4] * cos(arg);
      for (int d = 0; d < 3; d++) g[d] -= f.scale * md[4] * md[d] * sin(arg);
    }
    if (f.type == IFEM_GPU_FN_EXP_FOURIER) {
      const double e = exp(f.mean + f.scale * s);
      for (int d = 0; d < 3; d++) g[d] *= e;
    }
    return;
  }
  default:
    return;
  }
}

struct NormArgs {
  AsmArgs a;
  const double* x;     // solution, equation order
  const double* xdof;  // or the expanded solution per DOF (nullptr: use x)
  DevFunction exact;
  int has_exact;
  double* part;     // 6 x gridDim.x partial sums
};

template <int P, int NC>
__global__ __launch_bounds__(256) void k_norms(NormArgs na, int64_t total)
{
  constexpr int P1 = P + 1;
  const AsmArgs& a = na.a;
  const int ng = a.ng, gp3 = ng * ng * ng;
  double acc[6] = {0, 0, 0, 0, 0, 0};
  for (int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; id < total;
       id += (int64_t)gridDim.x * blockDim.x) {
    const int64_t e = id / gp3;
    const int q = (int)(id - e * gp3);
    const int q1 = q % ng, q2 = (q / ng) % ng, q3 = q / (ng * ng);
    const int e1 = (int)(e % a.nel1), e2 = (int)((e / a.nel1) % a.nel2),
              e3 = (int)(e / ((int64_t)a.nel1 * a.nel2));
    double J[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    double X[3] = {0, 0, 0}, uh[NC], gr[NC][3];
    for (int c = 0; c < NC; c++) {
      uh[c] = 0.0;
      gr[c][0] = gr[c][1] = gr[c][2] = 0.0;
    }
    for (int b3 = 0; b3 < P1; b3++)
      for (int b2 = 0; b2 < P1; b2++)
#pragma unroll
        for (int b1 = 0; b1 < P1; b1++) {
          const double n1 = a.tabN1[(e1 * ng + q1) * P1 + b1], d1 = a.tabD1[(e1 * ng + q1) * P1 + b1];
          const double n2 = a.tabN2[(e2 * ng + q2) * P1 + b2], d2 = a.tabD2[(e2 * ng + q2) * P1 + b2];
          const double n3 = a.tabN3[(e3 * ng + q3) * P1 + b3], d3 = a.tabD3[(e3 * ng + q3) * P1 + b3];
          const double g0 = d1 * n2 * n3, g1 = n1 * d2 * n3, g2 = n1 * n2 * d3, nv = n1 * n2 * n3;
          const int64_t node =
              (int64_t)(e1 + b1) + (int64_t)a.n1 * ((e2 + b2) + (int64_t)a.n2 * (e3 + b3));
#pragma unroll
          for (int i = 0; i < 3; i++) {
            const double xi = a.coefs[3 * node + i];
            J[3 * i + 0] += xi * g0;
            J[3 * i + 1] += xi * g1;
            J[3 * i + 2] += xi * g2;
            X[i] += xi * nv;
          }
#pragma unroll
          for (int c = 0; c < NC; c++) {
            const int eqn = a.eq[node * NC + c];
            const double ub = na.xdof ? na.xdof[node * NC + c]
                                      : (eqn >= 0 ? na.x[eqn] : (a.gval ? a.gval[node * NC + c] : 0.0));
            uh[c] += nv * ub;
            gr[c][0] += g0 * ub;
            gr[c][1] += g1 * ub;
            gr[c][2] += g2 * ub;
          }
        }
    const double det = J[0] * (J[4] * J[8] - J[7] * J[5]) - J[1] * (J[3] * J[8] - J[6] * J[5]) +
                       J[2] * (J[3] * J[7] - J[6] * J[4]);
    if (det <= 1e-12 && det >= -1e-12) continue;
    double Ji[9];
    Ji[0] = (J[4] * J[8] - J[7] * J[5]) / det;
    Ji[3] = -(J[3] * J[8] - J[6] * J[5]) / det;
    Ji[6] = (J[3] * J[7] - J[6] * J[4]) / det;
    Ji[1] = -(J[1] * J[8] - J[7] * J[2]) / det;
    Ji[4] = (J[0] * J[8] - J[6] * J[2]) / det;
    Ji[7] = -(J[0] * J[7] - J[6] * J[1]) / det;
    Ji[2] = (J[1] * J[5] - J[4] * J[2]) / det;
    Ji[5] = -(J[0] * J[5] - J[3] * J[2]) / det;
    Ji[8] = (J[0] * J[4] - J[3] * J[1]) / det;
    const double dV = 0.125 * (a.span1[e1] * a.span2[e2] * a.span3[e3]);
    const double w = det * (dV * a.gw[q1] * a.gw[q2] * a.gw[q3]);
    // grad u_h: G_cj = sum_i ghat_ci Ji[i][j]
    double G[NC][3];
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
      for (int j = 0; j < 3; j++)
        G[c][j] = gr[c][0] * Ji[j] + gr[c][1] * Ji[3 + j] + gr[c][2] * Ji[6 + j];
    if (NC == 1) {
      const double kap = field_varies(a.kappa) ? eval_field(a.kappa, X[0], X[1], X[2]) : a.kappa_c;
      acc[0] += w * uh[0] * uh[0];
      acc[1] += w * kap * (G[0][0] * G[0][0] + G[0][1] * G[0][1] + G[0][2] * G[0][2]);
      if (na.has_exact) {
        double ge[3];
        const double ue = eval_field(na.exact, X[0], X[1], X[2]);
        eval_field_grad(na.exact, X[0], X[1], X[2], ge);
        const double d0 = ge[0] - G[0][0], d1 = ge[1] - G[0][1], d2 = ge[2] - G[0][2];
        acc[2] += w * ue * ue;
        acc[3] += w * kap * (ge[0] * ge[0] + ge[1] * ge[1] + ge[2] * ge[2]);
        acc[4] += w * (ue - uh[0]) * (ue - uh[0]);
        acc[5] += w * kap * (d0 * d0 + d1 * d1 + d2 * d2);
      }
    } else {
      double tr = 0.0, ee = 0.0;
#pragma unroll
      for (int r = 0; r < 3; r++) tr += G[r][r];
#pragma unroll
      for (int r = 0; r < 3; r++)
#pragma unroll
        for (int cc = 0; cc < 3; cc++) {
          const double eps = 0.5 * (G[r][cc] + G[cc][r]);
          ee += eps * eps;
        }
      double u2 = 0.0;
#pragma unroll
      for (int c = 0; c < NC; c++) u2 += uh[c] * uh[c];
      acc[0] += w * u2;
      acc[1] += w * (a.lam * tr * tr + 2.0 * a.mu * ee);
    }
  }
  __shared__ double sh[4];
  for (int m = 0; m < 6; m++) {
    double v = acc[m];
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) na.part[m * gridDim.x + blockIdx.x] = sh[0] + sh[1] + sh[2] + sh[3];
  }
}

// Squared norm integrals of one patch added to sq[6].
static int norms_patch(Context& c, const PatchRec& Pt, const int* eqmap, const double* gval,
                       const double* xdof, const ifem_gpu_integrand& itg, const int ng[3],
                       const ifem_gpu_function* exact, double* sq);

int integrate_norms(Context& c, const ifem_gpu_integrand& itg, const int ng[3],
                    const ifem_gpu_function* exact, double* out)
{
  double sq[6] = {0, 0, 0, 0, 0, 0};
  if (c.mpc) { // slaves with masters: integrate the expanded solution
    int rc = mpc_expand_device(c);
    if (!rc) rc = norms_patch(c, c.patches[c.patch], c.d_eq, c.d_gval, c.mpc->d_xdof, itg, ng,
                              exact, sq);
    if (rc) return rc;
  } else if (c.multi.empty()) {
    int rc = norms_patch(c, c.patches[c.patch], c.d_eq, c.d_gval, nullptr, itg, ng, exact, sq);
    if (rc) return rc;
  } else {
    for (const SubPatch& sp : c.multi) {
      int rc = norms_patch(c, c.patches[sp.patch], sp.d_leq, sp.d_lgval, nullptr, itg, ng, exact,
                           sq);
      if (rc) return rc;
    }
  }
  for (int m = 0; m < 6; m++) out[m] = sq[m] < 0.0 ? -std::sqrt(-sq[m]) : std::sqrt(sq[m]);
  return IFEM_GPU_OK;
}

static int norms_patch(Context& c, const PatchRec& Pt, const int* eqmap, const double* gval,
                       const double* xdof, const ifem_gpu_integrand& itg, const int ng[3],
                       const ifem_gpu_function* exact, double* sq)
{
  const int p = Pt.p[0];
  if (ng[0] != ng[1] || ng[0] != ng[2] || ng[0] < 1 || ng[0] > kMaxNG)
    return fail(IFEM_GPU_EUNSUPPORTED, "norms: equal Gauss counts 1..5 per direction needed");
  if (exact && c.ncomp != 1)
    return fail(IFEM_GPU_EUNSUPPORTED, "norms: exact solutions are scalar (Poisson) only");
  const int g = ng[0];
  GaussArgs ga{};
  gauss_rule(g, ga.xi, ga.w);
  Tables tb;
  int rc = 0;
  switch (p) {
  case 1: rc = make_tables<1>(c, Pt, g, tb, ga); break;
  case 2: rc = make_tables<2>(c, Pt, g, tb, ga); break;
  case 3: rc = make_tables<3>(c, Pt, g, tb, ga); break;
  default: return fail(IFEM_GPU_EUNSUPPORTED, "norms: degree out of range");
  }
  if (rc) return rc;
  NormArgs na{};
  AsmArgs& a = na.a;
  a.n1 = Pt.n[0]; a.n2 = Pt.n[1]; a.n3 = Pt.n[2];
  a.nel1 = Pt.nel[0]; a.nel2 = Pt.nel[1]; a.nel3 = Pt.nel[2];
  a.coefs = Pt.d_coefs;
  a.tabN1 = tb.tabN[0]; a.tabD1 = tb.tabD[0]; a.span1 = tb.span[0];
  a.tabN2 = tb.tabN[1]; a.tabD2 = tb.tabD[1]; a.span2 = tb.span[1];
  a.tabN3 = tb.tabN[2]; a.tabD3 = tb.tabD[2]; a.span3 = tb.span[2];
  for (int k = 0; k < kMaxNG; k++) a.gw[k] = ga.w[k];
  a.eq = eqmap;
  a.gval = gval;
  a.ng = g;
  a.ncomp = c.ncomp;
  rc = upload_function(c, itg.kappa, a.kappa, 0);
  if (rc) return rc;
  a.kappa_c = const_value(itg.kappa, 1.0);
  if (itg.kind == IFEM_GPU_ELASTICITY) {
    a.lam = itg.E * itg.nu / ((1.0 + itg.nu) * (1.0 - 2.0 * itg.nu));
    a.mu = itg.E / (2.0 * (1.0 + itg.nu));
  }
  if (exact) {
    rc = upload_function(c, *exact, na.exact, 2);
    if (rc) return rc;
    na.has_exact = 1;
  }
  na.x = c.w.x;
  na.xdof = xdof;
  const int64_t total = (int64_t)Pt.nel[0] * Pt.nel[1] * Pt.nel[2] * g * g * g;
  const int grid = 1024;
  double* part = nullptr;
  IFEM_HIP(hipMalloc(&part, sizeof(double) * 6 * grid));
  na.part = part;
  if (c.ncomp == 3) {
    switch (p) {
    case 1: k_norms<1, 3><<<grid, 256, 0, c.stream>>>(na, total); break;
    case 2: k_norms<2, 3><<<grid, 256, 0, c.stream>>>(na, total); break;
    default: k_norms<3, 3><<<grid, 256, 0, c.stream>>>(na, total); break;
    }
  } else {
    switch (p) {
    case 1: k_norms<1, 1><<<grid, 256, 0, c.stream>>>(na, total); break;
    case 2: k_norms<2, 1><<<grid, 256, 0, c.stream>>>(na, total); break;
    default: k_norms<3, 1><<<grid, 256, 0, c.stream>>>(na, total); break;
    }
  }
  const hipError_t le = hipGetLastError();
  std::vector<double> h(6 * grid);
  const hipError_t ce = hipMemcpyAsync(h.data(), part, sizeof(double) * 6 * grid,
                                       hipMemcpyDeviceToHost, c.stream);
  const hipError_t se = hipStreamSynchronize(c.stream);
  hipFree(part);
  if (le != hipSuccess || ce != hipSuccess || se != hipSuccess)
    return fail(IFEM_GPU_EDEVICE, "norms: device error");
  for (int m = 0; m < 6; m++) {
    double sum = 0.0;
    for (int b = 0; b < grid; b++) sum += h[m * grid + b];
    sq[m] += sum;
  }
  return IFEM_GPU_OK;
}

} // namespace ifem
