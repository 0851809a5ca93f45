// asmargs.hpp -- arguments and geometry records shared by the geometry pass
// (assemble.hip) and the line kernels (lines.hpp).
#pragma once

#include <hip/hip_runtime.h>

#include "internal.hpp"

namespace ifem {

struct AsmArgs {
  int n1, n2, n3;
  int nel1, nel2, nel3;
  const double* coefs;                 // nnod*3
  const double *tabN1, *tabD1, *span1; // direction tables
  const double *tabN2, *tabD2, *span2;
  const double *tabN3, *tabD3, *span3;
  double gw[kMaxNG];                   // Gauss weights
  const int* eq;                       // per DOF: 0-based eq or -1
  const int64_t* rowptr;
  double* val64;
  float* val32;
  double* rhs;                         // FP64 RHS (nullptr: not written)
  DevFunction kappa, source;
  double body[3];
  double lam, mu;
  int ng;                              // Gauss points per direction
  int ncomp;                           // 1 scalar, 3 vector (elasticity)
  // geometry record per (element, Gauss point), [element][GeoRec::N][gp]
  // with element e1 + nel1*(e2 + nel2*e3) and gp q1 + ng*(q2 + ng*q3),
  // written by k_gp_geometry, read by the line kernels
  double* gp_geo;
  int geo_pairs;                       // vector records in rows of pairs
  double kappa_c, source_c;            // values of constant fields
  // per DOF prescribed value of eliminated DOFs (FP64 pass only; nullptr:
  // homogeneous); the eliminated columns move to the RHS, b_i -= K_ij g_j
  const double* gval;
  // several patches in one system: rows are shared across patches, so
  // values are added at the column found by binary search in the sorted row
  const int32_t* colind;
  int accum;
  // accumulate mode with precomputed positions (SubPatch::d_pmap / d_pptr)
  const int64_t* pmap;
  const int64_t* pptr;
};

// Geometry record of one Gauss point.  Vector problems: J^-1 (row-major, 9)
// and w*detJ.  Scalar problems: M = w*detJ*kappa(X) * J^-1 J^-T (symmetric:
// m00 m01 m02 m11 m12 m22) and w*detJ*f(X).  Stored per element as N rows of
// ng^3 values (value c of point q of element e at (e*N + c)*ng^3 + q), so that
// consecutive points are consecutive in memory for the pass that writes them
// and for the line kernels that read them.  The direct line kernels read all
// values of a point in one thread: vector records for them are N/2 rows of
// pairs (AsmArgs::geo_pairs), half the loads; single values made cubic
// elasticity 1.3 % slower (31x24x35: 7.05 against 6.93 ms).
template <int NC>
struct GeoRec {
  static constexpr int N = NC == 1 ? 7 : 10;
};

// The line kernels read their AsmArgs from a device buffer through the
// constant address space: the fields are uniform, read-only loads that the
// compiler may re-issue instead of holding them all in registers.
typedef const __attribute__((address_space(4))) AsmArgs ConstArgs;

__device__ inline ConstArgs* const_args(const AsmArgs* p)
{
  return (ConstArgs*)p;
}

} // namespace ifem
