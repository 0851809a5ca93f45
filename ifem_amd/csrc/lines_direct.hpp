// lines_direct.hpp -- line kernels by direct quadrature (vector problems) or
// per-element sum factorisation (scalar problems with more than 27 Gauss
// points per element), one line per workgroup: degree 3, degree 2 with 4x4x4
// points, and FP32 elasticity of degree 2.  One 256-thread workgroup owns a line of control points; in
// each element layer the (p+1)^2 elements touching the line are processed in
// chunks: phase A (thread per element and Gauss point) forms the row
// functions' transformed gradients, phase B (thread per element and column
// function) sums over the Gauss points, the sums enter an LDS window of p+1
// dense rows in element order, and phase D writes each completed row once.
#pragma once

#include <algorithm>
#include <type_traits>

#include "lines_launch.hpp"

namespace ifem {

// Chunk of layer elements processed together so that CH*NG^3 ~ one block;
// HALF = 1 selects half of that (an autotuning variant: less LDS, more
// phases); HALF = 2 keeps the full chunk and splits its Gauss points into
// two slabs of q3 rows (half the geometry LDS: three workgroups per CU).
template <int P, int NG, int HALF = 0>
struct Chunk {
  static constexpr int P1 = P + 1;
  static constexpr int NB = P1 * P1;
  static constexpr int GP3 = NG * NG * NG;
  static constexpr int full = (256 / GP3) < 1 ? 1 : ((256 / GP3) > NB ? NB : (256 / GP3));
  static constexpr int v = HALF == 1 ? ((full + 1) / 2) : full;
  static constexpr int NSL = HALF == 2 ? 2 : 1;                    // Gauss-point slabs
  static constexpr int SLQ = NG * NG * ((NG + NSL - 1) / NSL);     // points per slab (max)
};

constexpr int kBlock = 256;

// Block barrier after LDS writes that other waves read right after it: the
// wave first waits for its own LDS operations to complete (s_waitcnt
// lgkmcnt(0)).  The compiler emits no such wait before the barrier of a loop
// whose body ends in LDS stores (the element rounds of the window update),
// and without it a round's reads could see a window entry before the
// previous round's store to it had landed (observed as lost contributions on
// entries shared by consecutive bundle elements, in workgroups sharing a CU).
__device__ __forceinline__ void lds_barrier()
{
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __syncthreads();
}

// LDS of one line workgroup.  T: arithmetic type of the element integrals
// (double: FP64 path, float: FP32 path).  NC: components (1 Poisson,
// 3 elasticity).  SPLIT: number of blocks per line sharing the row
// components (NC/SPLIT rows each).  HALF: half-size element chunks.
template <int P, int NG, int NC, typename T, int SPLIT, bool HAS_RHS, int HALF, bool ORDL = false>
struct LineLds {
  static constexpr int P1 = P + 1;
  static constexpr int NEN = P1 * P1 * P1;
  static constexpr int GP3 = NG * NG * NG;
  static constexpr int NB = P1 * P1;
  static constexpr int W1 = 2 * P + 1;
  static constexpr int WN = W1 * W1 * W1;
  static constexpr int NCR = NC / SPLIT;
  static constexpr bool SACC = (NC == 3 && SPLIT == 1); // accumulate S_ij, apply lam/mu later
  static constexpr int NS = NC == 1 ? 1 : (SACC ? 9 : 3);
  static constexpr int CH = Chunk<P, NG, HALF>::v;
  static constexpr int NSL = Chunk<P, NG, HALF>::NSL;
  static constexpr int SLQ = Chunk<P, NG, HALF>::SLQ;
  static constexpr int GEO = (NC == 3 ? 9 : 0) + 3 * P1;
  static constexpr int NRHS = HAS_RHS ? P1 * NC : 1;
  // scalar problems with more than 27 Gauss points per element (the ordered,
  // not pipelined path): phase B by sum factorisation, see line_impl
  static constexpr bool SF =
      NC == 1 && GP3 > 27 && HALF != 1 && CH * NEN <= 256 && P >= 2 && P1 <= NG;

  // every member 16-byte aligned: lets the compiler use 128-bit LDS loads
  alignas(16) T win[P1][NCR][WN][NC];
  alignas(16) T geo[CH * SLQ][GEO];
  // ORDL (ordered window updates): no stage; RHS stage of w*detJ*N_a only
  alignas(16) T stage[ORDL ? 1 : CH][NEN][P1][NS];
  alignas(16) T rstage[HAS_RHS ? CH * SLQ : 1][ORDL ? (HAS_RHS ? P1 : 1) : NRHS];
  alignas(16) T rwin[P1][NC];
  alignas(16) T tN1[NG][P1];
  alignas(16) T tD1[NG][P1];
  alignas(16) T tN2[P1][NG][P1];
  alignas(16) T tD2[P1][NG][P1];
  alignas(16) T tN3[P1][NG][P1];
  alignas(16) T tD3[P1][NG][P1];
  alignas(16) int be2[NB];
  alignas(16) int be3[NB];
  static constexpr int NT = (WN * NC + 63) / 64;
  // neighbour equation numbers kept in LDS for phase D (not for p = 3,
  // whose LDS budget goes to the element chunk, nor for the slab variant,
  // whose budget is three workgroups per CU)
  static constexpr bool PFD = P < 3 && NSL == 1;
  // two buffers: row e1's (being filled) and row e1-1's (written out at the
  // top of layer e1)
  alignas(16) int eqw[2][PFD ? NT * 64 : 1];
  alignas(16) int64_t pbase[2][NCR];
  int prow[2][NCR];
  int nbundle;
};

// The LDS arrays come in as separate __restrict__ pointers so that, after
// inlining, the compiler knows they do not alias (fields of one struct with
// run-time indices would otherwise be assumed to overlap).
template <int P, int NG, int NC, typename T, int SPLIT, bool HAS_RHS, int HALF, bool PIPE, bool ORD,
          bool SEMI = false>
__device__ __forceinline__ void line_impl(
    ConstArgs& a, const int line, const int split,
    T (*__restrict__ win)[LineLds<P, NG, NC, T, SPLIT, HAS_RHS, HALF>::NCR]
                         [LineLds<P, NG, NC, T, SPLIT, HAS_RHS, HALF>::WN][NC],
    T (*__restrict__ geo)[LineLds<P, NG, NC, T, SPLIT, HAS_RHS, HALF>::GEO],
    T (*__restrict__ stage)[LineLds<P, NG, NC, T, SPLIT, HAS_RHS, HALF>::NEN][P + 1]
                           [LineLds<P, NG, NC, T, SPLIT, HAS_RHS, HALF>::NS],
    T* __restrict__ rstage,
    T (*__restrict__ rwin)[NC],
    T (*__restrict__ tN1)[P + 1], T (*__restrict__ tD1)[P + 1],
    T (*__restrict__ tN2)[NG][P + 1], T (*__restrict__ tD2)[NG][P + 1],
    T (*__restrict__ tN3)[NG][P + 1], T (*__restrict__ tD3)[NG][P + 1],
    int* __restrict__ be2, int* __restrict__ be3,
    int (*__restrict__ eqw)[LineLds<P, NG, NC, T, SPLIT, HAS_RHS, HALF>::PFD
                            ? LineLds<P, NG, NC, T, SPLIT, HAS_RHS, HALF>::NT * 64 : 1],
    int64_t (*__restrict__ pbase)[LineLds<P, NG, NC, T, SPLIT, HAS_RHS, HALF>::NCR],
    int (*__restrict__ prow)[LineLds<P, NG, NC, T, SPLIT, HAS_RHS, HALF>::NCR],
    int* __restrict__ nbundlep)
{
  using LL = LineLds<P, NG, NC, T, SPLIT, HAS_RHS, HALF>;
  constexpr int P1 = LL::P1;
  constexpr int NEN = LL::NEN;
  constexpr int GP3 = LL::GP3;
  constexpr int W1 = LL::W1;
  constexpr int WN = LL::WN;
  constexpr int NCR = LL::NCR;
  constexpr bool SACC = LL::SACC;
  constexpr int NS = LL::NS;
  constexpr int CH = LL::CH;
  constexpr int NSL = LL::NSL; // Gauss-point slabs per chunk (geometry rows in LDS per slab)
  constexpr int SLQ = LL::SLQ;
  static_assert(NSL == 1 || (ORD && PIPE), "Gauss-point slabs need the ordered, pipelined path");
  // ORD: the whole bundle in one chunk, column sums added to the window
  // element by element (no stage); the RHS stage then holds w*detJ*N_a and
  // the body force is applied after the sum
  static_assert(!ORD || CH * LL::NEN <= kBlock, "ordered updates need one item per thread");
  constexpr int RS = ORD ? (HAS_RHS ? P1 : 1) : LL::NRHS; // RHS stage row length
  const int rc = split * NCR; // first row component of the block

  const int tid = threadIdx.x;
  const int jc = line % a.n2, kc = line / a.n2;
  // split: row components [split*NCR, split*NCR+NCR)

  // bundle of elements touching the line, fixed order (e3 outer, e2 inner)
  if (tid == 0) {
    int nb = 0;
    for (int m3 = 0; m3 < P1; m3++)
      for (int m2 = 0; m2 < P1; m2++) {
        const int e2 = jc - P + m2, e3 = kc - P + m3;
        if (e2 >= 0 && e2 < a.nel2 && e3 >= 0 && e3 < a.nel3) {
          be2[nb] = e2;
          be3[nb] = e3;
          nb++;
        }
      }
    *nbundlep = nb;
  }
  // direction 2/3 tables for elements jc-P..jc and kc-P..kc
  for (int t = tid; t < P1 * NG * P1; t += kBlock) {
    const int m = t / (NG * P1), r = t % (NG * P1);
    const int g = r / P1, q = r % P1;
    const int e2 = jc - P + m, e3 = kc - P + m;
    T n2 = 0, d2 = 0, n3 = 0, d3 = 0;
    if (e2 >= 0 && e2 < a.nel2) {
      n2 = (T)a.tabN2[(e2 * NG + g) * P1 + q];
      d2 = (T)a.tabD2[(e2 * NG + g) * P1 + q];
    }
    if (e3 >= 0 && e3 < a.nel3) {
      n3 = (T)a.tabN3[(e3 * NG + g) * P1 + q];
      d3 = (T)a.tabD3[(e3 * NG + g) * P1 + q];
    }
    tN2[m][g][q] = n2;
    tD2[m][g][q] = d2;
    tN3[m][g][q] = n3;
    tD3[m][g][q] = d3;
  }
  for (int t = tid; t < P1 * NCR * WN * NC; t += kBlock) (&win[0][0][0][0])[t] = T(0);
  for (int t = tid; t < P1 * NC; t += kBlock) (&rwin[0][0])[t] = T(0);
  __syncthreads();
  const int nb = *nbundlep;

  const T lam = (T)a.lam, mu = (T)a.mu;

  constexpr int NT = LL::NT; // phase D: 64-column steps per row
  // ---- phase D: write row i of the window out (row e1-1 at the top of layer
  // e1, while phase A runs; the last layer's rows at its end).  pf: the
  // equation numbers of the row are in buffer pb (from the layer top);
  // zero_rhs: clear the row's right-hand side entries after reading them.
  auto row_out = [&](int i, bool pf, int pb, bool zero_rhs) {
    const int slot = i % P1;
    const int64_t node = (int64_t)i + (int64_t)a.n1 * (jc + (int64_t)a.n2 * kc);
    const int wave = tid >> 6, lane = tid & 63;
    if (wave < NCR) {
      const int ic = split * NCR + wave;
      const int req = pf ? prow[pb][wave] : a.eq[node * NC + ic];
      const bool pfe = LL::PFD && pf;
      if (req >= 0) {
        const int64_t base = pf ? pbase[pb][wave] : a.rowptr[req];
        const double* __restrict__ gv = a.gval;
        double corr = 0.0;
        int64_t pos = 0;
#pragma unroll 1
        for (int k = 0; k < NT; k++) {
          const int t = k * 64 + lane;
          const int ev = pfe ? eqw[pb][t] : window_eq<P, NC>(a, i, jc, kc, t);
          const bool valid = ev >= 0;
          const unsigned long long m = __ballot(valid);
          if (valid && a.accum && a.pmap) {
            const T v = win[slot][wave][t / NC][t % NC];
            const int64_t at = a.pmap[a.pptr[node * NC + ic] + pos + __popcll(m & ((1ull << lane) - 1ull))];
            if (a.val32) a.val32[at] += (float)v;
            else a.val64[at] += (double)v;
          } else if (valid && a.accum) {
            const T v = win[slot][wave][t / NC][t % NC];
            int64_t lo = base, hi = a.rowptr[req + 1] - 1;
            while (lo <= hi) {
              const int64_t mid = (lo + hi) >> 1;
              const int cm = a.colind[mid];
              if (cm == ev) {
                if (a.val32) a.val32[mid] += (float)v;
                else a.val64[mid] += (double)v;
                break;
              }
              if (cm < ev) lo = mid + 1;
              else hi = mid - 1;
            }
          } else if (valid) {
            const int64_t at = base + pos + __popcll(m & ((1ull << lane) - 1ull));
            const T v = win[slot][wave][t / NC][t % NC];
            if (a.val32) a.val32[at] = (float)v;
            else a.val64[at] = (double)v;
          } else if (gv && ev == -1) { // eliminated column inside the patch
            const int nbr = t / NC;
            const int ii = i + nbr % W1 - P, jj = jc + (nbr / W1) % W1 - P, kk = kc + nbr / (W1 * W1) - P;
            const int64_t gdof = ((int64_t)ii + (int64_t)a.n1 * (jj + (int64_t)a.n2 * kk)) * NC + t % NC;
            corr += (double)win[slot][wave][t / NC][t % NC] * gv[gdof];
          }
          pos += __popcll(m);
        }
        if (gv) {
#pragma unroll
          for (int off = 32; off >= 1; off >>= 1) corr += __shfl_xor(corr, off, 64);
        }
        if ((HAS_RHS || gv) && a.rhs && lane == 0) {
          if (a.accum) a.rhs[req] += (double)rwin[slot][ic] - corr;
          else a.rhs[req] = (double)rwin[slot][ic] - corr;
        }
      }
      if (zero_rhs && lane == 0) rwin[slot][ic] = T(0);
    }
    if (zero_rhs && tid == 0)
      for (int c = 0; c < NC; c++)
        if (c < split * NCR || c >= split * NCR + NCR) rwin[slot][c] = T(0);
  };
  for (int e1 = 0; e1 < a.nel1; e1++) {
    // ---- direction-1 tables of this layer ----------------------------------
    // with the equation numbers of row e1 and of its neighbour columns for
    // phase D (their loads overlap those of the tables)
    for (int t = tid; t < NG * P1; t += kBlock) {
      (&tN1[0][0])[t] = (T)a.tabN1[e1 * NG * P1 + t];
      (&tD1[0][0])[t] = (T)a.tabD1[e1 * NG * P1 + t];
    }
    const int buf = e1 & 1;
    // equation numbers of row e1's neighbour columns for its phase D (at the
    // top of the next layer): for elasticity without a body force loaded now
    // and stored after phase B (after phase A in the unordered variants; EQE),
    // so that their latency is not exposed at the barrier below; elsewhere the
    // two registers would cost a wave per SIMD, and they are stored here
    constexpr bool EQE = LL::PFD && NC == 3 && !HAS_RHS;
    constexpr int NEQV = EQE ? (NT * 64 + kBlock - 1) / kBlock : 1;
    int eqv[NEQV];
#pragma unroll
    for (int k = 0; k < NEQV; k++) {
      const int t = tid + k * kBlock;
      eqv[k] = (EQE && t < NT * 64) ? window_eq<P, NC>(a, e1, jc, kc, t) : -2;
    }
    if (LL::PFD && !EQE)
      for (int t = tid; t < NT * 64; t += kBlock) eqw[buf][t] = window_eq<P, NC>(a, e1, jc, kc, t);
    if (tid < NCR) {
      const int64_t node = (int64_t)e1 + (int64_t)a.n1 * (jc + (int64_t)a.n2 * kc);
      prow[buf][tid] = a.eq[node * NC + split * NCR + tid];
    }
    __syncthreads();
    // row start of row e1, read while phase A runs
    int64_t pf_base = 0;
    if (tid < NCR && prow[buf][tid] >= 0) pf_base = a.rowptr[prow[buf][tid]];
    // row e1-1, complete since the last layer, goes out now: its loads and
    // stores overlap phase A (its window slot is cleared after phase A, and
    // its right-hand side entries by the threads that read them)
    if (e1 > 0) row_out(e1 - 1, true, buf ^ 1, true);

    for (int c0 = 0; c0 < nb; c0 += CH) {
      const int nch = (nb - c0) < CH ? (nb - c0) : CH;

      // ---- phase A: geometry per (element, Gauss point) of the points
      // [qa, qa + ngs) (all of them unless the chunk runs in slabs) --------
      auto phase_a = [&](const int qa, const int ngs) {
      for (int t = tid; t < nch * ngs; t += kBlock) {
        const int le = t / ngs, q = qa + t % ngs;
        const int e2 = be2[c0 + le], e3 = be3[c0 + le];
        const int m2 = e2 - jc + P, m3 = e3 - kc + P; // table slots
        const int q1 = q % NG, q2 = (q / NG) % NG, q3 = q / (NG * NG);
        // geometry record of this (element, Gauss point), computed once per
        // element by k_gp_geometry: J^-1 and w*detJ (vector), or
        // M = w*detJ*kappa*J^-1 J^-T and w*detJ*f (scalar)
        const int64_t ge = (int64_t)e1 + (int64_t)a.nel1 * (e2 + (int64_t)a.nel2 * e3);
        T R[GeoRec<NC>::N];
        if constexpr (NC == 3) {
          const double2* __restrict__ rec =
              reinterpret_cast<const double2*>(a.gp_geo) + ge * (GP3 * (GeoRec<NC>::N / 2)) + q;
#pragma unroll
          for (int k = 0; k < GeoRec<NC>::N / 2; k++) {
            const double2 v = rec[k * GP3];
            R[2 * k] = (T)v.x;
            R[2 * k + 1] = (T)v.y;
          }
        } else {
          const double* __restrict__ rec = a.gp_geo + ge * (GP3 * GeoRec<NC>::N) + q;
#pragma unroll
          for (int k = 0; k < GeoRec<NC>::N; k++)
            R[k] = k == 6 && !HAS_RHS ? T(0) : (T)rec[k * GP3];
        }
        if (NC == 3) {
#pragma unroll
          for (int m = 0; m < 9; m++) geo[t][m] = R[m];
        }
        const int a2r = jc - e2, a3r = kc - e3; // row node's local (a2, a3)
        const T n2a = tN2[m2][q2][a2r], d2a = tD2[m2][q2][a2r];
        const T n3a = tN3[m3][q3][a3r], d3a = tD3[m3][q3][a3r];
        if constexpr (LL::SF) {
          // W_kl = M_kl * A2_k(q2) * A3_k(q3) for the line's row functions in
          // directions 2 and 3 (A_k: derivative in direction k, else value)
          const T M[9] = {R[0], R[1], R[2], R[1], R[3], R[4], R[2], R[4], R[5]};
          const T a2[3] = {n2a, d2a, n2a}, a3[3] = {n3a, n3a, d3a};
          // stored [element][kl][q1][q2][q3]: the (q2, q3) slab of each q1
          // is contiguous, and its T2 later overwrites it in place
          T* __restrict__ wf = &geo[0][0] + (int64_t)le * 9 * GP3 + (q1 * NG + q2) * NG + q3;
#pragma unroll
          for (int k = 0; k < 3; k++)
#pragma unroll
            for (int l = 0; l < 3; l++) wf[(3 * k + l) * GP3] = M[3 * k + l] * a2[k] * a3[k];
        }
#pragma unroll
        for (int a1 = 0; a1 < P1; a1++) {
          const T n1 = tN1[q1][a1], d1 = tD1[q1][a1];
          const T r0 = d1 * n2a * n3a, r1 = n1 * d2a * n3a, r2 = n1 * n2a * d3a;
          if (NC == 1 && LL::SF) {
            // written once below the a1 loop
          } else if (NC == 1) {
            // h_a = M grad_ref N_a: S_ab = grad_ref N_b . h_a
            geo[t][3 * a1 + 0] = R[0] * r0 + R[1] * r1 + R[2] * r2;
            geo[t][3 * a1 + 1] = R[1] * r0 + R[3] * r1 + R[4] * r2;
            geo[t][3 * a1 + 2] = R[2] * r0 + R[4] * r1 + R[5] * r2;
          } else {
            // w g_a = w J^-T grad_ref N_a  (dNdX = dNdu * J^-1)
            const T w = R[9];
            geo[t][9 + 3 * a1 + 0] = w * (r0 * R[0] + r1 * R[3] + r2 * R[6]);
            geo[t][9 + 3 * a1 + 1] = w * (r0 * R[1] + r1 * R[4] + r2 * R[7]);
            geo[t][9 + 3 * a1 + 2] = w * (r0 * R[2] + r1 * R[5] + r2 * R[8]);
          }
          if (HAS_RHS) {
            const T Na = n1 * n2a * n3a;
            if (NC == 1) {
              rstage[t * RS + a1] = R[6] * Na;
            } else if (ORD) {
              rstage[t * RS + a1] = R[9] * Na;
            } else {
#pragma unroll
              for (int c = 0; c < NC; c++) rstage[t * RS + a1 * NC + c] = R[9] * (T)a.body[c] * Na;
            }
          }
        }
      }
      };
      // ---- RHS: fixed-order reduction over (element, GP) of a slab ---------
      auto rhs_reduce = [&](const int ngs) {
        const int v = tid >> 4, l = tid & 15;
        T s = T(0);
        const int vs = (ORD && NC == 3) ? v / NC : v;
        if (v < P1 * NC)
          for (int pr = l; pr < nch * ngs; pr += 16) s += rstage[pr * RS + vs];
#pragma unroll
        for (int off = 8; off >= 1; off >>= 1) s += __shfl_xor(s, off, 16);
        if (v < P1 * NC && l == 0) {
          const int a1 = v / NC, c = v % NC;
          rwin[(e1 + a1) % P1][c] += (ORD && NC == 3) ? s * (T)a.body[c] : s;
        }
      };
      phase_a(0, NSL == 1 ? GP3 : SLQ);
      if (c0 == 0 && tid < NCR) pbase[buf][tid] = pf_base;
      __syncthreads();
      // (ordered updates: after phase B, further from the loads)
      if (EQE && !ORD && c0 == 0) {
#pragma unroll
        for (int k = 0; k < NEQV; k++) {
          const int t = tid + k * kBlock;
          if (t < NT * 64) eqw[buf][t] = eqv[k];
        }
      }
      if (c0 == 0 && e1 > 0) { // slot of row e1-1, read out before the barrier
        const int zs = (e1 - 1) % P1;
        for (int t = tid; t < NCR * WN * NC; t += kBlock) (&win[zs][0][0][0])[t] = T(0);
      }

      if (HAS_RHS) rhs_reduce(NSL == 1 ? GP3 : SLQ);

      // ---- phase B: element-row x column-node products ----------------------
      if constexpr (ORD) {
      // One (element, column node b) item per thread for the chunk (the
      // whole bundle when it fits), Gauss loop as in the pipelined or the
      // row-prefetching variant below; the sums stay in
      // registers and go into the row window one element after the other
      // (element order fixed, so every window entry is summed in that order).
      const bool has = tid < nch * NEN;
      const int le = has ? tid / NEN : 0, b = has ? tid % NEN : 0;
      const int b1 = b % P1, b2 = (b / P1) % P1, b3 = b / (P1 * P1);
      const int e2 = be2[c0 + le], e3 = be3[c0 + le];
      T acc[P1][NS];
#pragma unroll
      for (int a1 = 0; a1 < P1; a1++)
#pragma unroll
        for (int s = 0; s < NS; s++) acc[a1][s] = 0;
        if constexpr (PIPE) {
        static_assert(NC == 3 && !HAS_RHS, "FP32 elasticity with 3x3x3 points");
        const int m2 = e2 - jc + P, m3 = e3 - kc + P;
        T vn1[NG], vd1[NG], vn2[NG], vd2[NG], vn3[NG], vd3[NG];
#pragma unroll
        for (int q = 0; q < NG; q++) {
          vn1[q] = tN1[q][b1]; vd1[q] = tD1[q][b1];
          vn2[q] = tN2[m2][q][b2]; vd2[q] = tD2[m2][q][b2];
          vn3[q] = tN3[m3][q][b3]; vd3[q] = tD3[m3][q][b3];
        }
        // Gauss points in NSL slabs: the geometry rows of slab sl > 0 replace
        // those of slab sl-1 in LDS (every thread takes part in the barriers)
        // (a compile-time slab index, so that each slab's Gauss loop unrolls)
        auto slab_b = [&](auto slc) {
        constexpr int qa = decltype(slc)::value * SLQ;
        constexpr int ngs = (GP3 - qa) < SLQ ? (GP3 - qa) : SLQ;
        if (has) {
        // one workgroup per CU and SIMD pair: the next point's geometry row
        // is prefetched into registers; with slabs (three workgroups per CU)
        // the rows are read from LDS where they are used, the other
        // workgroups hiding the latency
        constexpr bool PREF = NSL == 1;
        const T* __restrict__ Gbase = geo[le * ngs];
        T Gc[PREF ? LL::GEO : 1];
        if constexpr (PREF) {
#pragma unroll
          for (int m = 0; m < LL::GEO; m++) Gc[m] = Gbase[m];
        }
#pragma unroll
        for (int qq = 0; qq < ngs; qq++) {
          const int q = qa + qq;
          T Gn[PREF ? LL::GEO : 1];
          if (PREF && qq + 1 < ngs) {
#pragma unroll
            for (int m = 0; m < LL::GEO; m++) Gn[m] = Gbase[(qq + 1) * LL::GEO + m];
          }
          const int q1 = q % NG, q2 = (q / NG) % NG, q3 = q / (NG * NG);
          const T n23 = vn2[q2] * vn3[q3], d23 = vd2[q2] * vn3[q3], n2d3 = vn2[q2] * vd3[q3];
          const T r0 = vd1[q1] * n23, r1 = vn1[q1] * d23, r2 = vn1[q1] * n2d3;
          const T* G = PREF ? Gc : Gbase + qq * LL::GEO;
          const T gb0 = r0 * G[0] + r1 * G[3] + r2 * G[6];
          const T gb1 = r0 * G[1] + r1 * G[4] + r2 * G[7];
          const T gb2 = r0 * G[2] + r1 * G[5] + r2 * G[8];
#pragma unroll
          for (int a1 = 0; a1 < P1; a1++) {
            const T wa0 = G[9 + 3 * a1], wa1 = G[10 + 3 * a1], wa2 = G[11 + 3 * a1];
            if constexpr (SACC) {
              acc[a1][0] += wa0 * gb0; acc[a1][1] += wa0 * gb1; acc[a1][2] += wa0 * gb2;
              acc[a1][3] += wa1 * gb0; acc[a1][4] += wa1 * gb1; acc[a1][5] += wa1 * gb2;
              acc[a1][6] += wa2 * gb0; acc[a1][7] += wa2 * gb1; acc[a1][8] += wa2 * gb2;
            } else {
              const T wa[3] = {wa0, wa1, wa2}, gb[3] = {gb0, gb1, gb2};
              const T dot = wa0 * gb0 + wa1 * gb1 + wa2 * gb2;
#pragma unroll
              for (int jj = 0; jj < 3; jj++)
                acc[a1][jj] += lam * wa[rc] * gb[jj] + mu * wa[jj] * gb[rc] +
                               (jj == rc ? mu * dot : T(0));
            }
          }
          if (PREF && qq + 1 < ngs) {
#pragma unroll
            for (int m = 0; m < LL::GEO; m++) Gc[m] = Gn[m];
          }
        }
        }
        };
        slab_b(std::integral_constant<int, 0>{});
        if constexpr (NSL > 1) {
          static_assert(NSL == 2, "two slabs");
          constexpr int qa1 = SLQ, ngs1 = GP3 - SLQ;
          __syncthreads();
          phase_a(qa1, ngs1);
          __syncthreads();
          slab_b(std::integral_constant<int, 1>{});
        }
        } else if constexpr (LL::SF) {
        // Sum factorisation (scalar problems): for the line's row functions
        // a = (a1, a2, a3) with a2, a3 fixed by the line,
        //   S_ab = sum_kl sum_q W_kl(q) A1_k(a1,q1) B1_l(b1,q1) B2_l(b2,q2) B3_l(b3,q3)
        // contracted over q3 (T1), then q2 (T2, in the geometry rows' LDS),
        // then q1 with the direction-1 functions, each step in fixed order:
        // 9*NG*NG*P1 + 9*NG*P1*P1 + 3*NG*(P1+3)*NEN operations per element
        // and line instead of 3*GP3*P1*NEN.
        // one thread per (element, kl, q1): its (q2, q3) slab of W into
        // registers, T1(q2, b3) over q3, T2(b2, b3) over q2, written back
        // over the slab (no other thread touches it, so no barrier between
        // the read and the write)
        T* __restrict__ gf = &geo[0][0]; // W, then T2, [element][kl][q1][...] with stride GP3
        for (int t = tid; t < nch * 9 * NG; t += kBlock) {
          const int q1 = t % NG, kl = (t / NG) % 9, lq = t / (9 * NG);
          const int l = kl % 3;
          const int mm2 = be2[c0 + lq] - jc + P, mm3 = be3[c0 + lq] - kc + P;
          T* __restrict__ w = gf + (int64_t)(lq * 9 + kl) * GP3 + q1 * NG * NG;
          T wv[NG][NG];
#pragma unroll
          for (int q2 = 0; q2 < NG; q2++)
#pragma unroll
            for (int q3 = 0; q3 < NG; q3++) wv[q2][q3] = w[q2 * NG + q3];
          T t1[NG][P1];
#pragma unroll
          for (int q2 = 0; q2 < NG; q2++)
#pragma unroll
            for (int bb3 = 0; bb3 < P1; bb3++) {
              T sum = 0;
#pragma unroll
              for (int q3 = 0; q3 < NG; q3++)
                sum += wv[q2][q3] * (l == 2 ? tD3[mm3][q3][bb3] : tN3[mm3][q3][bb3]);
              t1[q2][bb3] = sum;
            }
#pragma unroll
          for (int bb2 = 0; bb2 < P1; bb2++)
#pragma unroll
            for (int bb3 = 0; bb3 < P1; bb3++) {
              T sum = 0;
#pragma unroll
              for (int q2 = 0; q2 < NG; q2++)
                sum += t1[q2][bb3] * (l == 1 ? tD2[mm2][q2][bb2] : tN2[mm2][q2][bb2]);
              w[bb2 * P1 + bb3] = sum; // T2(q1, b2, b3)
            }
        }
        __syncthreads();
        if (has) {
          // per (k, q1): U = T2_k0 B1'(b1) + (T2_k1 + T2_k2) B1(b1) (direction 1
          // carries the derivative for l = 0 only), then U A1_k(a1) per row
          const T* __restrict__ v = gf + (int64_t)le * 9 * GP3 + b2 * P1 + b3;
          T bn[NG], bd[NG];
#pragma unroll
          for (int q1 = 0; q1 < NG; q1++) {
            bn[q1] = tN1[q1][b1];
            bd[q1] = tD1[q1][b1];
          }
#pragma unroll
          for (int k = 0; k < 3; k++) {
#pragma unroll
            for (int q1 = 0; q1 < NG; q1++) {
              const T* __restrict__ vk = v + 3 * k * GP3 + q1 * NG * NG;
              const T u = vk[0] * bd[q1] + (vk[GP3] + vk[2 * GP3]) * bn[q1];
#pragma unroll
              for (int a1 = 0; a1 < P1; a1++)
                acc[a1][0] += u * (k == 0 ? tD1[q1][a1] : tN1[q1][a1]);
            }
          }
        }
        } else {
      if (has) {
        const int m2 = e2 - jc + P, m3 = e3 - kc + P;
        T vn1[NG], vd1[NG];
#pragma unroll
        for (int q = 0; q < NG; q++) {
          vn1[q] = tN1[q][b1];
          vd1[q] = tD1[q][b1];
        }
        const T* __restrict__ Gbase = geo[le * GP3];
        T Gc[LL::GEO];
#pragma unroll
        for (int m = 0; m < LL::GEO; m++) Gc[m] = Gbase[m];
        // fully unrolled up to 4x4 rows: the loads of later points can then be
        // issued well ahead of their use; the two copies differ only in the
        // unroll directive
        if constexpr (NG * NG <= 16) {
#pragma unroll
          for (int g23 = 0; g23 < NG * NG; g23++) {
            const int q2 = g23 % NG, q3 = g23 / NG;
            const T n3 = tN3[m3][q3][b3], d3 = tD3[m3][q3][b3];
            const T n2 = tN2[m2][q2][b2], d2 = tD2[m2][q2][b2];
            const T n23 = n2 * n3, d23 = d2 * n3, n2d3 = n2 * d3;
#pragma unroll
            for (int q1 = 0; q1 < NG; q1++) {
              const int qn = g23 * NG + q1 + 1 < GP3 ? g23 * NG + q1 + 1 : GP3 - 1;
              T Gn[LL::GEO];
#pragma unroll
              for (int m = 0; m < LL::GEO; m++) Gn[m] = Gbase[qn * LL::GEO + m];
              const T r0 = vd1[q1] * n23, r1 = vn1[q1] * d23, r2 = vn1[q1] * n2d3;
              const T* G = Gc;
              if (NC == 1) {
#pragma unroll
                for (int a1 = 0; a1 < P1; a1++)
                  acc[a1][0] += r0 * G[3 * a1] + r1 * G[3 * a1 + 1] + r2 * G[3 * a1 + 2];
              } else {
                const T gb0 = r0 * G[0] + r1 * G[3] + r2 * G[6];
                const T gb1 = r0 * G[1] + r1 * G[4] + r2 * G[7];
                const T gb2 = r0 * G[2] + r1 * G[5] + r2 * G[8];
#pragma unroll
                for (int a1 = 0; a1 < P1; a1++) {
                  const T wa0 = G[9 + 3 * a1], wa1 = G[10 + 3 * a1], wa2 = G[11 + 3 * a1];
                  if constexpr (SACC) {
                    acc[a1][0] += wa0 * gb0; acc[a1][1] += wa0 * gb1; acc[a1][2] += wa0 * gb2;
                    acc[a1][3] += wa1 * gb0; acc[a1][4] += wa1 * gb1; acc[a1][5] += wa1 * gb2;
                    acc[a1][6] += wa2 * gb0; acc[a1][7] += wa2 * gb1; acc[a1][8] += wa2 * gb2;
                  } else {
                    const T wa[3] = {wa0, wa1, wa2}, gb[3] = {gb0, gb1, gb2};
                    const T dot = wa0 * gb0 + wa1 * gb1 + wa2 * gb2;
#pragma unroll
                    for (int jj = 0; jj < 3; jj++)
                      acc[a1][jj] += lam * wa[rc] * gb[jj] + mu * wa[jj] * gb[rc] +
                                     (jj == rc ? mu * dot : T(0));
                  }
                }
              }
#pragma unroll
              for (int m = 0; m < LL::GEO; m++) Gc[m] = Gn[m];
            }
          }
        } else {
          for (int g23 = 0; g23 < NG * NG; g23++) {
            const int q2 = g23 % NG, q3 = g23 / NG;
            const T n3 = tN3[m3][q3][b3], d3 = tD3[m3][q3][b3];
            const T n2 = tN2[m2][q2][b2], d2 = tD2[m2][q2][b2];
            const T n23 = n2 * n3, d23 = d2 * n3, n2d3 = n2 * d3;
#pragma unroll
            for (int q1 = 0; q1 < NG; q1++) {
              const int qn = g23 * NG + q1 + 1 < GP3 ? g23 * NG + q1 + 1 : GP3 - 1;
              T Gn[LL::GEO];
#pragma unroll
              for (int m = 0; m < LL::GEO; m++) Gn[m] = Gbase[qn * LL::GEO + m];
              const T r0 = vd1[q1] * n23, r1 = vn1[q1] * d23, r2 = vn1[q1] * n2d3;
              const T* G = Gc;
              if (NC == 1) {
#pragma unroll
                for (int a1 = 0; a1 < P1; a1++)
                  acc[a1][0] += r0 * G[3 * a1] + r1 * G[3 * a1 + 1] + r2 * G[3 * a1 + 2];
              } else {
                const T gb0 = r0 * G[0] + r1 * G[3] + r2 * G[6];
                const T gb1 = r0 * G[1] + r1 * G[4] + r2 * G[7];
                const T gb2 = r0 * G[2] + r1 * G[5] + r2 * G[8];
#pragma unroll
                for (int a1 = 0; a1 < P1; a1++) {
                  const T wa0 = G[9 + 3 * a1], wa1 = G[10 + 3 * a1], wa2 = G[11 + 3 * a1];
                  if constexpr (SACC) {
                    acc[a1][0] += wa0 * gb0; acc[a1][1] += wa0 * gb1; acc[a1][2] += wa0 * gb2;
                    acc[a1][3] += wa1 * gb0; acc[a1][4] += wa1 * gb1; acc[a1][5] += wa1 * gb2;
                    acc[a1][6] += wa2 * gb0; acc[a1][7] += wa2 * gb1; acc[a1][8] += wa2 * gb2;
                  } else {
                    const T wa[3] = {wa0, wa1, wa2}, gb[3] = {gb0, gb1, gb2};
                    const T dot = wa0 * gb0 + wa1 * gb1 + wa2 * gb2;
#pragma unroll
                    for (int jj = 0; jj < 3; jj++)
                      acc[a1][jj] += lam * wa[rc] * gb[jj] + mu * wa[jj] * gb[rc] +
                                     (jj == rc ? mu * dot : T(0));
                  }
                }
              }
#pragma unroll
              for (int m = 0; m < LL::GEO; m++) Gc[m] = Gn[m];
            }
          }
        }
      }
        }
      // rounds over the bundle elements: in round r the items of element r
      // add their column sums (distinct window entries within a round)
      // p <= 2 (STAGED): the geometry rows are no longer needed once the sums
      // are in registers; their LDS takes the sums of GS elements at a time,
      // which are then reduced per window entry in fixed element order (as
      // phase C below) and added to the window, group after group.  p = 3:
      // element rounds (measured faster there).
      if (EQE && c0 == 0) {
#pragma unroll
        for (int k = 0; k < NEQV; k++) {
          const int t = tid + k * kBlock;
          if (t < NT * 64) eqw[buf][t] = eqv[k];
        }
      }
      constexpr bool STAGED = P <= 2;
      if constexpr (STAGED) {
      constexpr int GS0 = (CH * SLQ * LL::GEO) / (NEN * P1 * NS);
      constexpr int GS = GS0 < 1 ? 1 : (GS0 > CH ? CH : GS0);
      T (*stg)[NEN][P1][NS] = reinterpret_cast<T (*)[NEN][P1][NS]>(&geo[0][0]);
      for (int g0 = 0; g0 < nch; g0 += GS) {
        const int g1 = g0 + GS < nch ? g0 + GS : nch;
        lds_barrier(); // geometry reads (or the previous group) done
        if (has && le >= g0 && le < g1) {
#pragma unroll
          for (int a1 = 0; a1 < P1; a1++)
#pragma unroll
            for (int s = 0; s < NS; s++) stg[le - g0][b][a1][s] = acc[a1][s];
        }
        __syncthreads();
        for (int t = tid; t < P1 * P1 * W1 * W1; t += kBlock) {
          const int a1 = t % P1, r = t / P1;
          const int cb1 = r % P1, r2 = r / P1;
          const int cjr = r2 % W1, ckr = r2 / W1;
          const int cjj = jc - P + cjr, ckk = kc - P + ckr;
          T sm[NS];
#pragma unroll
          for (int m = 0; m < NS; m++) sm[m] = 0;
          bool any = false;
          for (int l = g0; l < g1; l++) {
            const int cb2 = cjj - be2[c0 + l], cb3 = ckk - be3[c0 + l];
            if (cb2 < 0 || cb2 > P || cb3 < 0 || cb3 > P) continue;
            any = true;
            const int cb = cb1 + P1 * (cb2 + P1 * cb3);
#pragma unroll
            for (int m = 0; m < NS; m++) sm[m] += stg[l - g0][cb][a1][m];
          }
          if (!any) continue;
          const int slot = (e1 + a1) % P1;
          const int di = cb1 - a1, dj = cjj - jc, dk = ckk - kc;
          const int nbr = ((dk + P) * W1 + (dj + P)) * W1 + (di + P);
          if (NC == 1) {
            win[slot][0][nbr][0] += sm[0];
          } else if (SACC) {
            const T tr = sm[0] + sm[4] + sm[8];
#pragma unroll
            for (int i = 0; i < 3; i++)
#pragma unroll
              for (int j = 0; j < 3; j++)
                win[slot][i][nbr][j] += lam * sm[3 * i + j] + mu * sm[3 * j + i] + (i == j ? mu * tr : T(0));
          } else {
#pragma unroll
            for (int j = 0; j < 3; j++) win[slot][0][nbr][j] += sm[j];
          }
        }
      }
      } else {
      // Each thread's window entries are distinct, so all of them are read
      // first and written after (one LDS round trip per round, not one per
      // entry).
      const int cj = e2 + b2, ck = e3 + b3;
      constexpr int NV = NC == 1 ? 1 : (SACC ? 9 : 3); // window values per row function
      T* wp[P1];
#pragma unroll
      for (int a1 = 0; a1 < P1; a1++) {
        const int slot = (e1 + a1) % P1;
        const int di = b1 - a1, dj = cj - jc, dk = ck - kc;
        const int nbr = ((dk + P) * W1 + (dj + P)) * W1 + (di + P);
        wp[a1] = &win[slot][0][nbr][0];
      }
      T add[P1][NV];
#pragma unroll
      for (int a1 = 0; a1 < P1; a1++) {
        const T* sv = acc[a1];
        if (NC == 1) {
          add[a1][0] = sv[0];
        } else if (SACC) {
          const T tr = sv[0] + sv[4] + sv[8];
#pragma unroll
          for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < 3; j++)
              add[a1][3 * i + j] = lam * sv[3 * i + j] + mu * sv[3 * j + i] + (i == j ? mu * tr : T(0));
        } else {
#pragma unroll
          for (int j = 0; j < 3; j++) add[a1][j] = sv[j];
        }
      }
      // offset of value v of a row function inside win[slot]: (i, j) of the
      // 3x3 block -> [i][nbr][j]
      constexpr int ISTR = LL::WN * NC;
      for (int r = 0; r < nch; r++) {
        lds_barrier();
        if (has && le == r) {
          T cur[P1][NV];
#pragma unroll
          for (int a1 = 0; a1 < P1; a1++)
#pragma unroll
            for (int v = 0; v < NV; v++)
              cur[a1][v] = wp[a1][(NV == 9 ? v / 3 : 0) * ISTR + (NV == 9 ? v % 3 : v)];
#pragma unroll
          for (int a1 = 0; a1 < P1; a1++)
#pragma unroll
            for (int v = 0; v < NV; v++)
              wp[a1][(NV == 9 ? v / 3 : 0) * ISTR + (NV == 9 ? v % 3 : v)] = cur[a1][v] + add[a1][v];
        }
      }
      }
      } else if constexpr (SEMI) {
      // Larger Gauss rules: loop over the (q2, q3) rows with the q1 row
      // unrolled; the next point's geometry row is loaded into registers while
      // the current one is used (across rows too), the column node's
      // direction-1 basis values are held in registers.
      for (int t = tid; t < nch * NEN; t += kBlock) {
        const int le = t / NEN, b = t % NEN;
        const int b1 = b % P1, b2 = (b / P1) % P1, b3 = b / (P1 * P1);
        const int e2 = be2[c0 + le], e3 = be3[c0 + le];
        const int m2 = e2 - jc + P, m3 = e3 - kc + P;
        T vn1[NG], vd1[NG];
#pragma unroll
        for (int q = 0; q < NG; q++) {
          vn1[q] = tN1[q][b1];
          vd1[q] = tD1[q][b1];
        }
        T acc[P1][NS];
#pragma unroll
        for (int a1 = 0; a1 < P1; a1++)
#pragma unroll
          for (int s = 0; s < NS; s++) acc[a1][s] = 0;
        const T* __restrict__ Gbase = geo[le * GP3];
        T Gc[LL::GEO];
#pragma unroll
        for (int m = 0; m < LL::GEO; m++) Gc[m] = Gbase[m];
        for (int g23 = 0; g23 < NG * NG; g23++) {
          const int q2 = g23 % NG, q3 = g23 / NG;
          const T n3 = tN3[m3][q3][b3], d3 = tD3[m3][q3][b3];
          const T n2 = tN2[m2][q2][b2], d2 = tD2[m2][q2][b2];
          const T n23 = n2 * n3, d23 = d2 * n3, n2d3 = n2 * d3;
#pragma unroll
          for (int q1 = 0; q1 < NG; q1++) {
            // next row (the last point reloads itself: in bounds, unused)
            const int qn = g23 * NG + q1 + 1 < GP3 ? g23 * NG + q1 + 1 : GP3 - 1;
            T Gn[LL::GEO];
#pragma unroll
            for (int m = 0; m < LL::GEO; m++) Gn[m] = Gbase[qn * LL::GEO + m];
            const T r0 = vd1[q1] * n23, r1 = vn1[q1] * d23, r2 = vn1[q1] * n2d3;
            const T* G = Gc;
            if (NC == 1) {
#pragma unroll
              for (int a1 = 0; a1 < P1; a1++)
                acc[a1][0] += r0 * G[3 * a1] + r1 * G[3 * a1 + 1] + r2 * G[3 * a1 + 2];
            } else {
              const T gb0 = r0 * G[0] + r1 * G[3] + r2 * G[6];
              const T gb1 = r0 * G[1] + r1 * G[4] + r2 * G[7];
              const T gb2 = r0 * G[2] + r1 * G[5] + r2 * G[8];
#pragma unroll
              for (int a1 = 0; a1 < P1; a1++) {
                const T wa0 = G[9 + 3 * a1], wa1 = G[10 + 3 * a1], wa2 = G[11 + 3 * a1];
                if (SACC) {
                  acc[a1][0] += wa0 * gb0; acc[a1][1] += wa0 * gb1; acc[a1][2] += wa0 * gb2;
                  acc[a1][3] += wa1 * gb0; acc[a1][4] += wa1 * gb1; acc[a1][5] += wa1 * gb2;
                  acc[a1][6] += wa2 * gb0; acc[a1][7] += wa2 * gb1; acc[a1][8] += wa2 * gb2;
                } else {
                  const T wa[3] = {wa0, wa1, wa2}, gb[3] = {gb0, gb1, gb2};
                  const int ic = split * NCR;
                  const T dot = wa0 * gb0 + wa1 * gb1 + wa2 * gb2;
#pragma unroll
                  for (int jj = 0; jj < 3; jj++)
                    acc[a1][jj] += lam * wa[ic] * gb[jj] + mu * wa[jj] * gb[ic] +
                                   (jj == ic ? mu * dot : T(0));
                }
              }
            }
#pragma unroll
            for (int m = 0; m < LL::GEO; m++) Gc[m] = Gn[m];
          }
        }
#pragma unroll
        for (int a1 = 0; a1 < P1; a1++)
#pragma unroll
          for (int s = 0; s < NS; s++) stage[le][b][a1][s] = acc[a1][s];
      }
      } else if constexpr (!PIPE) {
      // one thread per (element, column node b), Gauss points in fixed order
      for (int t = tid; t < nch * NEN; t += kBlock) {
        const int le = t / NEN, b = t % NEN;
        const int b1 = b % P1, b2 = (b / P1) % P1, b3 = b / (P1 * P1);
        const int e2 = be2[c0 + le], e3 = be3[c0 + le];
        const int m2 = e2 - jc + P, m3 = e3 - kc + P;
        T acc[P1][NS];
#pragma unroll
        for (int a1 = 0; a1 < P1; a1++)
#pragma unroll
          for (int s = 0; s < NS; s++) acc[a1][s] = 0;
        for (int q3 = 0; q3 < NG; q3++) {
          const T n3 = tN3[m3][q3][b3], d3 = tD3[m3][q3][b3];
          for (int q2 = 0; q2 < NG; q2++) {
            const T n2 = tN2[m2][q2][b2], d2 = tD2[m2][q2][b2];
            const T n23 = n2 * n3, d23 = d2 * n3, n2d3 = n2 * d3;
#pragma unroll
            for (int q1 = 0; q1 < NG; q1++) {
              const int pr = le * GP3 + (q3 * NG + q2) * NG + q1;
              const T n1 = tN1[q1][b1], d1 = tD1[q1][b1];
              const T r0 = d1 * n23, r1 = n1 * d23, r2 = n1 * n2d3;
              const T* G = geo[pr];
              if (NC == 1) {
#pragma unroll
                for (int a1 = 0; a1 < P1; a1++)
                  acc[a1][0] += r0 * G[3 * a1] + r1 * G[3 * a1 + 1] + r2 * G[3 * a1 + 2];
              } else {
                const T gb0 = r0 * G[0] + r1 * G[3] + r2 * G[6];
                const T gb1 = r0 * G[1] + r1 * G[4] + r2 * G[7];
                const T gb2 = r0 * G[2] + r1 * G[5] + r2 * G[8];
#pragma unroll
                for (int a1 = 0; a1 < P1; a1++) {
                  const T wa0 = G[9 + 3 * a1], wa1 = G[10 + 3 * a1], wa2 = G[11 + 3 * a1];
                  if (SACC) {
                    acc[a1][0] += wa0 * gb0; acc[a1][1] += wa0 * gb1; acc[a1][2] += wa0 * gb2;
                    acc[a1][3] += wa1 * gb0; acc[a1][4] += wa1 * gb1; acc[a1][5] += wa1 * gb2;
                    acc[a1][6] += wa2 * gb0; acc[a1][7] += wa2 * gb1; acc[a1][8] += wa2 * gb2;
                  } else {
                    const T wa[3] = {wa0, wa1, wa2}, gb[3] = {gb0, gb1, gb2};
                    const int ic = split * NCR;
                    const T dot = wa0 * gb0 + wa1 * gb1 + wa2 * gb2;
#pragma unroll
                    for (int jj = 0; jj < 3; jj++)
                      acc[a1][jj] += lam * wa[ic] * gb[jj] + mu * wa[jj] * gb[ic] +
                                     (jj == ic ? mu * dot : T(0));
                  }
                }
              }
            }
          }
        }
#pragma unroll
        for (int a1 = 0; a1 < P1; a1++)
#pragma unroll
          for (int s = 0; s < NS; s++) stage[le][b][a1][s] = acc[a1][s];
      }
      } else {
      // One thread per (element, column node b); the Gauss points are fully
      // unrolled with the next point's geometry row loaded into registers
      // while the current one is used, and the column node's 1D basis
      // values held in registers.
      for (int t = tid; t < nch * NEN; t += kBlock) {
        const int le = t / NEN, b = t % NEN;
        const int b1 = b % P1, b2 = (b / P1) % P1, b3 = b / (P1 * P1);
        const int e2 = be2[c0 + le], e3 = be3[c0 + le];
        const int m2 = e2 - jc + P, m3 = e3 - kc + P;
        T vn1[NG], vd1[NG], vn2[NG], vd2[NG], vn3[NG], vd3[NG];
#pragma unroll
        for (int q = 0; q < NG; q++) {
          vn1[q] = tN1[q][b1]; vd1[q] = tD1[q][b1];
          vn2[q] = tN2[m2][q][b2]; vd2[q] = tD2[m2][q][b2];
          vn3[q] = tN3[m3][q][b3]; vd3[q] = tD3[m3][q][b3];
        }
        T acc[P1][NS];
#pragma unroll
        for (int a1 = 0; a1 < P1; a1++)
#pragma unroll
          for (int s = 0; s < NS; s++) acc[a1][s] = 0;
        const T* __restrict__ Gbase = geo[le * GP3];
        T Gc[LL::GEO];
#pragma unroll
        for (int m = 0; m < LL::GEO; m++) Gc[m] = Gbase[m];
#pragma unroll
        for (int q = 0; q < GP3; q++) {
          T Gn[LL::GEO];
          if (q + 1 < GP3) {
#pragma unroll
            for (int m = 0; m < LL::GEO; m++) Gn[m] = Gbase[(q + 1) * LL::GEO + m];
          }
          const int q1 = q % NG, q2 = (q / NG) % NG, q3 = q / (NG * NG);
          const T n23 = vn2[q2] * vn3[q3], d23 = vd2[q2] * vn3[q3], n2d3 = vn2[q2] * vd3[q3];
          const T r0 = vd1[q1] * n23, r1 = vn1[q1] * d23, r2 = vn1[q1] * n2d3;
          const T* G = Gc;
          if (NC == 1) {
#pragma unroll
            for (int a1 = 0; a1 < P1; a1++)
              acc[a1][0] += r0 * G[3 * a1] + r1 * G[3 * a1 + 1] + r2 * G[3 * a1 + 2];
          } else {
            const T gb0 = r0 * G[0] + r1 * G[3] + r2 * G[6];
            const T gb1 = r0 * G[1] + r1 * G[4] + r2 * G[7];
            const T gb2 = r0 * G[2] + r1 * G[5] + r2 * G[8];
#pragma unroll
            for (int a1 = 0; a1 < P1; a1++) {
              const T wa0 = G[9 + 3 * a1], wa1 = G[10 + 3 * a1], wa2 = G[11 + 3 * a1];
              if (SACC) {
                acc[a1][0] += wa0 * gb0; acc[a1][1] += wa0 * gb1; acc[a1][2] += wa0 * gb2;
                acc[a1][3] += wa1 * gb0; acc[a1][4] += wa1 * gb1; acc[a1][5] += wa1 * gb2;
                acc[a1][6] += wa2 * gb0; acc[a1][7] += wa2 * gb1; acc[a1][8] += wa2 * gb2;
              } else {
                const T wa[3] = {wa0, wa1, wa2}, gb[3] = {gb0, gb1, gb2};
                const int ic = split * NCR;
                const T dot = wa0 * gb0 + wa1 * gb1 + wa2 * gb2;
#pragma unroll
                for (int jj = 0; jj < 3; jj++)
                  acc[a1][jj] += lam * wa[ic] * gb[jj] + mu * wa[jj] * gb[ic] +
                                 (jj == ic ? mu * dot : T(0));
              }
            }
          }
          if (q + 1 < GP3) {
#pragma unroll
            for (int m = 0; m < LL::GEO; m++) Gc[m] = Gn[m];
          }
        }
#pragma unroll
        for (int a1 = 0; a1 < P1; a1++)
#pragma unroll
          for (int s = 0; s < NS; s++) stage[le][b][a1][s] = acc[a1][s];
      }
      }
      __syncthreads();

      // ---- phase C: ordered reduction of the chunk into the row window ------
      if (!ORD)
      for (int t = tid; t < P1 * P1 * W1 * W1; t += kBlock) {
        const int a1 = t % P1, r = t / P1;
        const int b1 = r % P1, r2 = r / P1;
        const int cjr = r2 % W1, ckr = r2 / W1;
        const int cj = jc - P + cjr, ck = kc - P + ckr;
        T s[NS];
#pragma unroll
        for (int m = 0; m < NS; m++) s[m] = 0;
        bool any = false;
        for (int le = 0; le < nch; le++) {
          const int b2 = cj - be2[c0 + le], b3 = ck - be3[c0 + le];
          if (b2 < 0 || b2 > P || b3 < 0 || b3 > P) continue;
          any = true;
          const int b = b1 + P1 * (b2 + P1 * b3);
#pragma unroll
          for (int m = 0; m < NS; m++) s[m] += stage[le][b][a1][m];
        }
        if (!any) continue;
        const int slot = (e1 + a1) % P1;
        const int di = b1 - a1, dj = cj - jc, dk = ck - kc;
        const int nbr = ((dk + P) * W1 + (dj + P)) * W1 + (di + P);
        if (NC == 1) {
          win[slot][0][nbr][0] += s[0];
        } else if (SACC) {
          const T tr = s[0] + s[4] + s[8];
#pragma unroll
          for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < 3; j++)
              win[slot][i][nbr][j] += lam * s[3 * i + j] + mu * s[3 * j + i] + (i == j ? mu * tr : T(0));
        } else {
#pragma unroll
          for (int j = 0; j < 3; j++) win[slot][0][nbr][j] += s[j];
        }
      }
      __syncthreads();
    }

    // ---- phase D (last layer): rows e1 .. e1+p are complete ------------------
    if (e1 == a.nel1 - 1) {
      for (int i = e1; i <= e1 + P; i++) {
        const int slot = i % P1;
        row_out(i, i == e1, buf, false);
        __syncthreads();
        for (int t = tid; t < NCR * WN * NC; t += kBlock) (&win[slot][0][0][0])[t] = T(0);
        if (tid < NC) rwin[slot][tid] = T(0);
        __syncthreads();
      }
    }
  }
}

// Single patch: the LDS arrays are separate __shared__ variables.  The
// Gauss-point slab variant (HALF = 2) is built for three workgroups per CU.
template <int P, int NG, int NC, typename T, int SPLIT, bool HAS_RHS, int HALF>
__global__ __launch_bounds__(kBlock, HALF == 2 ? 3 : 1) void k_assemble_lines(
    const AsmArgs* __restrict__ args)
{
  ConstArgs& a = *const_args(args);
  using LL = LineLds<P, NG, NC, T, SPLIT, HAS_RHS, HALF>;
  constexpr int P1 = P + 1;
  // register-pipelined phase B where the unrolled Gauss loop stays small;
  // ordered window updates (no stage) where the whole bundle is one chunk
  constexpr bool PIPE = LL::GP3 <= 27;
  constexpr bool ORD = (HALF == 0 || HALF == 2) && LL::CH * LL::NEN <= kBlock;
  __shared__ T win[P1][LL::NCR][LL::WN][NC];
  __shared__ T geo[LL::CH * LL::SLQ][LL::GEO];
  __shared__ T stage[ORD ? 1 : LL::CH][LL::NEN][P1][LL::NS];
  __shared__ T rstage[HAS_RHS ? LL::CH * LL::SLQ * (ORD ? P1 : LL::NRHS) : 1];
  __shared__ T rwin[P1][NC];
  __shared__ T tN1[NG][P1], tD1[NG][P1];
  __shared__ T tN2[P1][NG][P1], tD2[P1][NG][P1];
  __shared__ T tN3[P1][NG][P1], tD3[P1][NG][P1];
  __shared__ int be2[LL::NB], be3[LL::NB];
  __shared__ int eqw[2][LL::PFD ? LL::NT * 64 : 1];
  __shared__ int64_t pbase[2][LL::NCR];
  __shared__ int prow[2][LL::NCR];
  __shared__ int nbundle;
  line_impl<P, NG, NC, T, SPLIT, HAS_RHS, HALF, PIPE, ORD, !PIPE>(a, blockIdx.x, blockIdx.y, win, geo, stage,
                                                      rstage, rwin, tN1, tD1, tN2, tD2, tN3, tD3,
                                                      be2, be3, eqw, pbase, prow, &nbundle);
}

// Persistent batch assembly of a batch's patches of degree 3 (ng = 4; degrees
// 1 and 2: k_lines_batch), with the single-patch kernel's own phase-B and
// window-update variants and its own register and LDS budget.  Work items are
// whole lines of a patch sorted by decreasing cost; blocks take the next item
// from the degree's queue counter, so load balances over patches of uneven
// size.  Each line's rows are written by exactly one block, so the result does
// not depend on which block takes which item.  HALF: the element-chunk variant
// (BatchTune::half).
template <int P, typename T, bool HAS_RHS, int HALF>
__global__ __launch_bounds__(kBlock, 3) void k_assemble_batch(const AsmArgs* __restrict__ args,
                                                           const LineItem* __restrict__ items,
                                                           int nitems, int* __restrict__ queue)
{
  constexpr int NG = P + 1;
  using LL = LineLds<P, NG, 1, T, 1, HAS_RHS, HALF>;
  constexpr int P1 = P + 1;
  constexpr bool PIPE = LL::GP3 <= 27;
  constexpr bool ORD = (HALF == 0 || HALF == 2) && LL::CH * LL::NEN <= kBlock;
  __shared__ T win[P1][LL::NCR][LL::WN][1];
  __shared__ T geo[LL::CH * LL::SLQ][LL::GEO];
  __shared__ T stage[ORD ? 1 : LL::CH][LL::NEN][P1][LL::NS];
  __shared__ T rstage[HAS_RHS ? LL::CH * LL::SLQ * (ORD ? P1 : LL::NRHS) : 1];
  __shared__ T rwin[P1][1];
  __shared__ T tN1[NG][P1], tD1[NG][P1];
  __shared__ T tN2[P1][NG][P1], tD2[P1][NG][P1];
  __shared__ T tN3[P1][NG][P1], tD3[P1][NG][P1];
  __shared__ int be2[LL::NB], be3[LL::NB];
  __shared__ int eqw[2][LL::PFD ? LL::NT * 64 : 1];
  __shared__ int64_t pbase[2][LL::NCR];
  __shared__ int prow[2][LL::NCR];
  __shared__ int nbundle;
  __shared__ int next;
  while (true) {
    if (threadIdx.x == 0) next = atomicAdd(queue, 1);
    __syncthreads();
    const int it = __builtin_amdgcn_readfirstlane(next);
    if (it >= nitems) break;
    const LineItem w = items[it];
    ConstArgs& a = const_args(args)[w.patch];
    line_impl<P, NG, 1, T, 1, HAS_RHS, HALF, PIPE, ORD, !PIPE>(a, w.j0 + a.n2 * w.k, 0, win, geo, stage, rstage,
                                                               rwin, tN1, tD1, tN2, tD2, tN3, tD3,
                                                               be2, be3, eqw, pbase, prow, &nbundle);
    __syncthreads();
  }
}

template <int P, int NG, int NC, typename T, int HALF>
static void launch_direct(Context& c, const AsmArgs& a, bool rhs)
{
  // One block per line holds all three row components where the window fits
  // the LDS (p = 3 with full chunks of 4x4x4 points: 144 KB in FP64, one
  // workgroup per CU), measured 1.7-1.9x faster than three blocks that each
  // recompute the geometry rows and the column gradients; half chunks and
  // 5x5x5 rules keep three blocks (their window and chunk exceed 160 KB).
  constexpr int SPLIT = (NC == 3 && P >= 3 && (HALF || NG > 4)) ? 3 : 1;
  const dim3 grid(a.n2 * a.n3, SPLIT);
  const AsmArgs* d = static_cast<const AsmArgs*>(c.d_asmargs);
  if (sizeof(T) == 8 && rhs)
    k_assemble_lines<P, NG, NC, T, SPLIT, sizeof(T) == 8, HALF><<<grid, kBlock, 0, c.stream>>>(d);
  else
    k_assemble_lines<P, NG, NC, T, SPLIT, false, HALF><<<grid, kBlock, 0, c.stream>>>(d);
}

template <int P, int NG, int NC, typename T>
static void launch_direct_v(Context& c, const AsmArgs& a, bool rhs, int variant)
{
  // built-in choice: at p = 2, Gauss-point slabs for 3x3x3 points (FP32, 64^3
  // elasticity: 3.9 ms against 5.2 ms for full chunks), else half chunks for
  // FP64 elasticity, which keep two workgroups per CU
  constexpr bool SLABS = P == 2 && NG == 3;
  if (variant < 0) variant = SLABS ? 2 : (sizeof(T) == 8 && NC == 3 && P < 3) ? 1 : 0;
  if constexpr (SLABS) {
    if (variant == 2) {
      launch_direct<P, NG, NC, T, 2>(c, a, rhs);
      return;
    }
  }
  if (variant == 1) launch_direct<P, NG, NC, T, 1>(c, a, rhs);
  else launch_direct<P, NG, NC, T, 0>(c, a, rhs);
}

template <int P, int NG>
static int launch_lines_direct(Context& c, const AsmArgs& a, bool fp32, bool rhs, int variant)
{
  if (c.ncomp == 1)
    fp32 ? launch_direct_v<P, NG, 1, float>(c, a, rhs, variant)
         : launch_direct_v<P, NG, 1, double>(c, a, rhs, variant);
  else
    fp32 ? launch_direct_v<P, NG, 3, float>(c, a, rhs, variant)
         : launch_direct_v<P, NG, 3, double>(c, a, rhs, variant);
  IFEM_HIP(hipGetLastError());
  return IFEM_GPU_OK;
}

} // namespace ifem
