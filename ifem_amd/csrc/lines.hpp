// lines.hpp -- line kernels of the numeric volume assembly: K and b of the
// rows of node lines from the geometry records, by sum factorisation.
//
// Row-owned: a workgroup owns the rows i0 <= i < i1 of the control points of
// one line (vector problems) or of NL neighbouring lines (j, k fixed per
// line) and walks the element layers e1 that touch them.  For the row
// functions a = (a1, a2, a3) of a line, a2 and a3 are fixed by the line, and
//   S_ab = sum_kl sum_q G_kl(q) A1_k A2_k A3_k (q) B1_l B2_l B3_l (q)
// (A_k, B_l: 1D value, or derivative in direction k resp. l; scalar problems:
// G_kl = M_kl; vector problems, for each component pair (i, j): G_kl =
// w Jinv_ki Jinv_lj) is contracted direction by direction, over the Gauss
// points of ALL elements of the layer that touch the line:
//   units    one thread per (q1, k, l, slot): T1(q3; dj) = sum_q2, then
//            T2(dk, dj) = sum_q3, in registers.  slot: the component pair
//            (i, j) of one line (9 slots), or the line (scalar problems).
//   columns  one thread per (slot, dk, dj): sum over (q1, k, l) with the
//            direction-1 functions into the P+1 open rows of its column line,
//            in registers (k, l = 2, 3 carry the same direction-1 functions,
//            so nine (k, l) merge to four); exchange through LDS.
//   row out  after layer e1 row e1 is complete; it goes through LDS to
//            coalesced stores.  A row whose whole neighbour window is free
//            (its CSR length says so) is written by position; the others are
//            compacted by ballots over their neighbours' equation numbers.
// Per line and layer that is NG*9*slots * (Q*Q + ...) multiply-adds with Q =
// (P+1)*NG points per direction instead of (P+1)^2*NEN*NG^3 products per
// component pair, and the sum over the layer's elements needs no reduction.
// Bound: the units read two LDS values per four FP64 operations (one in
// scalar problems), which makes LDS bandwidth and FP64 issue about equal (34 %
// and 38 % of the time at 64^3 p = 2 elasticity, two waves per SIMD); the rest
// is latency between the barriers.  Against direct quadrature with one line
// per workgroup (lines_direct.hpp): 64^3 p = 2 elasticity 6.39 -> 4.15 ms, two
// 16x32x32 patches 0.89 -> 0.65 ms each, 45x37x51 p = 2 Poisson 1.12 -> 0.26 ms.
// Each XCD runs a contiguous range of groups: 2.0 GB are fetched instead of 4.9
// at 64^3 elasticity (the records are 0.57 GB).
// Every K entry is written once, without atomics, and all sums have a fixed
// order that does not depend on how the rows are split into workgroups, so
// results are bitwise reproducible.
#pragma once

#include <cstdint>
#include <type_traits>

#include "asmargs.hpp"

namespace ifem {

// Rows i0 <= i < i1 of lines j0 .. j0+nl-1 at k of a patch of a batch.
struct LineItem {
  int patch, j0, nl, k, i0, i1;
};

constexpr int line_max(int a, int b) { return a > b ? a : b; }

// Row stride (in values) of the Gauss-point rows in LDS: even (16-byte
// aligned rows of doubles) and 2 or 14 modulo 16, so that rows of neighbouring
// components start in different banks.
constexpr int line_row_stride(int n)
{
  int r = n + (n & 1);
  while (r % 16 != 2 && r % 16 != 14) r += 2;
  return r;
}

template <int P, int NG, int NC>
struct LineCfg {
  static_assert(P <= 2, "the direction-2 factors and T2 of a unit are held in registers");
  static constexpr int P1 = P + 1, W1 = 2 * P + 1, WW = W1 * W1, WN = W1 * WW;
  static constexpr int GP3 = NG * NG * NG;
  // slots: component pairs, or lines per workgroup (as many as fill the
  // workgroup's units and column threads about equally)
  static constexpr int SL = NC == 3 ? 9
                            : P == 1 ? (NG == 2 ? 12 : 8)
                                     : 8;
  static constexpr int NL = NC == 3 ? 1 : SL;     // lines per workgroup (most)
  static constexpr int NU = NG * 9 * SL;          // units
  static constexpr int NR = NG * NL;              // right-hand side units
  static constexpr int NCT = SL * WW;             // column threads
  static constexpr int TH = (line_max(NU + NR, NCT) + 63) / 64 * 64;
  static constexpr int Q2 = P1 * NG;              // points per line in direction 2
  static constexpr int NE2 = NL + P;              // elements in direction 2
  static constexpr int NQ2 = NE2 * NG;
  static constexpr int RS = line_row_stride(NG * NQ2);
  static constexpr int NROW = NC == 3 ? 3 : NL;   // rows per line position
  static constexpr int NCOL = WN * NC;            // columns of a full row
  static constexpr int ES = WW | 1;               // exchange: odd stride per unit
  // offsets of a group's records in 64 bits (WIDE): where NE2 elements of
  // direction 2 lie 2^31 values apart.  In 32 bits elsewhere: the wider
  // offsets cost vector problems of degree 2 with a body force their second
  // wave per SIMD (249 -> 256 registers and more)
  static constexpr bool wide(int nel1)
  {
    constexpr int64_t rec = (int64_t)GeoRec<NC>::N * GP3;
    return ((int64_t)(NE2 - 1) * nel1 + 1) * rec > INT32_MAX;
  }
};

template <int P, int NG, int NC, typename T, bool RHS>
struct LineShared {
  using C = LineCfg<P, NG, NC>;
  // Gauss-point components of a chunk: w Jinv (9), Jinv (9) [, w, 1], or M (6) [, w f]
  static constexpr int NCOMP = NC == 3 ? (RHS ? 20 : 18) : (RHS ? 7 : 6);
  static constexpr int CHUNK = NCOMP * NG * C::RS;
  static constexpr int EX = (C::NU + (RHS ? C::NR : 0)) * C::ES;
  // two chunk buffers, or the exchange
  alignas(16) T buf[line_max(2 * CHUNK, EX)];
  alignas(16) double row[C::SL * C::WN]; // complete rows, per column line and slot
  alignas(16) T c3[5][C::P1 * NG][C::P1];
  double rrow[C::NL];
  int64_t base[C::NROW];
  int req[C::NROW], full[C::NROW];
};

// Waits for the wave's LDS operations, then for the workgroup; global loads
// stay in flight.
__device__ __forceinline__ void line_barrier()
{
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

typedef const __attribute__((address_space(4))) double* ConstTable;

// Equation number of neighbour DOF t (node offset t / NC in the (2p+1)^3
// window around node (i, jc, kc), component t % NC); -2 outside the patch.
template <int P, int NC>
__device__ __forceinline__ int window_eq(ConstArgs& a, int i, int jc, int kc, int t)
{
  constexpr int W1 = 2 * P + 1;
  const int nbr = t / NC, cc = t % NC;
  const int ii = i + nbr % W1 - P, jj = jc + (nbr / W1) % W1 - P, kk = kc + nbr / (W1 * W1) - P;
  if (t >= W1 * W1 * W1 * NC || ii < 0 || ii >= a.n1 || jj < 0 || jj >= a.n2 || kk < 0 || kk >= a.n3)
    return -2;
  return a.eq[((int64_t)ii + (int64_t)a.n1 * (jj + (int64_t)a.n2 * kk)) * NC + cc];
}

// ACCUM: the rows are shared with other patches, values are added to them.
// WIDE: see LineCfg::wide.
template <int P, int NG, int NC, typename T, bool RHS, bool ACCUM, bool WIDE>
__device__ __forceinline__ void line_group(ConstArgs& a, const int j0, const int nl, const int kc,
                                           const int i0, const int i1,
                                           LineShared<P, NG, NC, T, RHS>& sh)
{
  using C = LineCfg<P, NG, NC>;
  using S = LineShared<P, NG, NC, T, RHS>;
  constexpr int P1 = C::P1, W1 = C::W1, WW = C::WW, WN = C::WN, SL = C::SL, NL = C::NL, TH = C::TH;
  constexpr int NCOMP = S::NCOMP, RN = GeoRec<NC>::N;
  const int tid = threadIdx.x;

  // ---- the thread's unit (surplus threads repeat unit 0 and store nothing) --
  const bool runit = RHS && tid >= C::NU && tid < C::NU + C::NR;
  const bool unit = tid < C::NU || runit;
  const int u = tid < C::NU ? tid : 0;
  const int ri = runit ? tid - C::NU : 0;
  const int us = runit ? (NC == 1 ? ri % NL : 0) : u % SL;
  const int kl = runit ? 0 : (u / SL) % 9;
  const int q1 = runit ? ri / NL : u / (9 * SL);
  const int uk = kl / 3, ul = kl % 3;
  const int lj = NC == 1 ? us : 0;
  int oA, oB = 0;
  if (NC == 3) {
    oA = ((runit ? 18 : 3 * uk + us / 3) * NG + q1) * C::RS;
    oB = ((runit ? 19 : 9 + 3 * ul + us % 3) * NG + q1) * C::RS;
  } else {
    const int lo = uk < ul ? uk : ul, hi = uk < ul ? ul : uk;
    oA = ((runit ? 6 : lo == 0 ? hi : lo + hi + 1) * NG + q1) * C::RS + lj * NG;
  }
  const int v2 = runit ? 4 : 2 * (uk == 1) + (ul == 1);
  const int v3 = runit ? 4 : 2 * (uk == 2) + (ul == 2);

  // ---- factors A B of directions 2 and 3, [variant][point][column function];
  // variants 2*(A is the derivative) + (B is the derivative); variant 4 (right-
  // hand side): A alone, placed so that all its sums meet in column dj = dk = 0
  auto factor = [&](const double* tN, const double* tD, int e, int g, int m, int b, int v) -> T {
    const int at = (e * NG + g) * P1;
    if (v == 4) return b == P - m ? (T)tN[at + P - m] : T(0);
    return (T)((v & 2 ? tD : tN)[at + P - m] * (v & 1 ? tD : tN)[at + b]);
  };
  for (int t = tid; t < 5 * C::Q2 * P1; t += TH) {
    const int b = t % P1, g = (t / P1) % C::Q2, v = t / (P1 * C::Q2);
    const int m = g / NG, e = kc - P + m;
    sh.c3[v][g][b] = e >= 0 && e < a.nel3 ? factor(a.tabN3, a.tabD3, e, g % NG, m, b, v) : T(0);
  }
  T c2r[C::Q2][P1];
#pragma unroll
  for (int g = 0; g < C::Q2; g++) {
    const int m = g / NG, e = j0 + lj - P + m;
    const bool ok = lj < nl && e >= 0 && e < a.nel2;
#pragma unroll
    for (int b = 0; b < P1; b++) c2r[g][b] = ok ? factor(a.tabN2, a.tabD2, e, g % NG, m, b, v2) : T(0);
  }

  // ---- Gauss-point loader: the items (element m2, component, point) of a
  // chunk (element row m3); the next chunk's are
  // loaded into registers while the current one is used
  constexpr int NLC = NC == 3 ? (RHS ? 10 : 9) : NCOMP; // loaded components
  constexpr int NIT = C::NE2 * NLC * C::GP3;
  constexpr int NI = (NIT + TH - 1) / TH;
  using Offset = std::conditional_t<WIDE, int64_t, int>;
  Offset goff[NI];
  int dst[NI];
#pragma unroll
  for (int n = 0; n < NI; n++) {
    const int it = tid + n * TH;
    const int g = it % C::GP3, c = (it / C::GP3) % NLC, m2 = it / (C::GP3 * NLC);
    const int e2 = j0 - P + m2;
    const int g1 = g % NG, g2 = (g / NG) % NG, g3 = g / (NG * NG);
    const bool ok = it < NIT && m2 < nl + P && e2 >= 0 && e2 < a.nel2;
    goff[n] = ok ? ((Offset)m2 * a.nel1 * RN + c) * C::GP3 + g : -1;
    const int cl = NC == 3 && c == 9 ? 18 : c;
    dst[n] = it < NIT ? (cl * NG + g1) * C::RS + g3 * C::NQ2 + m2 * NG + g2 : -1;
  }
  double pv[NI], pw[NC == 3 ? NI : 1];
  auto load_chunk = [&](int e1, int m3) {
    const double* __restrict__ src =
        a.gp_geo +
        ((int64_t)e1 + (int64_t)a.nel1 * ((j0 - P) + (int64_t)a.nel2 * (kc - P + m3))) * (RN * C::GP3);
#pragma unroll
    for (int n = 0; n < NI; n++) {
      const int it = tid + n * TH;
      const bool ok = goff[n] >= 0;
      pv[n] = ok ? src[goff[n]] : 0.0;
      if constexpr (NC == 3) pw[n] = ok ? src[goff[n] + (9 - (it / C::GP3) % NLC) * C::GP3] : 0.0;
    }
  };
  auto store_chunk = [&](T* __restrict__ cb) {
#pragma unroll
    for (int n = 0; n < NI; n++) {
      if (NIT % TH != 0 && dst[n] < 0) continue;
      if constexpr (NC == 3) {
        const bool wc = RHS && ((tid + n * TH) / C::GP3) % NLC == 9;
        cb[dst[n]] = wc ? (T)pw[n] : (T)pw[n] * (T)pv[n];
        cb[dst[n] + (wc ? NG * C::RS : 9 * NG * C::RS)] = wc ? T(1) : (T)pv[n];
      } else {
        cb[dst[n]] = (T)pv[n];
      }
    }
  };

  // ---- unit sums of one chunk
  T t2[W1][W1];
  auto units = [&](const T* __restrict__ cb, auto m3c) {
    constexpr int m3 = decltype(m3c)::value;
    const T* __restrict__ A = cb + oA;
    const T* __restrict__ B = cb + oB;
#pragma unroll
    for (int q3 = 0; q3 < NG; q3++) {
      T t1[W1];
#pragma unroll
      for (int d = 0; d < W1; d++) t1[d] = T(0);
#pragma unroll
      for (int g = 0; g < C::Q2; g++) {
        T v = A[q3 * C::NQ2 + g];
        if (NC == 3) v *= B[q3 * C::NQ2 + g];
#pragma unroll
        for (int b = 0; b < P1; b++) t1[g / NG + b] += v * c2r[g][b];
      }
#pragma unroll
      for (int b = 0; b < P1; b++) {
        const T f = sh.c3[v3][m3 * NG + q3][b];
#pragma unroll
        for (int d = 0; d < W1; d++) t2[m3 + b][d] += f * t1[d];
      }
    }
  };

  // ---- the thread's column line: (slot cs, dk, dj), with its open rows
  const int cs = tid / WW, cd = tid % WW;
  const bool col = tid < C::NCT && (NC == 3 || cs < nl);
  // (double also where the units sum in float: this step and the window cost
  // little, and the FP32 matrix is then closer to the FP64 one)
  double sw[P1][W1]; // [row - e1][di]
  double rw[P1];     // right-hand side moments of line tid (tid < NL)
#pragma unroll
  for (int r = 0; r < P1; r++) {
#pragma unroll
    for (int d = 0; d < W1; d++) sw[r][d] = 0.0;
    rw[r] = 0.0;
  }
  auto columns = [&](int e1) {
    ConstTable tn = (ConstTable)a.tabN1 + (int64_t)e1 * NG * P1;
    ConstTable td = (ConstTable)a.tabD1 + (int64_t)e1 * NG * P1;
    if (tid < C::NCT) {
      const T* __restrict__ E = sh.buf + cs * C::ES + cd;
#pragma unroll
      for (int q = 0; q < NG; q++) {
        const T* __restrict__ Eq = E + q * 9 * SL * C::ES;
        constexpr int KS = SL * C::ES;
        auto e = [&](int n) { return (double)Eq[n * KS]; };
        const double v00 = e(0), v01 = e(1) + e(2), v10 = e(3) + e(6);
        const double v11 = (e(4) + e(5)) + (e(7) + e(8));
        double u0[P1], u1[P1];
#pragma unroll
        for (int b = 0; b < P1; b++) {
          const double n = tn[q * P1 + b], d = td[q * P1 + b];
          u0[b] = v00 * d + v01 * n;
          u1[b] = v10 * d + v11 * n;
        }
#pragma unroll
        for (int r = 0; r < P1; r++) {
          const double n = tn[q * P1 + r], d = td[q * P1 + r];
#pragma unroll
          for (int b = 0; b < P1; b++) sw[r][b - r + P] += d * u0[b] + n * u1[b];
        }
      }
    }
    if (RHS && tid < NL) {
      const T* __restrict__ E = sh.buf + (C::NU + tid) * C::ES + P * W1 + P;
#pragma unroll
      for (int q = 0; q < NG; q++) {
        const double m = E[q * NL * C::ES];
#pragma unroll
        for (int r = 0; r < P1; r++) rw[r] += tn[q * P1 + r] * m;
      }
    }
  };

  // ---- row position i of the lines: CSR rows and starts (threads < NROW)
  const int rj = NC == 3 ? 0 : tid, rcomp = NC == 3 ? tid : 0;
  const bool rthread = tid < C::NROW && (NC == 3 || tid < nl);
  const int64_t rdof0 =
      ((int64_t)a.n1 * ((j0 + rj) + (int64_t)a.n2 * kc)) * NC + rcomp; // + i*NC
  const bool by_map = ACCUM && a.pmap != nullptr;

  auto value = [&](int r, int t) -> T {
    if constexpr (NC == 1) {
      return (T)sh.row[r * WN + t];
    } else {
      const int nbr = t / 3, j = t - 3 * nbr;
      const double* __restrict__ s = sh.row + nbr * 9;
      double v = a.lam * s[3 * r + j] + a.mu * s[3 * j + r];
      if (r == j) v += a.mu * (s[0] + s[4] + s[8]);
      return (T)v;
    }
  };
  auto put = [&](int64_t at, T v) {
    if constexpr (sizeof(T) == 4) {
      if (ACCUM) a.val32[at] += v;
      else a.val32[at] = v;
    } else {
      if (ACCUM) a.val64[at] += v;
      else a.val64[at] = v;
    }
  };
  auto put_rhs = [&](int req, double v) {
    if (ACCUM) a.rhs[req] += v;
    else a.rhs[req] = v;
  };
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  constexpr int NW = TH / 64;
  auto row_out = [&](int i) {
    // rows with a full window: entry t at position t, 64 columns per wave and
    // step (no loads here unless the rows are shared: a wait for one would
    // also wait for the stores before it)
    constexpr int NSEG = (C::NCOL + 63) / 64, NSTEP = (C::NROW * NSEG + NW - 1) / NW;
    if constexpr (ACCUM) {
      // positions, then old values, then sums: the loads of a phase overlap
      int64_t at[NSTEP];
      T old[NSTEP];
#pragma unroll
      for (int k = 0; k < NSTEP; k++) {
        const int sg = wave + k * NW, r = sg / NSEG, t = (sg - r * NSEG) * 64 + lane;
        const bool ok = sg < C::NROW * NSEG && t < C::NCOL && sh.full[r < C::NROW ? r : 0];
        at[k] = ok ? a.pmap[sh.base[r] + t] : -1;
      }
#pragma unroll
      for (int k = 0; k < NSTEP; k++)
        if constexpr (sizeof(T) == 4) old[k] = at[k] >= 0 ? a.val32[at[k]] : T(0);
        else old[k] = at[k] >= 0 ? a.val64[at[k]] : T(0);
#pragma unroll
      for (int k = 0; k < NSTEP; k++) {
        const int sg = wave + k * NW, r = sg / NSEG, t = (sg - r * NSEG) * 64 + lane;
        if (at[k] < 0) continue;
        const T v = old[k] + value(r, t);
        if constexpr (sizeof(T) == 4) a.val32[at[k]] = v;
        else a.val64[at[k]] = v;
      }
    } else {
#pragma unroll
      for (int k = 0; k < NSTEP; k++) {
        const int sg = wave + k * NW;
        if (sg >= C::NROW * NSEG) break;
        const int r = sg / NSEG, t = (sg - r * NSEG) * 64 + lane;
        const int64_t base = sh.base[r];
        if (!__builtin_amdgcn_readfirstlane(sh.full[r])) continue;
        if (C::NCOL % 64 == 0 || t < C::NCOL) put(base + t, value(r, t));
      }
    }
    if (RHS && tid < C::NROW && sh.full[tid] && a.rhs)
      put_rhs(sh.req[tid], NC == 3 ? sh.rrow[0] * a.body[tid] : sh.rrow[tid]);
    // the others: one wave per row, ballot compaction over the window
    const double* __restrict__ gv = a.gval;
    for (int r = wave; r < C::NROW; r += NW) {
      const int req = sh.req[r];
      if (req < 0 || sh.full[r]) continue;
      const int jc = NC == 3 ? j0 : j0 + r;
      const int64_t base = sh.base[r];
      double corr = 0.0;
      int64_t pos = 0;
#pragma unroll 1
      for (int t0 = 0; t0 < C::NCOL; t0 += 64) {
        const int t = t0 + lane;
        const int ev = window_eq<P, NC>(a, i, jc, kc, t);
        const bool valid = ev >= 0;
        const unsigned long long m = __ballot(valid);
        if (ACCUM && valid && !a.pmap) { // no position map: search the row
          int64_t lo = a.rowptr[req], hi = a.rowptr[req + 1] - 1;
          while (lo < hi) {
            const int64_t mid = (lo + hi) >> 1;
            if (a.colind[mid] < ev) lo = mid + 1;
            else hi = mid;
          }
          put(lo, value(r, t));
        } else if (valid) {
          const int64_t at = base + pos + __popcll(m & ((1ull << lane) - 1ull));
          put(by_map ? a.pmap[at] : at, value(r, t));
        } else if (gv && ev == -1) { // eliminated column inside the patch
          const int nbr = t / NC;
          const int ii = i + nbr % W1 - P, jj = jc + (nbr / W1) % W1 - P, kk = kc + nbr / WW - P;
          const int64_t gdof = ((int64_t)ii + (int64_t)a.n1 * (jj + (int64_t)a.n2 * kk)) * NC + t % NC;
          corr += (double)value(r, t) * gv[gdof];
        }
        pos += __popcll(m);
      }
      if (gv) {
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) corr += __shfl_xor(corr, off, 64);
      }
      if ((RHS || gv) && a.rhs && lane == 0) {
        const double m = !RHS ? 0.0
                         : NC == 3 ? sh.rrow[0] * a.body[r]
                                   : sh.rrow[r];
        put_rhs(req, m - corr);
      }
    }
  };

  // ---- layers ---------------------------------------------------------------
  const int mlo = line_max(0, P - kc), mhi = a.nel3 - 1 - kc + P < P ? a.nel3 - 1 - kc + P : P;
  const int ea = i0 - P > 0 ? i0 - P : 0;            // first layer of these rows
  const int eb = i1 < a.nel1 ? i1 : a.nel1;          // past their last layer
  int rq = rthread ? a.eq[rdof0 + (int64_t)ea * NC] : -1, rqn = -1;
  int buf = 0;
  load_chunk(ea, mlo);
  store_chunk(sh.buf);
#pragma unroll 1
  for (int i = ea; i < i1; i++) {
    // CSR start and length of row i, and the equation of row i+1 (used after
    // the layer's sums: the loads are long back by then)
    int64_t rb = 0, re = 0;
    if (rq >= 0) {
      const int64_t* __restrict__ ptr = by_map ? a.pptr + rdof0 + (int64_t)i * NC : a.rowptr + rq;
      rb = ptr[0];
      re = ptr[1];
    }
    rqn = rthread && i + 1 < i1 ? a.eq[rdof0 + (int64_t)(i + 1) * NC] : -1;
    if (i < eb) {
#pragma unroll
      for (int k = 0; k < W1; k++)
#pragma unroll
        for (int d = 0; d < W1; d++) t2[k][d] = T(0);
      // the current chunk is in buffer buf; the next chunk of the layer goes
      // to the other one, the next layer's first chunk stays in registers
      // until the exchange over the buffers is over
      auto row3 = [&](auto m3c) {
        constexpr int m3 = decltype(m3c)::value;
        if (m3 < mlo || m3 > mhi) return;
        line_barrier();
        const bool more = m3 < mhi;
        if (more) load_chunk(i, m3 + 1);
        else if (i + 1 < eb) load_chunk(i + 1, mlo);
        units(sh.buf + buf * S::CHUNK, m3c);
        buf ^= 1;
        if (more) store_chunk(sh.buf + buf * S::CHUNK);
      };
      row3(std::integral_constant<int, 0>{});
      row3(std::integral_constant<int, 1>{});
      if constexpr (P >= 2) row3(std::integral_constant<int, 2>{});
      // exchange (over the chunk buffers) and direction 1
      line_barrier();
      if (unit) {
#pragma unroll
        for (int k = 0; k < W1; k++)
#pragma unroll
          for (int d = 0; d < W1; d++) sh.buf[tid * C::ES + k * W1 + d] = t2[k][d];
      }
      line_barrier();
      columns(i);
    }
    const bool out = i >= i0;
    if (out) {
      if (col) {
#pragma unroll
        for (int d = 0; d < W1; d++) {
          if (NC == 3) sh.row[(cd * W1 + d) * 9 + cs] = sw[0][d];
          else sh.row[cs * WN + cd * W1 + d] = sw[0][d];
        }
      }
      if (RHS && tid < NL) sh.rrow[tid] = rw[0];
      if (tid < C::NROW) {
        sh.req[tid] = rq;
        sh.base[tid] = rb;
        sh.full[tid] = rq >= 0 && (!ACCUM || by_map) && re - rb == C::NCOL;
      }
    }
#pragma unroll
    for (int r = 0; r < P1; r++) {
#pragma unroll
      for (int d = 0; d < W1; d++) sw[r][d] = r < P ? sw[r + 1 < P1 ? r + 1 : r][d] : 0.0;
      rw[r] = r < P ? rw[r + 1 < P1 ? r + 1 : r] : 0.0;
    }
    rq = rqn;
    line_barrier(); // rows complete in LDS; the exchange has been read
    if (i + 1 < eb) store_chunk(sh.buf + buf * S::CHUNK);
    if (out) row_out(i);
    if (i + 1 >= eb) line_barrier(); // no chunk barrier before the next row
  }
}

// Rows of one group of lines: the lines [j0, j0 + nl) at k and the segment
// [i0, i1) of their rows, from the group's index (segment fastest, then line
// group, then k).
template <int P, int NG, int NC, typename T, bool RHS, bool ACCUM, bool WIDE>
__global__ __launch_bounds__((LineCfg<P, NG, NC>::TH), ACCUM ? 2 : 1) void k_lines(const AsmArgs* __restrict__ args,
                                                                    int ngj, int nseg, int total)
{
  __shared__ LineShared<P, NG, NC, T, RHS> sh;
  ConstArgs& a = *const_args(args);
  // consecutive groups share elements: each XCD takes a contiguous range, so
  // that its L2 serves the shared records
  const int per = (total + 7) / 8;
  const int g = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || g >= total) return;
  const int seg = g % nseg, jg = (g / nseg) % ngj, kc = g / (nseg * ngj);
  const int j0 = (int)((int64_t)a.n2 * jg / ngj), j1 = (int)((int64_t)a.n2 * (jg + 1) / ngj);
  const int i0 = (int)((int64_t)a.n1 * seg / nseg), i1 = (int)((int64_t)a.n1 * (seg + 1) / nseg);
  line_group<P, NG, NC, T, RHS, ACCUM, WIDE>(a, j0, j1 - j0, kc, i0, i1, sh);
}

// Batch of scalar patches: persistent workgroups take the next item of the
// degree's list (largest first) from its queue counter.  An item's rows are
// written by one workgroup and their sums do not depend on the split, so
// results do not depend on which workgroup takes which item.
template <int P, typename T, bool RHS, bool WIDE>
__global__ __launch_bounds__((LineCfg<P, P + 1, 1>::TH), 2) void k_lines_batch(
    const AsmArgs* __restrict__ args, const LineItem* __restrict__ items, int nitems,
    int* __restrict__ queue)
{
  __shared__ LineShared<P, P + 1, 1, T, RHS> sh;
  __shared__ int next;
  while (true) {
    if (threadIdx.x == 0) next = atomicAdd(queue, 1);
    __syncthreads();
    const int it = __builtin_amdgcn_readfirstlane(next);
    if (it >= nitems) break;
    const LineItem w = items[it];
    line_group<P, P + 1, 1, T, RHS, false, WIDE>(const_args(args)[w.patch], w.j0, w.nl, w.k, w.i0, w.i1, sh);
    __syncthreads();
  }
}

} // namespace ifem
