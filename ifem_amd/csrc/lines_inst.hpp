// lines_inst.hpp -- launches of the sum-factorised line kernels (included by
// the files of the degrees that use them, which compile side by side).
#pragma once

#include <algorithm>

#include "lines_launch.hpp"

namespace ifem {

// Workgroups of kernel f that one compute unit holds.
template <typename F>
static int resident_blocks(F f, int threads)
{
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, reinterpret_cast<const void*>(f), threads, 0) != hipSuccess)
    n = 1;
  return std::max(1, n);
}

// Row segments per line: the time of a split is taken as the layers of a
// workgroup (its rows, the P layers before them that it repeats, and about
// two layers' worth of set-up) times the rounds of workgroups, where a
// compute unit that holds fewer than `res` workgroups is bound by latency.
// Segments of fewer than 2 P rows repeat more than they own and are taken
// only while the workgroups are no more than the compute units: the line
// kernel of 5x5x5 scalar quadratic elements, 7 rows a line, takes 23.6 us with
// seven segments and 46 with one (FP32: 21 and 42).
static int row_segments(int n1, int p, int64_t groups, int res, int ncu)
{
  int best = 1;
  double t_best = 1e300;
  const int most = (int)std::max<int64_t>(1, std::max<int64_t>(n1 / (2 * p), std::min<int64_t>(n1, ncu / groups)));
  for (int s = 1; s <= most; s++) {
    const int64_t g = groups * s;
    const int64_t per_cu = (g + ncu - 1) / ncu;
    const int64_t rounds = (per_cu + res - 1) / res;
    const double t = (double)((n1 + s - 1) / s + p + 2) * std::max<double>((double)per_cu, 1.6 * rounds);
    if (t < 0.97 * t_best) {
      t_best = t;
      best = s;
    }
  }
  return best;
}

template <int P, int NG, int NC, typename T, bool RHS, bool ACCUM, bool WIDE>
static int launch_lines_w(Context& c, const AsmArgs& a, int variant)
{
  using C = LineCfg<P, NG, NC>;
  static const int res = resident_blocks(k_lines<P, NG, NC, T, RHS, ACCUM, WIDE>, C::TH);
  const int ngj = (a.n2 + C::NL - 1) / C::NL;
  int nseg = variant == 2 ? 1 : row_segments(a.n1, P, (int64_t)ngj * a.n3, res, 256);
  if (variant == 1) nseg = std::min(2 * nseg, a.n1);
  const int total = ngj * a.n3 * nseg;
  k_lines<P, NG, NC, T, RHS, ACCUM, WIDE><<<(total + 7) / 8 * 8, C::TH, 0, c.stream>>>(
      static_cast<const AsmArgs*>(c.d_asmargs), ngj, nseg, total);
  IFEM_HIP(hipGetLastError());
  return IFEM_GPU_OK;
}

template <int P, int NG, int NC, typename T, bool RHS, bool ACCUM>
static int launch_lines_a(Context& c, const AsmArgs& a, int variant)
{
  return LineCfg<P, NG, NC>::wide(a.nel1) ? launch_lines_w<P, NG, NC, T, RHS, ACCUM, true>(c, a, variant)
                                          : launch_lines_w<P, NG, NC, T, RHS, ACCUM, false>(c, a, variant);
}

template <int P, int NG, int NC, typename T, bool RHS>
static int launch_lines_t(Context& c, const AsmArgs& a, int variant)
{
  return a.accum ? launch_lines_a<P, NG, NC, T, RHS, true>(c, a, variant)
                 : launch_lines_a<P, NG, NC, T, RHS, false>(c, a, variant);
}

template <int P, int NG, int NC>
static int launch_lines_nc(Context& c, const AsmArgs& a, bool fp32, bool rhs, int variant)
{
  return fp32  ? launch_lines_t<P, NG, NC, float, false>(c, a, variant)
         : rhs ? launch_lines_t<P, NG, NC, double, true>(c, a, variant)
               : launch_lines_t<P, NG, NC, double, false>(c, a, variant);
}

template <int P, int NG>
static int launch_lines_ng(Context& c, const AsmArgs& a, bool fp32, bool rhs, int variant)
{
  return c.ncomp == 1 ? launch_lines_nc<P, NG, 1>(c, a, fp32, rhs, variant)
                      : launch_lines_nc<P, NG, 3>(c, a, fp32, rhs, variant);
}

template <int P, typename T, bool RHS, bool WIDE>
static int launch_batch_w(Context& c, const AsmArgs* args, const LineItem* items, int n, int* queue,
                          int ncu)
{
  using C = LineCfg<P, P + 1, 1>;
  static const int res = resident_blocks(k_lines_batch<P, T, RHS, WIDE>, C::TH);
  k_lines_batch<P, T, RHS, WIDE><<<std::max(1, std::min(n, res * ncu)), C::TH, 0, c.stream>>>(
      args, items, n, queue);
  IFEM_HIP(hipGetLastError());
  return IFEM_GPU_OK;
}

template <int P, typename T, bool RHS>
static int launch_batch_t(Context& c, const AsmArgs* args, const LineItem* items, int n, int* queue,
                          int ncu)
{
  bool wide = false;
  for (const BatchPatch& bp : c.batch->pp)
    wide |= bp.p == P && LineCfg<P, P + 1, 1>::wide(c.patches[bp.patch].nel[0]);
  return wide ? launch_batch_w<P, T, RHS, true>(c, args, items, n, queue, ncu)
              : launch_batch_w<P, T, RHS, false>(c, args, items, n, queue, ncu);
}

} // namespace ifem
