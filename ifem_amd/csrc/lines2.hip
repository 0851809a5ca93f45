// lines2.hip -- line kernels of degree 2.
#include "lines_direct.hpp"
#include "lines_inst.hpp"

namespace ifem {

int launch_lines2(Context& c, const AsmArgs& a, int ng, bool fp32, bool rhs, int variant)
{
  if (ng == 4) return launch_lines_direct<2, 4>(c, a, fp32, rhs, variant);
  // FP32 elasticity stays with the direct kernel: the sum-factorised FP32
  // matrix is closer to the FP64 one (4.5e-8 against 7.4e-8 relative), but
  // the mixed-precision solve, whose time it is made for, then needs 7 %
  // more inner iterations: 718 against 671 on 40^3 elasticity, 465 against 432
  // on 24^3, means of 12 systems.  Both errors are far below the inner
  // tolerance of 1e-4, and why the rounding tells is not known; 7 % of a
  // solve is more than the whole FP32 assembly takes (64^3 4.4 ms)
  if (fp32 && c.ncomp == 3) {
    launch_direct_v<2, 3, 3, float>(c, a, false, variant);
    IFEM_HIP(hipGetLastError());
    return IFEM_GPU_OK;
  }
  return c.ncomp == 1 ? launch_lines_nc<2, 3, 1>(c, a, fp32, rhs, variant)
         : rhs        ? launch_lines_t<2, 3, 3, double, true>(c, a, variant)
                      : launch_lines_t<2, 3, 3, double, false>(c, a, variant);
}

int launch_lines_batch2(Context& c, const AsmArgs* args, const LineItem* items, int n, int* queue,
                        int ncu, bool fp32)
{
  return fp32 ? launch_batch_t<2, float, false>(c, args, items, n, queue, ncu)
              : launch_batch_t<2, double, true>(c, args, items, n, queue, ncu);
}

} // namespace ifem
