// lines1.hip -- line kernels of degree 1.
#include "lines_inst.hpp"

namespace ifem {

int launch_lines1(Context& c, const AsmArgs& a, int ng, bool fp32, bool rhs, int variant)
{
  return ng == 2 ? launch_lines_ng<1, 2>(c, a, fp32, rhs, variant)
                 : launch_lines_ng<1, 3>(c, a, fp32, rhs, variant);
}

int launch_lines_batch1(Context& c, const AsmArgs* args, const LineItem* items, int n, int* queue,
                        int ncu, bool fp32)
{
  return fp32 ? launch_batch_t<1, float, false>(c, args, items, n, queue, ncu)
              : launch_batch_t<1, double, true>(c, args, items, n, queue, ncu);
}

} // namespace ifem
