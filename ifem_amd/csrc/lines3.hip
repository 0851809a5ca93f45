// lines3.hip -- line kernels of degree 3.
#include "lines_direct.hpp"

namespace ifem {

int launch_lines3(Context& c, const AsmArgs& a, int ng, bool fp32, bool rhs, int variant)
{
  return ng == 4 ? launch_lines_direct<3, 4>(c, a, fp32, rhs, variant)
                 : launch_lines_direct<3, 5>(c, a, fp32, rhs, variant);
}

template <typename T, bool RHS, int HALF>
static int launch_batch_direct(Context& c, const AsmArgs* args, const LineItem* items, int n,
                               int* queue, int ncu)
{
  int per_cu = 0;
  IFEM_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(
      &per_cu, reinterpret_cast<const void*>(&k_assemble_batch<3, T, RHS, HALF>), kBlock, 0));
  k_assemble_batch<3, T, RHS, HALF><<<std::max(1, std::min(n, std::max(1, per_cu) * ncu)), kBlock, 0,
                                      c.stream>>>(args, items, n, queue);
  IFEM_HIP(hipGetLastError());
  return IFEM_GPU_OK;
}

int launch_lines_batch3(Context& c, const AsmArgs* args, const LineItem* items, int n, int* queue,
                        int ncu, bool fp32)
{
  const bool half = c.batch->tune[3].half != 0;
  if (fp32)
    return half ? launch_batch_direct<float, false, 1>(c, args, items, n, queue, ncu)
                : launch_batch_direct<float, false, 0>(c, args, items, n, queue, ncu);
  return half ? launch_batch_direct<double, true, 1>(c, args, items, n, queue, ncu)
              : launch_batch_direct<double, true, 0>(c, args, items, n, queue, ncu);
}

} // namespace ifem
