// lines_launch.hpp -- host side of the line kernels (lines.hpp), one file per
// degree: lines1.hip, lines2.hip, lines3.hip.
#pragma once

#include "asmargs.hpp"
#include "lines.hpp"

namespace ifem {

// Rows of the bound patch: variant 0 splits the lines into row segments by
// the rule in row_segments, 1 into twice as many, 2 not at all.
int launch_lines1(Context& c, const AsmArgs& args, int ng, bool fp32, bool rhs, int variant);
int launch_lines2(Context& c, const AsmArgs& args, int ng, bool fp32, bool rhs, int variant);
int launch_lines3(Context& c, const AsmArgs& args, int ng, bool fp32, bool rhs, int variant);

// n items of one degree of the batch, from the queue counter (zeroed).
int launch_lines_batch1(Context& c, const AsmArgs* args, const LineItem* items, int n, int* queue, int ncu, bool fp32);
int launch_lines_batch2(Context& c, const AsmArgs* args, const LineItem* items, int n, int* queue, int ncu, bool fp32);
int launch_lines_batch3(Context& c, const AsmArgs* args, const LineItem* items, int n, int* queue, int ncu, bool fp32);

// Most lines per item of the batch at degree p.
constexpr int batch_lines_per_item(int p)
{
  return p == 1 ? LineCfg<1, 2, 1>::NL : p == 2 ? LineCfg<2, 3, 1>::NL : 1;
}

} // namespace ifem
