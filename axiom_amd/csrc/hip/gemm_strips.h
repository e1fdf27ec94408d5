// Interface between the GEMM dispatch and the one-launch kernel for few tiles (gemm_strips.hip).
#pragma once
#include "gemm_staged.h"

namespace axhip {
// A single fp32 product (k_range, stride_z, batch strides and col_scale are not looked at) in one launch, where that is the fastest
// way; any alignment, any K.  on_grid: the direct-to-LDS tiles would take it.  -1: not taken.
int strips_f32(const StagedArgs &g, int transa, int transb, bool on_grid);
}  // namespace axhip
