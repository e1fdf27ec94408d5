// Interface between the GEMM dispatch and the products of planes (gemm_planes.hip).
#pragma once
#include "gemm_staged.h"

namespace axhip {
// A single fp32 product (k_range, stride_z, batch strides and col_scale are not looked at) whose operands are cut into bf16 terms once,
// into planes in the shared workspace; any alignment, any K.  -1: not taken.
int planes_f32(const StagedArgs &g, int transa, int transb);
}  // namespace axhip
