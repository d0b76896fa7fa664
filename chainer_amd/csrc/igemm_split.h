// The implicit GEMM of igemm.h for float32 operands on the bfloat16 matrix pipes; the kernel and why it is exact enough: igemm_split.hip.
#pragma once

#include "igemm.h"

namespace hipcx {

// Launches `grid` workgroups of 64 * WM * WN threads as IGemmFastKernel<float, WM, WN, chunk_bytes, pm> would be.  False if the problem is outside what
// the kernel addresses.
template <int WM, int WN>
bool IGemmSplit(const IGemmArgs<float>& p, int chunk_bytes, bool pm, dim3 grid, hipStream_t stream);

}  // namespace hipcx
