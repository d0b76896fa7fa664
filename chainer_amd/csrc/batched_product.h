// float16 products summed over a batch, as the weight gradients of convolutions are; the kernel: batched_product.hip.
#pragma once

#include "common.h"

namespace hipcx {

// out[m][n] = sum over b < batch, k < depth of a[b][m][k] * bt[b][n][k].  Rows are dense along k; the operands and every stride (in elements) are
// multiples of 4 bytes, and depth is even.
struct BatchedOperands {
    const half_t* a;
    const half_t* b;
    half_t* out;  // dense [M][N]
    int M, N, depth, batch;
    int64_t a_row, a_slice, b_row, b_slice;
    // taps_s > 0: row j of bt_b is a window of a larger array: j = (c, r, s), c = j / (taps_r * taps_s), starts at b + c * b_row + r * r_stride + s % 2 * s_stride +
    // s / 2 * s_pair_stride
    int taps_r, taps_s;
    int64_t r_stride, s_stride, s_pair_stride;
};

// Workgroups per tile along the reduction; slices > 1 need slices * m * n floats of partial sums.
int HalfProductSlices(const BatchedOperands& o);

// Whether the operands' alignment, spans and extents are within what the kernel addresses.  Null operands: every address is taken to be aligned.
bool HalfProductApplies(const BatchedOperands& o);

void HalfProduct(const BatchedOperands& o, float* partial, int slices, hipStream_t stream);

}  // namespace hipcx
