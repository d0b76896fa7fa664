// The small matrix product (small_dot.h) as the rest of the library calls it.  Defined in small_dot.hip.
#pragma once

#include "common.h"

namespace hipcx {

// Whether an [m,k] . [k,n] product is small: fewer than 128 tiles of 128 x 128, 256 for fewer than 64 terms.
bool SmallDotShape(int64_t m, int64_t n, int64_t k);

// Bytes of partial sums that TrySmallDot would use.
size_t SmallDotWorkspace(const hipcx_array* a, const hipcx_array* b, int dtype);

// out = a . b (+ bias, one element per column) of one float dtype.  False if the shapes or strides are not the small product's.  `partial` holds
// SmallDotWorkspace bytes; without it the reduction is not split.
bool TrySmallDot(const hipcx_array* a, const hipcx_array* b, const hipcx_array* bias, const hipcx_array* out, float* partial, hipStream_t stream);

// outs[i] = a_i . b, i < n <= 4: float32 products with one shape whose left operands lie a_distance elements apart; one launch.  False if
// the shapes are not the small product's: use hipcx_dot.
bool DotSeveral(const hipcx_array* a0, int64_t a_distance, const hipcx_array* b, const hipcx_array* const* outs, int n, hipStream_t stream);

}  // namespace hipcx
