// The small matrix product for callers inside the library that need several of them at once.
// Defined in conv.hip.
#pragma once

#include "common.h"

namespace hipcx {

// outs[i] = a_i . b, i < n <= 4: float32 products with one shape whose left operands lie a_distance elements apart; one launch.  False if
// the shapes are not the small product's: use hipcx_dot.
bool DotSeveral(const hipcx_array* a0, int64_t a_distance, const hipcx_array* b, const hipcx_array* const* outs, int n, hipStream_t stream);

}  // namespace hipcx
