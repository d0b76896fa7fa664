// Forms of the small matrix product for callers inside the library that take its result apart or need several of them at once.
// Defined in conv.hip.
#pragma once

#include "common.h"

namespace hipcx {

// Ways the reduction of a float32 [m,k] . [k,n] is split by DotParts; 1: use hipcx_dot.
int DotPartSplits(int64_t m, int64_t n, int64_t k);

// parts[s][m][n], s < splits: the sums of a . b over `splits` parts of the reduction axis, whose sum, taken from s = 0 on, is the product.  The
// next kernel adds them up while it reads them, which takes out the pass that hipcx_dot needs for it.  float32.
void DotParts(const hipcx_array* a, const hipcx_array* b, float* parts, int splits, hipStream_t stream);

// outs[i] = a_i . b, i < n <= 4: float32 products with one shape whose left operands lie a_distance elements apart; one launch.  False if
// the shapes are not the small product's: use hipcx_dot.
bool DotSeveral(const hipcx_array* a0, int64_t a_distance, const hipcx_array* b, const hipcx_array* const* outs, int n, hipStream_t stream);

}  // namespace hipcx
