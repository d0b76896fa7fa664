// float32 and float16 convolutions of few terms per output (the first layer of a network); the kernel: thin_conv.hip.
#pragma once

#include "common.h"

namespace hipcx {

// Whether the convolution is one of those: dense NCHW arrays, channels x filter of at most 32 terms.
bool ThinConvTakes(const hipcx_array* x, const hipcx_array* w, const int64_t* stride, const int64_t* pad, const hipcx_array* out);

void ThinConv(const hipcx_array* x, const hipcx_array* w, const hipcx_array* b, const int64_t* stride, const int64_t* pad, const hipcx_array* out, hipStream_t stream);

}  // namespace hipcx
