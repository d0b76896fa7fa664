// float32 3x3 convolutions of dense NCHW arrays; the kernel: direct_conv.hip.
#pragma once

#include "common.h"

namespace hipcx {

// Whether the convolution is one of those, with dense filters: stride 1, padding 1, whole groups of eight channels.
bool DirectConvTakes(const hipcx_array* x, const hipcx_array* w, const int64_t* stride, const int64_t* pad, const hipcx_array* out);

void DirectConv(const hipcx_array* x, const hipcx_array* w, const hipcx_array* b, const hipcx_array* out, hipStream_t stream);

}  // namespace hipcx
