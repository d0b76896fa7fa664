// float16 convolutions of few output pixels; the kernel: small_conv.hip.
#pragma once

#include "nchw_conv.h"

namespace hipcx {

// Whether SmallConv beats NchwConvKernel.
bool SmallConvTakes(const NchwConvArgs& a, int taps);

// 1x1 (any stride; C % 32 == 0) and 3x3 (stride 1, padding 1; C % 16 == 0) over dense NCHW, with the fused tail; a.wp: the dense filters [K][C][taps],
// 16-byte aligned.  Spans below 2^31 bytes.
void SmallConv(const NchwConvArgs& a, int taps, hipStream_t stream);

}  // namespace hipcx
