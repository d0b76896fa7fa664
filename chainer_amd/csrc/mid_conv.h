// float16 convolutions of a few hundred output tiles; the kernel: mid_conv.hip.
#pragma once

#include "nchw_conv.h"

namespace hipcx {

// Whether MidConv beats NchwConvKernel (SmallConvTakes says where SmallConv beats both).
bool MidConvTakes(const NchwConvArgs& a, int taps);

// 3x3 (stride 1, padding 1; C % 16 == 0) over dense NCHW, with the fused tail; a.wp: packed filters [C/8][9][K][8].  Spans below 2^31 bytes.
void MidConv(const NchwConvArgs& a, hipStream_t stream);

}  // namespace hipcx
