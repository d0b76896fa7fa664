// Pairs of pixels of eight channel planes turned round into 16-byte groups of eight channels per pixel, in registers.
#pragma once

#include "igemm.h"

namespace hipcx {

// Halves `sel` of {hi, lo}: the low or high half of lo first, then of hi.
template <bool LO_HIGH, bool HI_HIGH>
__device__ __forceinline__ unsigned PickHalves(unsigned lo, unsigned hi) {
    constexpr unsigned sel = (LO_HIGH ? 0x0302u : 0x0100u) | ((HI_HIGH ? 0x0706u : 0x0504u) << 16);
    return __builtin_amdgcn_perm(hi, lo, sel);
}

// The two pixels' 16-byte groups of 8 channels from 8 dwords, one channel's pair of pixels each.
__device__ __forceinline__ void TurnPairs(const unsigned (&v)[8], Bytes16& first, Bytes16& second) {
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        first[d] = PickHalves<false, false>(v[2 * d], v[2 * d + 1]);
        second[d] = PickHalves<true, true>(v[2 * d], v[2 * d + 1]);
    }
}

}  // namespace hipcx
