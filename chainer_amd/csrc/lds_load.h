// Loads from global memory straight into LDS, and the wait that goes with them.
#pragma once

#include "common.h"

namespace hipcx {

typedef int int4_t __attribute__((ext_vector_type(4)));

// Raw buffer descriptor (base, no stride, size in bytes, 32-bit untyped data) as four scalars.
__device__ __forceinline__ int4_t RawRsrc(const void* ptr, unsigned bytes) {
    const uint64_t a = reinterpret_cast<uint64_t>(ptr);
    return int4_t{__builtin_amdgcn_readfirstlane(static_cast<int>(a & 0xffffffffu)), __builtin_amdgcn_readfirstlane(static_cast<int>((a >> 32) & 0xffffu)),
                  __builtin_amdgcn_readfirstlane(static_cast<int>(bytes)), 0x00020000};
}
// 16 bytes per lane from global memory straight into LDS at lds_addr + lane * 16 (lds_addr wave-uniform).  Written as
// assembly on purpose: the compiler orders every later LDS read behind an LDS-writing load it knows of with a wait for all
// outstanding loads, which would serialise the ring; the kernel waits for exactly the loads it needs.
__device__ __forceinline__ void LdsLoad16(int4_t rsrc, unsigned lds_addr, int voff, int soff) {
    asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(voff), "s"(rsrc),
                 "s"(__builtin_amdgcn_readfirstlane(soff))
                 : "memory", "m0");
}
// vmcnt <= N, nothing else waited for (gfx9 encoding: vmcnt in bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8)
template <int N>
__device__ __forceinline__ void WaitVmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
    __builtin_amdgcn_s_waitcnt((N & 0xf) | ((N >> 4) << 14) | (0x7 << 4) | (0xf << 8));
}

}  // namespace hipcx
