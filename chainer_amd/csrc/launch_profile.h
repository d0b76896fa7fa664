// Optional event bracketing of every matrix-product and convolution launch (hipcx_profile_start/stop): the events are recorded on the launch stream
// right before and after the kernel, so their elapsed time is the kernel's own duration and excludes the filter repack and any host work.
// Defined in conv.hip.
#pragma once

#include "common.h"

namespace hipcx {

struct ProfileScope {
    hipStream_t stream;
    hipEvent_t stop = nullptr;
    ProfileScope(hipStream_t s, double flops, double bytes);
    ~ProfileScope();
    ProfileScope(const ProfileScope&) = delete;
    ProfileScope& operator=(const ProfileScope&) = delete;
};

}  // namespace hipcx
