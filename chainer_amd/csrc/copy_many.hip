// Several copies in one launch: the parts of a concatenation, a stack, a network's weights packed side by side.
#include "common.h"

extern "C" int hipcx_copy(const hipcx_array* a, const hipcx_array* out, void* stream);

namespace hipcx {
namespace {

struct CopySegment {
    const char* src;
    char* dst;
    int64_t bytes;
    int block0;  // first workgroup
};

constexpr int kMaxSegments = 96;  // 32 bytes each: the descriptors travel as kernel arguments (4 KB at most), no table in memory

struct CopyManyArgs {
    CopySegment seg[kMaxSegments];
    int n;
};

struct __attribute__((packed, aligned(1))) Packed16 {
    uint4 v;
};

// A memory copy; what it saves is launches: 2.6 us per array in the stream and the host's share of each.  A workgroup moves 4096 * V
// bytes of one segment, 16 bytes per access at any address (the last access of a segment moves back over its predecessor instead of
// going element by element).  [35][20,650] float32 into one array: 35 launches of 2.6 us -> one of 3.4.
template <int V>
__global__ __launch_bounds__(256) void CopyManyKernel(CopyManyArgs p) {
    int lo = 0, hi = p.n;  // seg[lo].block0 <= blockIdx.x < seg[hi].block0
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (static_cast<int>(blockIdx.x) >= p.seg[mid].block0) lo = mid;
        else hi = mid;
    }
    const CopySegment s = p.seg[lo];
    const int64_t first = (static_cast<int64_t>(blockIdx.x) - s.block0) * (4096 * V) + threadIdx.x * 16;
    if (s.bytes < 16) {
        if (static_cast<int64_t>(threadIdx.x) < s.bytes) s.dst[threadIdx.x] = s.src[threadIdx.x];
        return;
    }
    Packed16 v[V];
#pragma unroll
    for (int i = 0; i < V; ++i) v[i] = *reinterpret_cast<const Packed16*>(s.src + min(first + i * 4096, s.bytes - 16));
#pragma unroll
    for (int i = 0; i < V; ++i) {
        if (first + i * 4096 < s.bytes) *reinterpret_cast<Packed16*>(s.dst + min(first + i * 4096, s.bytes - 16)) = v[i];
    }
}

template <int V>
void Launch(CopyManyArgs& p, hipStream_t stream) {
    int64_t blocks = 0;
    for (int i = 0; i < p.n; ++i) {
        p.seg[i].block0 = static_cast<int>(blocks);
        blocks += (p.seg[i].bytes + 4096 * V - 1) / (4096 * V);
    }
    hipLaunchKernelGGL(CopyManyKernel<V>, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, p);
    CheckLaunch("copy_many");
}

}  // namespace
}  // namespace hipcx

using namespace hipcx;

extern "C" int hipcx_copy_many(const hipcx_array* const* as, const hipcx_array* const* outs, int n, void* stream) {
    return Guard([&] {
        HIPCX_REQUIRE(n >= 0 && (n == 0 || (as != nullptr && outs != nullptr)), HIPCX_CHAINERX_ERROR, "copy_many: null arrays");
        CopyManyArgs p;
        p.n = 0;
        int64_t bytes = 0;
        auto flush = [&] {
            if (p.n == 0) return;
            // four accesses per thread once that still leaves every compute unit its workgroups
            if (bytes >= int64_t{4096} * 4 * 4 * NumCUs()) Launch<4>(p, AsStream(stream));
            else Launch<1>(p, AsStream(stream));
            p.n = 0;
            bytes = 0;
        };
        for (int i = 0; i < n; ++i) {
            ValidateArray(as[i], "a");
            ValidateArray(outs[i], "out");
            bool plain = as[i]->dtype == outs[i]->dtype && as[i]->ndim == outs[i]->ndim && IsContiguous(as[i]) && IsContiguous(outs[i]);
            for (int d = 0; plain && d < as[i]->ndim; ++d) plain = as[i]->shape[d] == outs[i]->shape[d];
            const int64_t size = plain ? TotalSize(as[i]) * ItemSize(as[i]->dtype) : 0;
            if (!plain || size >= (int64_t{1} << 36)) {  // other layouts, casts, and what has too many workgroups for one launch
                const int status = hipcx_copy(as[i], outs[i], stream);
                if (status != HIPCX_OK) throw Error(status, hipcx_last_error());
                continue;
            }
            if (size == 0) continue;
            if (p.n == kMaxSegments || bytes + size >= (int64_t{1} << 37)) flush();  // (a grid holds less than 2^32 threads)
            p.seg[p.n].src = static_cast<const char*>(as[i]->data);
            p.seg[p.n].dst = static_cast<char*>(outs[i]->data);
            p.seg[p.n++].bytes = size;
            bytes += size;
        }
        flush();
    });
}
