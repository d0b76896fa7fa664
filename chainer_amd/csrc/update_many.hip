// x - g * s of several arrays in one launch: the parameter updates of gradient descent.
#include "common.h"

extern "C" int hipcx_multiply_as(const hipcx_array* x1, hipcx_scalar x2, const hipcx_array* out, void* stream);
extern "C" int hipcx_subtract(const hipcx_array* x1, const hipcx_array* x2, const hipcx_array* out, void* stream);

namespace hipcx {
namespace {

constexpr int kMaxUpdates = 112;  // 36 bytes each: the descriptors travel as kernel arguments (4 KB at most), no table in memory

struct UpdateManyArgs {
    const void* x[kMaxUpdates];
    const void* g[kMaxUpdates];
    void* out[kMaxUpdates];
    int64_t size[kMaxUpdates];   // elements
    int block0[kMaxUpdates];     // first workgroup
    int n;
    float minus_scale;  // as the arrays' type holds it
};

template <typename T>
struct __attribute__((packed, aligned(alignof(T)))) Piece {
    T v[16 / sizeof(T)];
};

// Rounded to T after the product and after the difference, like Multiply and Subtract; the difference as a sum with the opposite, which is the same.
template <typename T>
__device__ __forceinline__ T Updated(T x, T g, float minus_s) {
    const T step = static_cast<T>(static_cast<float>(g) * minus_s);
    return static_cast<T>(static_cast<float>(x) + static_cast<float>(step));
}

// A pass over memory; what it saves is launches, two per array, and a pass over the product.  A workgroup takes 256 * V pieces of 16 bytes of one array,
// the last elements one by one.  ResNet-50's 161 arrays: 322 launches, 0.8 ms -> two of 30 us together (19 M float16 elements in 56 arrays 248 -> 23).
template <typename T, int V>
__global__ __launch_bounds__(256) void UpdateManyKernel(UpdateManyArgs p) {
    constexpr int E = 16 / sizeof(T);
    int lo = 0, hi = p.n;  // block0[lo] <= blockIdx.x < block0[hi]
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (static_cast<int>(blockIdx.x) >= p.block0[mid]) lo = mid;
        else hi = mid;
    }
    const T* const x = static_cast<const T*>(p.x[lo]);
    const T* const g = static_cast<const T*>(p.g[lo]);
    T* const out = static_cast<T*>(p.out[lo]);
    const int64_t size = p.size[lo], first = (static_cast<int64_t>(blockIdx.x) - p.block0[lo]) * (256 * E * V) + threadIdx.x * E;
    Piece<T> xv[V], gv[V];
#pragma unroll
    for (int i = 0; i < V; ++i) {
        const int64_t at = first + i * 256 * E;
        if (at + E <= size) {
            xv[i] = *reinterpret_cast<const Piece<T>*>(x + at);
            gv[i] = *reinterpret_cast<const Piece<T>*>(g + at);
        }
    }
#pragma unroll
    for (int i = 0; i < V; ++i) {
        const int64_t at = first + i * 256 * E;
        if (at + E <= size) {
#pragma unroll
            for (int e = 0; e < E; ++e) xv[i].v[e] = Updated<T>(xv[i].v[e], gv[i].v[e], p.minus_scale);
            *reinterpret_cast<Piece<T>*>(out + at) = xv[i];
        } else {
            for (int64_t j = at; j < size; ++j) out[j] = Updated<T>(x[j], g[j], p.minus_scale);
        }
    }
}

template <typename T>
struct Updates {
    UpdateManyArgs p{};
    int64_t bytes = 0;
    hipStream_t stream;

    template <int V>
    void Launch() {
        constexpr int64_t each = 256 * V * static_cast<int64_t>(16 / sizeof(T));
        int64_t blocks = 0;
        for (int i = 0; i < p.n; ++i) {
            p.block0[i] = static_cast<int>(blocks);
            blocks += (p.size[i] + each - 1) / each;
        }
        hipLaunchKernelGGL((UpdateManyKernel<T, V>), dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, p);
        CheckLaunch("update_many");
    }
    void Flush() {
        if (p.n == 0) return;
        // four pieces per thread once that still leaves every compute unit its workgroups
        if (bytes >= int64_t{4096} * 4 * 4 * NumCUs()) Launch<4>();
        else Launch<1>();
        p.n = 0;
        bytes = 0;
    }
    void Add(const hipcx_array* x, const hipcx_array* g, const hipcx_array* out, int64_t size) {
        const int64_t more = size * static_cast<int64_t>(sizeof(T));
        if (p.n == kMaxUpdates || bytes + more >= (int64_t{1} << 36)) Flush();  // (a grid holds less than 2^32 threads)
        p.x[p.n] = x->data, p.g[p.n] = g->data, p.out[p.n] = out->data, p.size[p.n++] = size;
        bytes += more;
    }
};

}  // namespace
}  // namespace hipcx

using namespace hipcx;

extern "C" int hipcx_update_many(const hipcx_array* const* xs, const hipcx_array* const* gs, hipcx_scalar scale, const hipcx_array* const* outs, int n, void* stream) {
    return Guard([&] {
        HIPCX_REQUIRE(n >= 0 && (n == 0 || (xs != nullptr && gs != nullptr && outs != nullptr)), HIPCX_CHAINERX_ERROR, "update_many: null arrays");
        Updates<half_t> halves;
        Updates<float> floats;
        halves.stream = floats.stream = AsStream(stream);
        halves.p.minus_scale = -static_cast<float>(ScalarTo<half_t>(scale));
        floats.p.minus_scale = -ScalarTo<float>(scale);
        for (int i = 0; i < n; ++i) {
            const hipcx_array *x = xs[i], *g = gs[i], *out = outs[i];
            ValidateArray(x, "x");
            ValidateArray(g, "g");
            ValidateArray(out, "out");
            HIPCX_REQUIRE(x->dtype == out->dtype && g->dtype == out->dtype, HIPCX_DTYPE_ERROR, "update_many: x, g and out must share a dtype");
            HIPCX_REQUIRE(IsFloatDtype(out->dtype), HIPCX_DTYPE_ERROR, "update_many: floating point arrays only");
            bool same = x->ndim == out->ndim && g->ndim == out->ndim;
            for (int d = 0; same && d < out->ndim; ++d) same = x->shape[d] == out->shape[d] && g->shape[d] == out->shape[d];
            HIPCX_REQUIRE(same, HIPCX_DIMENSION_ERROR, "update_many: x, g and out must have one shape");
        }
        for (int i = 0; i < n; ++i) {
            const hipcx_array *x = xs[i], *g = gs[i], *out = outs[i];
            const int64_t size = TotalSize(out);
            if (size == 0) continue;
            const bool plain = IsContiguous(x) && IsContiguous(g) && IsContiguous(out) && size < (int64_t{1} << 34);
            if (plain && out->dtype == HIPCX_FLOAT16) {
                halves.Add(x, g, out, size);
            } else if (plain && out->dtype == HIPCX_FLOAT32) {
                floats.Add(x, g, out, size);
            } else {  // float64, other layouts and what has too many workgroups for one launch
                int status = hipcx_multiply_as(g, scale, out, stream);
                if (status == HIPCX_OK) status = hipcx_subtract(x, out, out, stream);
                if (status != HIPCX_OK) throw Error(status, hipcx_last_error());
            }
        }
        halves.Flush();
        floats.Flush();
    });
}
