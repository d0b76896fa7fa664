// ConvGradWeightKernel (CX/kernels/connection.h:34-49) for dense NCHW float16 / float32 / float64 arrays.
//
// The native backend computes gw = TensorDot(gy, Im2Col(x)) over the batch and the output positions
// (CX/native/native_device/conv.cc:91-124).  Same product here, with both operands written once in the layout the MFMA matrix
// kernel reads -- the reduction index (n, oh, ow) as the unit-stride axis:
//     gy_t[k][n][oh][ow]            (one transposing copy of gy)
//     col_t[c][r][s][n][oh][ow]     (Im2Col in one launch instead of kh*kw strided copies of a padded image)
// and then gw[k][(c, r, s)] = Dot(gy_t, col_t^T), which for these shapes (few output tiles, long reduction) runs with the
// reduction split over workgroups.
//
// Filters larger than 1x1 at stride 1 (float16 / float32) avoid the kh*kw-fold Im2Col: x is written as zero-padded planes of rows of Wp elements, several
// copies of them shifted left by one element each, and gy once with its rows padded to Wp with zeros.  On that common grid tap (r, s) of channel c is a
// window of one of the copies, so
//     gw[k][c][r][s] = sum_n sum_q gy_p[n][k][q] * x_p[n][c][q + r*Wp + s],   q over OH*Wp
// is one accumulated matrix product per image whose right-hand rows alias windows of the copies; the zero columns of gy_p cancel
// the products that wrap around a row end.  In float16 the product reads at any even element: two copies serve every s, and rows are as long as x's with
// the padding of one side (the next row's stands in for the other), rounded up to even.  Otherwise there are kw copies and rows are whole 16-byte
// granules with both paddings.  A non-finite x value would meet a zero of gy_p in windows the reference never
// multiplies it into (0 * inf = NaN in filter taps that stay finite there), so the copy kernel flags every plane of x that holds
// an inf or NaN and, after the product, GradWeightChannelFixupKernel computes the filter taps of those planes' channels again the
// reference's way (the sum over the Im2Col windows, padding multiplied as zeros).  With finite data that kernel's workgroups read
// a channel's flags each and exit.
#include "batched_product.h"
#include "common.h"

namespace hipcx {
namespace {

struct GradWeightArgs {
    const void* x;
    const void* gy;
    void* col_t;
    void* gy_t;
    int N, C, H, W, K, kh, kw, OH, OW, sh, sw, ph, pw;
};

template <typename T, int VEC>
struct alignas(sizeof(T) * VEC) GVec {
    T v[VEC];
};

// One thread: VEC consecutive ow of one (c, r, s, n, oh).
template <typename T, int VEC>
__global__ __launch_bounds__(256) void Im2ColTKernel(GradWeightArgs p, int64_t total) {
    const T* x = static_cast<const T*>(p.x);
    T* col = static_cast<T*>(p.col_t);
    const int owv = p.OW / VEC;
    auto emit = [&](int64_t idx, int wv, int oh, int n, int s, int r, int c) {
        const int ih = oh * p.sh - p.ph + r;
        GVec<T, VEC> out;
        const T* row = x + ((static_cast<int64_t>(n) * p.C + c) * p.H + ih) * p.W;
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            const int iw = (wv * VEC + e) * p.sw - p.pw + s;
            out.v[e] = (ih >= 0 && ih < p.H && iw >= 0 && iw < p.W) ? row[iw] : T(0);
        }
        *reinterpret_cast<GVec<T, VEC>*>(col + idx * VEC) = out;  // idx enumerates the vectors of col_t in memory order
    };
    if (total < (int64_t{1} << 31)) {  // the usual case: five 32-bit divisions per vector instead of five 64-bit ones
        const uint32_t n_total = static_cast<uint32_t>(total), step = gridDim.x * 256u;
        for (uint32_t idx = blockIdx.x * 256u + threadIdx.x; idx < n_total; idx += step) {
            uint32_t t = idx;
            const uint32_t wv = t % static_cast<uint32_t>(owv);
            t /= static_cast<uint32_t>(owv);
            const uint32_t oh = t % static_cast<uint32_t>(p.OH);
            t /= static_cast<uint32_t>(p.OH);
            const uint32_t n = t % static_cast<uint32_t>(p.N);
            t /= static_cast<uint32_t>(p.N);
            const uint32_t s2 = t % static_cast<uint32_t>(p.kw);
            t /= static_cast<uint32_t>(p.kw);
            const uint32_t r = t % static_cast<uint32_t>(p.kh);
            emit(idx, static_cast<int>(wv), static_cast<int>(oh), static_cast<int>(n), static_cast<int>(s2), static_cast<int>(r),
                 static_cast<int>(t / static_cast<uint32_t>(p.kh)));
            if (idx + step < idx) break;  // the next index would wrap
        }
        return;
    }
    for (int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; idx < total; idx += static_cast<int64_t>(gridDim.x) * 256) {
        int64_t t = idx;
        const int wv = static_cast<int>(t % owv);
        t /= owv;
        const int oh = static_cast<int>(t % p.OH);
        t /= p.OH;
        const int n = static_cast<int>(t % p.N);
        t /= p.N;
        const int s2 = static_cast<int>(t % p.kw);
        t /= p.kw;
        const int r = static_cast<int>(t % p.kh);
        emit(idx, wv, oh, n, s2, r, static_cast<int>(t / p.kh));
    }
}

// gy_t[k][n][p] = gy[n][k][p], VEC consecutive p per thread.
template <typename T, int VEC>
__global__ __launch_bounds__(256) void TransposeNKKernel(GradWeightArgs p, int64_t total) {
    const T* gy = static_cast<const T*>(p.gy);
    T* gt = static_cast<T*>(p.gy_t);
    const int64_t pv = static_cast<int64_t>(p.OH) * p.OW / VEC;
    if (total < (int64_t{1} << 31)) {  // 32-bit index arithmetic
        const uint32_t n_total = static_cast<uint32_t>(total), step = gridDim.x * 256u, pv32 = static_cast<uint32_t>(pv);
        for (uint32_t idx = blockIdx.x * 256u + threadIdx.x; idx < n_total; idx += step) {
            uint32_t t = idx / pv32;
            const uint32_t v = idx - t * pv32;
            const uint32_t k = t / static_cast<uint32_t>(p.N);
            const uint32_t n = t - k * static_cast<uint32_t>(p.N);
            *reinterpret_cast<GVec<T, VEC>*>(gt + static_cast<int64_t>(idx) * VEC) =
                    *reinterpret_cast<const GVec<T, VEC>*>(gy + ((static_cast<int64_t>(n) * p.K + k) * pv + v) * VEC);
            if (idx + step < idx) break;  // the next index would wrap
        }
        return;
    }
    for (int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; idx < total; idx += static_cast<int64_t>(gridDim.x) * 256) {
        int64_t t = idx;
        const int64_t v = t % pv;
        t /= pv;
        const int n = static_cast<int>(t % p.N);
        const int k = static_cast<int>(t / p.N);
        *reinterpret_cast<GVec<T, VEC>*>(gt + idx * VEC) =
                *reinterpret_cast<const GVec<T, VEC>*>(gy + ((static_cast<int64_t>(n) * p.K + k) * pv + v) * VEC);
    }
}

// Planes [H][W] and where they lie in planes of rows of Wp elements: from row ph and column pw on, zeros around them.
struct PlaneSet {
    const void* from;
    void* to;  // [copies][planes][pitch]: copy s holds the plane's element q + s at q
    int planes, H, W, ph, pw, copies;
    int pitch;  // a multiple of 16 bytes
};

struct PlanesArgs {
    PlaneSet set[2];  // x, gy
    int Wp;
    int* nonfinite;  // [channels][images][parts]: whether that part of a plane of x holds an inf or NaN
    int images, channels;
    bool pairs;       // float16: rows of gy hold two elements or more and its copy's an even number
    int each;         // planes of a workgroup, kMostPlanes at most
    int parts, share;  // workgroups to a plane, where each is 1, and pieces that each of them takes
    int64_t blocks_x, blocks;
};
constexpr int kMostPlanes = 64;

struct __attribute__((packed, aligned(2))) AnyDword {
    unsigned v;
};
struct alignas(16) Dwords {
    unsigned v[4];
};

template <typename T>
__device__ __forceinline__ bool NonFinite(T v) {
    if constexpr (sizeof(T) == 2) {
        return (__builtin_bit_cast(unsigned short, v) & 0x7c00u) == 0x7c00u;
    } else {
        return (__builtin_bit_cast(unsigned, v) & 0x7f800000u) == 0x7f800000u;
    }
}

// Both sets in one pass.  A workgroup takes a few whole planes or a part of one, whose pieces of 16 bytes are dealt out to its threads; a piece's elements are
// gathered once, and each further copy takes one more, which is asked for with the rest.  Bound by the gathers, an element of x or two of gy a lane (324 channels of
// gy, 17 images of 60^2, element by element 26.3 us, 17.0 so), and by their latency where planes are few: two pieces to a thread and no parts of planes made
// 6 images of 80 to 125 channels on 5 x 5 18.0 us instead of 16.5, 2 of 41 to 12 on 62 x 62 20.1 instead of 15.5.  64 threads to a plane, of which the 33 pieces
// of a 14 x 14 one use half, make the whole call of 256 channels, 32 images, 38.9 us instead of 35.8.  us of the call in float16, three copies of rows of whole
// granules from two kernels and now, 32 images: 64 channels at 56^2 62 -> 52, 128 at 28^2 43 -> 39, 256 at 14^2 38 -> 35, 512 at 7^2 55 -> 37.
template <typename T>
__global__ __launch_bounds__(256) void PlanesKernel(PlanesArgs p) {
    constexpr int E = 16 / sizeof(T);
    __shared__ int flags[kMostPlanes];
    for (int64_t block = blockIdx.x; block < p.blocks; block += gridDim.x) {
        const bool of_x = block < p.blocks_x;
        const PlaneSet& o = p.set[of_x ? 0 : 1];
        const int64_t own = of_x ? block : block - p.blocks_x;
        const int64_t plane0 = p.parts > 1 ? static_cast<unsigned>(own) / static_cast<unsigned>(p.parts) : own * p.each;
        const int planes = static_cast<int>(min(static_cast<int64_t>(p.each), o.planes - plane0)), pieces = o.pitch / E;
        int begin = 0, end = planes * pieces, part = 0;
        if (p.parts > 1) {  // (of one plane)
            part = static_cast<int>(own - plane0 * p.parts);
            begin = part * p.share, end = min(pieces, begin + p.share);
        }
        if (of_x) {
            if (threadIdx.x < kMostPlanes) flags[threadIdx.x] = 0;
            __syncthreads();
        }
        for (int i = begin + threadIdx.x; i < end; i += 256) {
            const int local = static_cast<unsigned>(i) / static_cast<unsigned>(pieces), q = (i - local * pieces) * E;
            const int64_t plane = plane0 + local;
            const T* const from = static_cast<const T*>(o.from) + plane * o.H * o.W;
            T* const to = static_cast<T*>(o.to) + plane * o.pitch + q;
            int row = static_cast<unsigned>(q) / static_cast<unsigned>(p.Wp), col = q - row * p.Wp;
            if constexpr (sizeof(T) == 2) {
                if (!of_x && p.pairs) {  // rows of an even pitch without padding in front: both elements of a dword lie in one row
                    Dwords out;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const bool inside = row < o.H && col < o.W, alone = col + 1 == o.W;  // (nothing behind an odd row's last element is read)
                        const unsigned v = reinterpret_cast<const AnyDword*>(from + (inside ? row * o.W + col - alone : 0))->v >> (alone ? 16 : 0);
                        out.v[e] = inside ? v : 0u;
                        if ((col += 2) == p.Wp) col = 0, ++row;
                    }
                    *reinterpret_cast<Dwords*>(to) = out;
                    continue;
                }
            }
            auto next = [&] {
                const int h = row - o.ph, w = col - o.pw;
                const bool inside = h >= 0 && h < o.H && w >= 0 && w < o.W;
                const T v = from[inside ? h * o.W + w : 0];
                if (++col == p.Wp) col = 0, ++row;
                return inside ? v : T(0);
            };
            GVec<T, E> out;
#pragma unroll
            for (int e = 0; e < E; ++e) out.v[e] = next();
            T more = o.copies > 1 ? next() : T(0);
            bool bad = false;
#pragma unroll
            for (int e = 0; e < E; ++e) bad |= NonFinite<T>(out.v[e]);
            if (of_x && bad) flags[local] = 1;
            *reinterpret_cast<GVec<T, E>*>(to) = out;
            for (int s = 1; s < o.copies; ++s) {
#pragma unroll
                for (int e = 0; e + 1 < E; ++e) out.v[e] = out.v[e + 1];
                out.v[E - 1] = more;
                *reinterpret_cast<GVec<T, E>*>(to + static_cast<int64_t>(s) * o.planes * o.pitch) = out;
                if (s + 1 < o.copies) more = next();
            }
        }
        if (of_x) {
            __syncthreads();
            if (threadIdx.x < planes) {
                const int plane = static_cast<int>(plane0) + threadIdx.x, n = plane / p.channels;
                p.nonfinite[(static_cast<int64_t>(plane - n * p.channels) * p.images + n) * p.parts + part] = flags[threadIdx.x];
            }
            __syncthreads();
        }
    }
}

// Filter taps of the input channels of the planes flagged in `nonfinite`, summed the reference's way: gw[k][c][r][s] = sum over (n, oh, ow) of
// gy[n][k][oh][ow] * col, col = x[n][c][oh*sh - ph + r][ow*sw - pw + s] or the padding's zero (still multiplied, as TensorDot
// multiplies Im2Col's zeros: CX/native/native_device/conv.cc:91-124).  Grid (C, slices); a wave per output, lanes over the sum.
template <typename T>
__global__ __launch_bounds__(256) void GradWeightChannelFixupKernel(GradWeightArgs p, const int* nonfinite, int parts, T* gw) {
    const int c = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t flags = static_cast<int64_t>(p.N) * parts;
    int any = 0;
    for (int64_t i = lane; i < flags; i += 64) any |= nonfinite[c * flags + i];
    if (__ballot(any) == 0) return;  // (a wave)
    const T* x = static_cast<const T*>(p.x);
    const T* gy = static_cast<const T*>(p.gy);
    const int taps = p.kh * p.kw, outputs = p.K * taps;
    const int64_t plane = static_cast<int64_t>(p.OH) * p.OW, total = plane * p.N;
    for (int o = blockIdx.y * 4 + wave; o < outputs; o += gridDim.y * 4) {
        const int k = o / taps, r = (o - k * taps) / p.kw, s = o % p.kw;
        float acc = 0.0f;
        for (int64_t i = lane; i < total; i += 64) {
            const int n = static_cast<int>(i / plane);
            const int pix = static_cast<int>(i - n * plane);
            const int oh = pix / p.OW, ow = pix - oh * p.OW;
            const int ih = oh * p.sh - p.ph + r, iw = ow * p.sw - p.pw + s;
            const float xv = (ih >= 0 && ih < p.H && iw >= 0 && iw < p.W)
                                     ? static_cast<float>(x[((static_cast<int64_t>(n) * p.C + c) * p.H + ih) * p.W + iw]) : 0.0f;
            acc += static_cast<float>(gy[(static_cast<int64_t>(n) * p.K + k) * plane + pix]) * xv;
        }
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) acc += __shfl_down(acc, d);
        if (lane == 0) gw[(static_cast<int64_t>(k) * p.C + c) * taps + (o - k * taps)] = static_cast<T>(acc);
    }
}

int WidestVec(int64_t extent, int64_t item, const void* a, const void* b) {
    int v = static_cast<int>(16 / item);
    while (v > 1 && (extent % v != 0 || reinterpret_cast<uintptr_t>(a) % (v * item) != 0 || reinterpret_cast<uintptr_t>(b) % (v * item) != 0)) v /= 2;
    return v;
}

struct GradWeightPlan {
    GradWeightArgs a{};
    size_t col_bytes = 0, gyt_bytes = 0;
    hipcx_array gy_t{}, col_view{};  // Dot operands: [K, NP] and the [NP, C*kh*kw] view of col_t
};

size_t RoundUp256(size_t v) { return (v + 255) / 256 * 256; }

GradWeightPlan PlanGradWeight(const hipcx_array* x, const hipcx_array* gy, const hipcx_array* gw, const int64_t* stride, const int64_t* pad,
                              int cover_all) {
    ValidateArray(x, "x");
    ValidateArray(gy, "gy");
    ValidateArray(gw, "gw");
    HIPCX_REQUIRE(x->ndim == 4 && gy->ndim == 4 && gw->ndim == 4, HIPCX_NOT_IMPLEMENTED_ERROR, "hip convolution supports 2 spatial dimensions");
    HIPCX_REQUIRE(IsFloatDtype(gw->dtype) && x->dtype == gw->dtype && gy->dtype == gw->dtype, HIPCX_DTYPE_ERROR,
                  "conv_grad_weight: x and gy must have gw's floating point dtype (cast with hipcx_copy first)");
    HIPCX_REQUIRE(IsContiguous(x) && IsContiguous(gy) && IsContiguous(gw), HIPCX_NOT_IMPLEMENTED_ERROR,
                  "hip conv_grad_weight: x, gy and gw must be C-contiguous");
    HIPCX_REQUIRE(stride && pad && stride[0] > 0 && stride[1] > 0 && pad[0] >= 0 && pad[1] >= 0, HIPCX_DIMENSION_ERROR, "invalid stride or pad");
    HIPCX_REQUIRE(gw->shape[1] == x->shape[1], HIPCX_DIMENSION_ERROR, "conv_grad_weight: gw and x disagree on the input channels");
    const int64_t oh = hipcx_conv_out_dim(x->shape[2], gw->shape[2], stride[0], pad[0], cover_all);
    const int64_t ow = hipcx_conv_out_dim(x->shape[3], gw->shape[3], stride[1], pad[1], cover_all);
    HIPCX_REQUIRE(gy->shape[0] == x->shape[0] && gy->shape[1] == gw->shape[0] && gy->shape[2] == oh && gy->shape[3] == ow, HIPCX_DIMENSION_ERROR,
                  "gy has the wrong shape " + ShapeStr(gy));
    for (int i = 0; i < 4; ++i) {
        HIPCX_REQUIRE(x->shape[i] < (1LL << 31) && gw->shape[i] < (1LL << 31) && gy->shape[i] < (1LL << 31), HIPCX_NOT_IMPLEMENTED_ERROR, "extent too large");
    }
    GradWeightPlan pl;
    GradWeightArgs& a = pl.a;
    a.x = x->data;
    a.gy = gy->data;
    a.N = static_cast<int>(x->shape[0]), a.C = static_cast<int>(x->shape[1]), a.H = static_cast<int>(x->shape[2]), a.W = static_cast<int>(x->shape[3]);
    a.K = static_cast<int>(gw->shape[0]), a.kh = static_cast<int>(gw->shape[2]), a.kw = static_cast<int>(gw->shape[3]);
    a.OH = static_cast<int>(oh), a.OW = static_cast<int>(ow);
    a.sh = static_cast<int>(stride[0]), a.sw = static_cast<int>(stride[1]), a.ph = static_cast<int>(pad[0]), a.pw = static_cast<int>(pad[1]);
    const int64_t it = ItemSize(gw->dtype);
    const int64_t np = static_cast<int64_t>(a.N) * a.OH * a.OW;
    const int64_t ckk = static_cast<int64_t>(a.C) * a.kh * a.kw;
    pl.col_bytes = RoundUp256(static_cast<size_t>(ckk * np * it));
    pl.gyt_bytes = RoundUp256(static_cast<size_t>(a.K * np * it));
    pl.gy_t.dtype = gw->dtype, pl.gy_t.ndim = 2;
    pl.gy_t.shape[0] = a.K, pl.gy_t.shape[1] = np;
    pl.gy_t.strides[0] = np * it, pl.gy_t.strides[1] = it;
    pl.col_view.dtype = gw->dtype, pl.col_view.ndim = 2;
    pl.col_view.shape[0] = np, pl.col_view.shape[1] = ckk;
    pl.col_view.strides[0] = it, pl.col_view.strides[1] = np * it;
    return pl;
}

hipcx_array GwAsMatrix(const hipcx_array* gw) {
    hipcx_array m{};
    m.data = gw->data, m.dtype = gw->dtype, m.ndim = 2;
    m.shape[0] = gw->shape[0];
    m.shape[1] = gw->shape[1] * gw->shape[2] * gw->shape[3];
    m.strides[1] = ItemSize(gw->dtype);
    m.strides[0] = m.shape[1] * m.strides[1];
    return m;
}

template <typename T>
void RunLayouts(const GradWeightArgs& a, hipStream_t stream) {
    const int64_t cap = static_cast<int64_t>(NumCUs()) * 32;
    auto grid = [&](int64_t n) { int64_t b = (n + 255) / 256; return dim3(static_cast<unsigned>(b > cap ? cap : (b < 1 ? 1 : b))); };
    {
        const int v = WidestVec(a.OW, sizeof(T), a.col_t, a.col_t);
        const int64_t total = static_cast<int64_t>(a.C) * a.kh * a.kw * a.N * a.OH * (a.OW / v);
        switch (v) {
            case 8: hipLaunchKernelGGL((Im2ColTKernel<T, (sizeof(T) <= 2 ? 8 : 1)>), grid(total), dim3(256), 0, stream, a, total); break;
            case 4: hipLaunchKernelGGL((Im2ColTKernel<T, (sizeof(T) <= 4 ? 4 : 1)>), grid(total), dim3(256), 0, stream, a, total); break;
            case 2: hipLaunchKernelGGL((Im2ColTKernel<T, 2>), grid(total), dim3(256), 0, stream, a, total); break;
            default: hipLaunchKernelGGL((Im2ColTKernel<T, 1>), grid(total), dim3(256), 0, stream, a, total); break;
        }
        CheckLaunch("im2col (weight gradient)");
    }
    {
        const int64_t plane = static_cast<int64_t>(a.OH) * a.OW;
        const int v = WidestVec(plane, sizeof(T), a.gy, a.gy_t);
        const int64_t total = static_cast<int64_t>(a.K) * a.N * (plane / v);
        switch (v) {
            case 8: hipLaunchKernelGGL((TransposeNKKernel<T, (sizeof(T) <= 2 ? 8 : 1)>), grid(total), dim3(256), 0, stream, a, total); break;
            case 4: hipLaunchKernelGGL((TransposeNKKernel<T, (sizeof(T) <= 4 ? 4 : 1)>), grid(total), dim3(256), 0, stream, a, total); break;
            case 2: hipLaunchKernelGGL((TransposeNKKernel<T, 2>), grid(total), dim3(256), 0, stream, a, total); break;
            default: hipLaunchKernelGGL((TransposeNKKernel<T, 1>), grid(total), dim3(256), 0, stream, a, total); break;
        }
        CheckLaunch("gy transpose (weight gradient)");
    }
}

}  // namespace
}  // namespace hipcx

namespace hipcx {
// nd_ops.hip: arrays without exactly two spatial axes
void ConvGradWeightNd(const hipcx_array* x, const hipcx_array* gy, const int64_t* stride, const int64_t* pad, int cover_all, const hipcx_array* gw,
                      void* stream);
}  // namespace hipcx

using namespace hipcx;

// conv.hip: accumulated batch of matrix products on the MFMA kernel
int BatchedProductSlices(int64_t m, int64_t n, int64_t depth, int batch, int dtype);
size_t BatchedProductPartialBytes(int64_t m, int64_t n, int64_t depth, int batch, int dtype);
bool BatchedProductApplies(const void* a, int64_t a_row, int64_t a_slice, const void* bt, int64_t bt_row, int64_t bt_slice, int64_t depth,
                           const void* out, int dtype);
void LaunchBatchedProduct(int dtype, const void* a, int64_t a_row, int64_t a_slice, const void* bt, int64_t bt_row, int64_t bt_slice, int64_t m,
                          int64_t n, int64_t depth, int batch, void* out, float* partial, hipStream_t stream, int taps_r = 0, int taps_s = 0,
                          int64_t r_stride = 0, int64_t s_stride = 0);

namespace {
// The product behind a weight gradient and the float sums it splits into.  float16 within 2 GiB runs in batched_product.hip.
struct Product {
    BatchedOperands o{};  // (of the data type: float32 operands too)
    int dtype = 0;
    bool half = false;
    size_t partial_bytes = 0;
};

Product PlanProduct(const void* a, int64_t a_row, int64_t a_slice, const void* b, int64_t b_row, int64_t b_slice, int64_t m, int64_t n, int64_t depth, int64_t batch,
                    void* out, int dtype, int taps_r = 0, int taps_s = 0, int64_t r_stride = 0, int64_t s_stride = 0, int64_t s_pair_stride = 0) {
    Product pr;
    BatchedOperands& o = pr.o;
    o.a = static_cast<const half_t*>(a), o.b = static_cast<const half_t*>(b), o.out = static_cast<half_t*>(out);
    o.M = static_cast<int>(m), o.N = static_cast<int>(n), o.depth = static_cast<int>(depth), o.batch = static_cast<int>(batch);
    o.a_row = a_row, o.a_slice = a_slice, o.b_row = b_row, o.b_slice = b_slice;
    o.taps_r = taps_r, o.taps_s = taps_s, o.r_stride = r_stride, o.s_stride = s_stride, o.s_pair_stride = s_pair_stride;
    pr.dtype = dtype;
    pr.half = dtype == HIPCX_FLOAT16 && std::max(std::max(m, n), depth) < (1LL << 31) && HalfProductApplies(o);
    if (pr.half) {
        const int slices = HalfProductSlices(o);
        pr.partial_bytes = slices > 1 ? static_cast<size_t>(slices) * m * n * sizeof(float) : 0;
    } else {
        pr.partial_bytes = BatchedProductPartialBytes(m, n, depth, o.batch, dtype);
    }
    return pr;
}

void RunProduct(const Product& pr, void* partial, hipStream_t stream) {
    const BatchedOperands& o = pr.o;
    float* const sums = pr.partial_bytes ? static_cast<float*>(partial) : nullptr;
    if (pr.half) HalfProduct(o, sums, HalfProductSlices(o), stream);
    else LaunchBatchedProduct(pr.dtype, o.a, o.a_row, o.a_slice, o.b, o.b_row, o.b_slice, o.M, o.N, o.depth, o.batch, o.out, sums, stream, o.taps_r, o.taps_s, o.r_stride, o.s_stride);
}

// A 1x1 filter at stride 1 without padding: gw[k][c] = sum over images of gy_n [K, pixels] @ x_n [C, pixels]^T, which the matrix kernels
// read from gy and x where they lie (rows along the pixels, one matrix per image) -- no Im2Col, no transposed copy of gy.
Product PlanPointwise(const GradWeightPlan& pl, const void* x, const void* gy, void* gw, int dtype) {
    const GradWeightArgs& a = pl.a;
    const int64_t pixels = static_cast<int64_t>(a.H) * a.W;
    return PlanProduct(gy, pixels, a.K * pixels, x, pixels, a.C * pixels, a.K, a.C, pixels, a.N, gw, dtype);
}

// float16 planes of an even number of pixels, 32 at least, are read in place.  The general kernel takes whole 16-byte granules, long enough to fill
// reduction steps.
bool DirectPointwise(const GradWeightPlan& pl, const Product& pr, const hipcx_array* x, const hipcx_array* gy, const hipcx_array* gw) {
    static const bool enabled = [] { const char* e = getenv("HIPCX_GRAD_WEIGHT_DIRECT"); return e == nullptr || e[0] != '0'; }();
    const GradWeightArgs& a = pl.a;
    if (!enabled || a.kh != 1 || a.kw != 1 || a.sh != 1 || a.sw != 1 || a.ph != 0 || a.pw != 0 || a.OH != a.H || a.OW != a.W) return false;
    const int64_t pixels = static_cast<int64_t>(a.H) * a.W;
    if (a.N < 1) return false;
    if (pr.half) return true;
    return pixels >= 256 && BatchedProductApplies(gy->data, pixels, static_cast<int64_t>(a.K) * pixels, x->data, pixels, static_cast<int64_t>(a.C) * pixels,
                                                  pixels, gw->data, gw->dtype);
}

// Filters larger than 1x1 at stride 1: shifted zero-padded copies of x instead of Im2Col (see the top of the file).
struct ShiftedPlan {
    bool ok = false;
    PlanesArgs a{};
    Product product;  // (of null operands)
    size_t xs_bytes = 0, gyp_bytes = 0, flag_bytes = 0;
};

Product ShiftedProduct(const ShiftedPlan& sp, const GradWeightArgs& g, void* gw, int dtype) {
    const PlaneSet &x = sp.a.set[0], &gy = sp.a.set[1];
    const int64_t copy = static_cast<int64_t>(x.planes) * x.pitch;
    return PlanProduct(gy.to, gy.pitch, static_cast<int64_t>(g.K) * gy.pitch, x.to, x.pitch, static_cast<int64_t>(g.C) * x.pitch, g.K,
                       static_cast<int64_t>(g.C) * g.kh * g.kw, static_cast<int64_t>(g.OH) * sp.a.Wp, g.N, gw, dtype, g.kh, g.kw, sp.a.Wp, copy,
                       x.copies == g.kw ? 2 * copy : 2);
}

// `pairs`: two copies, rows rounded up to an even width, for the float16 product; false: kw copies of rows of whole granules.
ShiftedPlan PlanShifted(const GradWeightPlan& pl, int dtype, bool pairs) {
    ShiftedPlan sp;
    static const bool enabled = [] { const char* e = getenv("HIPCX_GRAD_WEIGHT_SHIFTED"); return e == nullptr || e[0] != '0'; }();
    const GradWeightArgs& g = pl.a;
    if (!enabled || (dtype != HIPCX_FLOAT16 && dtype != HIPCX_FLOAT32)) return sp;
    if (g.sh != 1 || g.sw != 1 || g.kh * g.kw == 1) return sp;
    if (g.OH != g.H + 2 * g.ph - g.kh + 1 || g.OW != g.W + 2 * g.pw - g.kw + 1) return sp;  // cover_all adds nothing at stride 1
    const int64_t N = g.N, it = ItemSize(dtype), epc = 16 / it, pw = g.pw, W = g.W;
    const int64_t Wp = pairs ? (std::max<int64_t>(W + pw, g.OW) + 1) / 2 * 2 : (W + 2 * pw + epc - 1) / epc * epc;
    const int64_t Hp = g.H + 2 * static_cast<int64_t>(g.ph), copies = pairs ? std::min(g.kw, 2) : g.kw;
    // windows of a pair's copies start up to kw - 1 elements later than those of copies of their own, and end as much later
    const int64_t pitch_x = (Hp * Wp + (pairs ? (g.kw - 1) / 2 * 2 : 0) + epc - 1) / epc * epc, pitch_gy = (g.OH * Wp + epc - 1) / epc * epc;
    // worth it when kw copies of rows of whole granules are smaller than the kh*kw-fold Im2Col, also where it is two copies of shorter rows: small planes and
    // filters are faster as one Dot.  us, Im2Col and two copies: 2x2 on 7 x 7 8.7 and 15.8, 3x3 on 9 x 3 10.5 and 19.1, 5x5 on 13 x 3 99 and 214.
    if (g.kw * Hp * ((W + 2 * pw + epc - 1) / epc * epc) >= static_cast<int64_t>(g.kh) * g.kw * g.OH * g.OW) return sp;
    const int64_t most = int64_t{1} << 31, planes = N * (static_cast<int64_t>(g.C) + g.K);
    if (static_cast<int64_t>(g.H) * W == 0 || planes == 0 || pitch_x + 256 * epc >= most || N * g.C >= most || N * g.K >= most) return sp;  // (the copy kernel's 32-bit indices)
    sp.a.set[0] = PlaneSet{g.x, nullptr, static_cast<int>(N * g.C), g.H, g.W, g.ph, g.pw, static_cast<int>(copies), static_cast<int>(pitch_x)};
    sp.a.set[1] = PlaneSet{g.gy, nullptr, static_cast<int>(N * g.K), g.OH, g.OW, 0, 0, 1, static_cast<int>(pitch_gy)};
    sp.a.Wp = static_cast<int>(Wp);
    sp.a.images = g.N, sp.a.channels = g.C;
    sp.a.pairs = Wp % 2 == 0 && g.OW >= 2;
    // A piece to a thread: planes together, or less where that leaves compute units without a workgroup, or parts of a plane; two pieces once the chip is full.
    const int64_t pieces = pitch_x / epc, cus = NumCUs();
    sp.a.each = static_cast<int>(std::max<int64_t>(1, std::min<int64_t>({kMostPlanes, (planes * pieces >= 4096 * cus ? 512 : 256) / pieces, planes / cus})));
    sp.a.parts = static_cast<int>(std::max<int64_t>(1, std::min<int64_t>((pieces + 255) / 256, 8 * cus / planes)));
    sp.a.share = static_cast<int>((pieces + sp.a.parts - 1) / sp.a.parts);
    sp.a.blocks_x = (sp.a.set[0].planes + int64_t{sp.a.each} - 1) / sp.a.each * sp.a.parts;
    sp.a.blocks = sp.a.blocks_x + (sp.a.set[1].planes + int64_t{sp.a.each} - 1) / sp.a.each * sp.a.parts;
    sp.flag_bytes = RoundUp256(static_cast<size_t>(N * g.C) * sp.a.parts * sizeof(int));
    sp.xs_bytes = RoundUp256(static_cast<size_t>(copies * N * g.C * pitch_x * it));
    sp.gyp_bytes = RoundUp256(static_cast<size_t>(N * g.K * pitch_gy * it));
    sp.product = ShiftedProduct(sp, g, nullptr, dtype);
    sp.ok = !pairs || sp.product.half;
    return sp;
}

ShiftedPlan PlanShifted(const GradWeightPlan& pl, int dtype) {
    if (dtype == HIPCX_FLOAT16) {
        const ShiftedPlan sp = PlanShifted(pl, dtype, true);
        if (sp.ok) return sp;
    }
    return PlanShifted(pl, dtype, false);
}

// The product of the staged operands, whose rows are the pixels of all images.  float16 of an even number of pixels only, and of 1 GFLOP or 2048 pixels at
// least: the rest are Dots.  (us of the call, batch 8, as
// product and as Dot: 1024 to 512 channels on 7 x 7, 392 pixels, 15.5, 11.9; 512 to 256 on 14 x 14, 1568 pixels, 18.4, 14.1; 256 to 128 on 28 x 28,
// 6272 pixels, 20, 33; 1024 to 2048 on 7 x 7, 1.6 GFLOP, 18, 22.5.)
Product StagedProduct(const GradWeightPlan& pl, void* gw, int dtype) {
    const int64_t np = pl.gy_t.shape[1];
    Product pr = PlanProduct(pl.a.gy_t, np, 0, pl.a.col_t, np, 0, pl.a.K, pl.col_view.shape[1], np, 1, gw, dtype);
    pr.half = pr.half && (np >= 2048 || 2.0 * pl.a.K * pl.col_view.shape[1] * np >= 1e9);
    return pr;
}

template <typename T>
void RunPlanes(const PlanesArgs& a, hipStream_t stream) {
    hipLaunchKernelGGL((PlanesKernel<T>), dim3(static_cast<unsigned>(std::min<int64_t>(a.blocks, 1 << 22))), dim3(256), 0, stream, a);
    CheckLaunch("padded planes (weight gradient)");
}

template <typename T>
void RunChannelFixup(const GradWeightArgs& g, const PlanesArgs& planes, void* gw, hipStream_t stream) {
    const int outputs = g.K * g.kh * g.kw;
    const int slices = std::max(1, std::min(outputs / 4, 16));
    hipLaunchKernelGGL((GradWeightChannelFixupKernel<T>), dim3(static_cast<unsigned>(g.C), static_cast<unsigned>(slices)), dim3(256), 0, stream, g,
                       planes.nonfinite, planes.parts, static_cast<T*>(gw));
    CheckLaunch("non-finite channels (weight gradient)");
}
}  // namespace

extern "C" {

size_t hipcx_conv_grad_weight_workspace_size(const hipcx_array* x, const hipcx_array* gy, const hipcx_array* gw, const int64_t* stride,
                                             const int64_t* pad, int cover_all) {
    try {
        if (x == nullptr || gy == nullptr || gw == nullptr) return 0;
        if (x->ndim != 4) return 0;  // the n-axis kernel needs none
        GradWeightPlan pl = PlanGradWeight(x, gy, gw, stride, pad, cover_all);
        hipcx_array out = GwAsMatrix(gw);
        // Which path the call takes depends on the alignment of the data pointers, which a caller sizing its workspace from
        // descriptors alone may not have yet: the answer covers both.
        const int64_t pixels = static_cast<int64_t>(pl.a.H) * pl.a.W;
        const Product in_place = PlanPointwise(pl, nullptr, nullptr, nullptr, gw->dtype), copied = StagedProduct(pl, nullptr, gw->dtype);
        const size_t direct = std::max(in_place.partial_bytes, BatchedProductPartialBytes(pl.a.K, pl.a.C, pixels, pl.a.N, gw->dtype)) + 256;
        const size_t staged = pl.col_bytes + pl.gyt_bytes + std::max(hipcx_dot_workspace_size(&pl.gy_t, &pl.col_view, &out), copied.half ? copied.partial_bytes : 0);
        const ShiftedPlan sp = PlanShifted(pl, gw->dtype);
        const size_t shifted = sp.ok ? sp.xs_bytes + sp.gyp_bytes + sp.product.partial_bytes + sp.flag_bytes + 256 : 0;
        return std::max(std::max(direct, staged), shifted);
    } catch (...) {
        return 0;
    }
}

int hipcx_conv_grad_weight(const hipcx_array* x, const hipcx_array* gy, const int64_t* stride, const int64_t* pad, int cover_all,
                           const hipcx_array* gw, void* workspace, size_t workspace_bytes, void* stream) {
    return Guard([&] {
        if (x != nullptr && x->ndim != 4) {  // not two spatial axes: nd_ops.hip
            ConvGradWeightNd(x, gy, stride, pad, cover_all, gw, stream);
            return;
        }
        GradWeightPlan pl = PlanGradWeight(x, gy, gw, stride, pad, cover_all);
        hipcx_array out = GwAsMatrix(gw);
        if (out.shape[0] == 0 || out.shape[1] == 0) return;
        if (pl.gy_t.shape[1] == 0) {  // an empty batch or plane: the sum over nothing
            hipcx_scalar zero{HIPCX_KIND_INT, 0, 0, 0.0};
            int rc = hipcx_fill(gw, zero, stream);
            HIPCX_REQUIRE(rc == HIPCX_OK, rc, hipcx_last_error());
            return;
        }
        const Product in_place = PlanPointwise(pl, x->data, gy->data, gw->data, gw->dtype);
        if (DirectPointwise(pl, in_place, x, gy, gw)) {
            HIPCX_REQUIRE(in_place.partial_bytes == 0 || (workspace != nullptr && workspace_bytes >= in_place.partial_bytes), HIPCX_CHAINERX_ERROR,
                          "conv_grad_weight workspace too small: need " + std::to_string(in_place.partial_bytes) + " bytes");
            HIPCX_REQUIRE(reinterpret_cast<uintptr_t>(workspace) % 16 == 0, HIPCX_CHAINERX_ERROR, "workspace must be 16-byte aligned");
            RunProduct(in_place, workspace, AsStream(stream));
            return;
        }
        ShiftedPlan sp = PlanShifted(pl, gw->dtype);
        if (sp.ok && reinterpret_cast<uintptr_t>(workspace) % 16 == 0 && reinterpret_cast<uintptr_t>(gw->data) % 16 == 0) {
            const size_t need = sp.xs_bytes + sp.gyp_bytes + sp.product.partial_bytes + sp.flag_bytes;
            HIPCX_REQUIRE(workspace != nullptr && workspace_bytes >= need, HIPCX_CHAINERX_ERROR,
                          "conv_grad_weight workspace too small: need " + std::to_string(need) + " bytes");
            char* ws = static_cast<char*>(workspace);
            sp.a.set[0].to = ws, sp.a.set[1].to = ws + sp.xs_bytes;
            sp.a.nonfinite = reinterpret_cast<int*>(ws + sp.xs_bytes + sp.gyp_bytes + sp.product.partial_bytes);
            hipStream_t st = AsStream(stream);
            if (gw->dtype == HIPCX_FLOAT16) RunPlanes<half_t>(sp.a, st);
            else RunPlanes<float>(sp.a, st);
            const GradWeightArgs& g = pl.a;
            RunProduct(ShiftedProduct(sp, g, gw->data, gw->dtype), ws + sp.xs_bytes + sp.gyp_bytes, st);
            if (gw->dtype == HIPCX_FLOAT16) RunChannelFixup<half_t>(g, sp.a, gw->data, st);
            else RunChannelFixup<float>(g, sp.a, gw->data, st);
            return;
        }
        const size_t dot_bytes = hipcx_dot_workspace_size(&pl.gy_t, &pl.col_view, &out);
        const size_t need = pl.col_bytes + pl.gyt_bytes + dot_bytes;
        HIPCX_REQUIRE(workspace != nullptr && workspace_bytes >= need, HIPCX_CHAINERX_ERROR,
                      "conv_grad_weight workspace too small: need " + std::to_string(need) + " bytes");
        HIPCX_REQUIRE(reinterpret_cast<uintptr_t>(workspace) % 16 == 0, HIPCX_CHAINERX_ERROR, "workspace must be 16-byte aligned");
        char* ws = static_cast<char*>(workspace);
        pl.a.col_t = ws;
        pl.a.gy_t = ws + pl.col_bytes;
        pl.col_view.data = pl.a.col_t;
        pl.gy_t.data = pl.a.gy_t;
        hipStream_t st = AsStream(stream);
        VisitFloatDtype(gw->dtype, [&](auto tag) {
            using T = typename decltype(tag)::type;
            RunLayouts<T>(pl.a, st);
        });
        const Product copied = StagedProduct(pl, gw->data, gw->dtype);
        if (copied.half && workspace_bytes >= pl.col_bytes + pl.gyt_bytes + copied.partial_bytes) {
            RunProduct(copied, ws + pl.col_bytes + pl.gyt_bytes, st);
            return;
        }
        int rc = hipcx_dot(&pl.gy_t, &pl.col_view, &out, ws + pl.col_bytes + pl.gyt_bytes, dot_bytes, stream);
        HIPCX_REQUIRE(rc == HIPCX_OK, rc, hipcx_last_error());
    });
}

}  // extern "C"
