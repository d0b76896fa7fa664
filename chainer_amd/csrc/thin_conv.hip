// float32 and float16 convolutions whose outputs are sums of at most 32 terms: a network's first layer, 3 channels x 3 x 3.
//
// Such a layer is its output: on the general kernel's 256 x 64 tiles, two steps long, the loads, the staging and the way out follow one another, after a
// channels-last copy of x.  Here a wave owns 64 filters, whose terms stay in its registers, and walks blocks of 32 output pixels: a lane gathers the
// terms of its pixel from NCHW, where neighbouring lanes' lie next to each other, as operands of v_mfma_f32_32x32x2_f32, and the sums leave as 128 bytes
// of a plane each.  Neither LDS nor a barrier.  Bound by writing the result.  us, against the general
// kernel and its copies: 256 images of 3 channels at 32^2, 3x3 into 64 62 -> 26, one image 23 -> 8; 256 of 1 at 28^2, 5x5 into 32 68 -> 22; 4 of 3 at 224^2
// into 64 56 -> 24; 1x1, 256 of 32 at 16^2 into 256 41 -> 29.  Relative error against 64 bits 9.2e-8 (9.3e-8 before).
// float16, the first and the third of these 44 -> 28 and 41 -> 24.
#include <algorithm>

#include "igemm.h"
#include "launch_profile.h"
#include "nchw_conv.h"
#include "thin_conv.h"

namespace hipcx {
namespace {

constexpr int kOut = 0x7fffffff;  // an offset beyond any buffer: loads give zeros, stores are dropped

struct ThinConvArgs {
    const void* x;
    const void* w;
    const void* bias;
    int64_t bias_stride;
    void* out;
    int C, H, W, K, R, S, OW, P;
    int stride_h, stride_w, pad_h, pad_w;
    int M;       // images * P
    int blocks;  // of 32 pixels
    unsigned x_bytes, w_bytes, out_bytes;
    FastDiv div_P, div_OW;
};

template <typename T>
__device__ __forceinline__ float LoadFloat(__amdgpu_buffer_rsrc_t r, int element, bool in) {
    if constexpr (sizeof(T) == 4) return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, in ? element * 4 : kOut, 0, 0));
    else return static_cast<float>(__builtin_bit_cast(half_t, static_cast<unsigned short>(__builtin_amdgcn_raw_buffer_load_b16(r, in ? element * 2 : kOut, 0, 0))));
}

// STEPS: pairs of terms.
template <typename T, int STEPS>
__global__ __launch_bounds__(256, 3) void ThinConvKernel(ThinConvArgs p) {
    const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n0 = blockIdx.y * 64;
    const int terms = p.C * p.R * p.S;
    const __amdgpu_buffer_rsrc_t xr = MakeRsrc(p.x, p.x_bytes), wr = MakeRsrc(p.w, p.w_bytes), outr = MakeRsrc(p.out, p.out_bytes);

    // term 2 * k + h of each step: where it lies from the window's corner, and its row and column of the filter
    int off[STEPS], at[STEPS];
    float wf[2][STEPS];
#pragma unroll
    for (int k = 0; k < STEPS; ++k) {
        const int term = 2 * k + h, c = term / (p.R * p.S), rs = term - c * p.R * p.S, fr = rs / p.S, fs = rs - fr * p.S;
        off[k] = (c * p.H + fr) * p.W + fs;
        at[k] = term < terms ? fr << 16 | fs : 0x7fff << 16;  // (a row beyond any plane)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int n = n0 + j * 32 + r;
            wf[j][k] = LoadFloat<T>(wr, n * terms + term, (term < terms) & (n < p.K));
        }
    }
    // lane holds pixel r, filters 8 * (v / 4) + 4 * h + v % 4 of each half
    float bias[2][16];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int n = n0 + j * 32 + 8 * (v / 4) + 4 * h + v % 4;
            bias[j][v] = p.bias != nullptr && n < p.K ? static_cast<float>(static_cast<const T*>(p.bias)[n * p.bias_stride]) : 0.f;
        }
    const bool whole = n0 + 64 <= p.K;

    for (int block = blockIdx.x * 4 + wave; block < p.blocks; block += gridDim.x * 4) {
        const int m = block * 32 + r;
        const bool in = m < p.M;
        const int img = p.div_P(in ? m : 0), px = (in ? m : 0) - img * p.P;
        const int oh = p.div_OW(px), ow = px - oh * p.OW;
        const int y = oh * p.stride_h - p.pad_h, x = ow * p.stride_w - p.pad_w;
        const int corner = (img * p.C * p.H + y) * p.W + x;
        float xf[STEPS];
#pragma unroll
        for (int k = 0; k < STEPS; ++k) {
            const int yy = y + (at[k] >> 16), xx = x + (at[k] & 0xffff);
            const bool ok = in & (yy >= 0) & (yy < p.H) & (xx >= 0) & (xx < p.W);
            xf[k] = LoadFloat<T>(xr, corner + off[k], ok);
        }
        float16_t acc[2];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[j][v] = 0.f;
#pragma unroll
        for (int k = 0; k < STEPS; ++k)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(wf[j][k], xf[k], acc[j], 0, 0, 0);
        const int to = ((img * p.K + n0 + 4 * h) * p.P + px) * static_cast<int>(sizeof(T));
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int n = j * 32 + 8 * (v / 4) + v % 4;  // + 4 * h
                const int o = in & (whole | (n0 + n + 4 * h < p.K)) ? to + n * p.P * static_cast<int>(sizeof(T)) : kOut;
                float s = acc[j][v];
                if (p.bias != nullptr) s += bias[j][v];
                if constexpr (sizeof(T) == 4) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(s), outr, o, 0, 0);
                else __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, static_cast<half_t>(s)), outr, o, 0, 0);
            }
    }
}

}  // namespace

bool ThinConvTakes(const hipcx_array* x, const hipcx_array* w, const int64_t* stride, const int64_t* pad, const hipcx_array* out) {
    if ((out->dtype != HIPCX_FLOAT32 && out->dtype != HIPCX_FLOAT16) || !IsContiguous(x) || !IsContiguous(w) || !IsContiguous(out)) return false;
    const int64_t N = x->shape[0], C = x->shape[1], H = x->shape[2], W = x->shape[3], K = w->shape[0], R = w->shape[2], S = w->shape[3];
    const int64_t OH = out->shape[2], OW = out->shape[3], P = OH * OW, terms = C * R * S;
    // (from 16 filters on, a quarter of a wave's: 51 -> 24 us for 256 images of 3 channels at 32^2)
    if (terms < 1 || terms > 32 || K < 16 || K > 4096) return false;
    // 32-bit offsets, 16-bit rows and columns; what lies in front of a plane's first row must not wrap
    const double limit = 2147483000.0 / 4;
    if (static_cast<double>(N) * C * H * W >= limit || static_cast<double>(N) * (K + 64) * P >= limit || static_cast<double>(K) * terms >= limit) return false;
    if (H >= 0x4000 || W >= 0x4000 || OH >= 0x4000 || OW >= 0x4000 || stride[0] >= 0x4000 || stride[1] >= 0x4000 || pad[0] >= 0x4000 || pad[1] >= 0x4000) return false;
    return OH * stride[0] < 0x3000 && OW * stride[1] < 0x3000;
}

void ThinConv(const hipcx_array* x, const hipcx_array* w, const hipcx_array* b, const int64_t* stride, const int64_t* pad, const hipcx_array* out, hipStream_t stream) {
    const int64_t N = x->shape[0], C = x->shape[1], H = x->shape[2], W = x->shape[3], K = w->shape[0], R = w->shape[2], S = w->shape[3];
    const int64_t OH = out->shape[2], OW = out->shape[3], P = OH * OW, terms = C * R * S;
    ThinConvArgs p{};
    const int64_t it = ItemSize(out->dtype);
    p.x = x->data, p.w = w->data, p.out = out->data;
    p.bias = b != nullptr ? b->data : nullptr;
    p.bias_stride = b != nullptr ? b->strides[0] / it : 0;
    p.C = static_cast<int>(C), p.H = static_cast<int>(H), p.W = static_cast<int>(W), p.K = static_cast<int>(K), p.R = static_cast<int>(R), p.S = static_cast<int>(S);
    p.OW = static_cast<int>(OW), p.P = static_cast<int>(P);
    p.stride_h = static_cast<int>(stride[0]), p.stride_w = static_cast<int>(stride[1]), p.pad_h = static_cast<int>(pad[0]), p.pad_w = static_cast<int>(pad[1]);
    p.M = static_cast<int>(N * P), p.blocks = (p.M + 31) / 32;
    p.x_bytes = static_cast<unsigned>(N * C * H * W * it), p.w_bytes = static_cast<unsigned>(K * terms * it), p.out_bytes = static_cast<unsigned>(N * K * P * it);
    p.div_P = FastDiv(p.P), p.div_OW = FastDiv(p.OW);
    const int columns = static_cast<int>((K + 63) / 64);
    // three workgroups to a compute unit, as the registers allow
    const int64_t groups = std::min<int64_t>((p.blocks + 3) / 4, std::max<int64_t>(1, 3LL * NumCUs() / columns));
    ProfileScope prof(stream, 2.0 * p.M * K * terms, it * (static_cast<double>(N) * C * H * W + static_cast<double>(K) * terms + static_cast<double>(p.M) * K));
    const dim3 grid(static_cast<unsigned>(groups), static_cast<unsigned>(columns));
    auto launch = [&](auto tag) {
        using T = decltype(tag);
        if (terms <= 16) hipLaunchKernelGGL((ThinConvKernel<T, 8>), grid, dim3(256), 0, stream, p);
        else hipLaunchKernelGGL((ThinConvKernel<T, 16>), grid, dim3(256), 0, stream, p);
    };
    if (out->dtype == HIPCX_FLOAT16) launch(half_t{});
    else launch(float{});
    CheckLaunch("thin_conv");
}

}  // namespace hipcx
