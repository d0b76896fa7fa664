// float16 convolutions of few output pixels (one image, or a handful of them in the deep layers).
//
// On 128 x 128 or 256 x 64 tiles such a layer is 8 to 32 workgroups that walk the whole reduction, and the filters are repacked first.  Here a workgroup
// owns 32 output channels x 32 pixels of an image and up to 16 waves split the reduction, in chunks of input channels; the waves' sums meet in LDS,
// where bias, batch norm, residual and ReLU follow.  Filters are read as they lie, whole lines, and regrouped through LDS that belongs to the wave;
// a lane's 144 contiguous bytes (8 channels x 9 taps) become nine operands by byte permutation.  Activations come as pairs of pixels of 8 channel planes and
// are turned round in registers into 16-byte groups of 8 channels per pixel; a 3x3 layer's patch is the rows around the tile's pixels, the taps
// that leave the plane are masked in the operands.  No barrier before the sums.  Bound by latency: launch, first loads, the waves' sums.  One image, us
// before (with the repacking) and now: 3x3 512 channels at 7^2 49.6 -> 10.1, 256 at 14^2 22.4 -> 8.7, 128 at 28^2 15.3 -> 7.4, 64 at 56^2 14.6 -> 7.7; 1x1
// 1024 -> 256 at 14^2 13.0 -> 5.4, 2048 -> 512 at 7^2 29.9 -> 11.9, 1024 -> 2048 at 14^2 with stride 2 18.6 -> 8.0.
#include <algorithm>

#include "mid_conv.h"
#include "pixel_pairs.h"
#include "small_conv.h"
#include "small_dot.h"

namespace hipcx {
namespace {

constexpr int MaxWaves(int taps) { return taps == 1 ? 16 : 8; }  // (a 3x3 chunk takes more registers)
constexpr int kTilePart = 32 * 33;  // floats of a wave's sums
constexpr int kOut = 0x7fffffff;    // an offset beyond any buffer: zeros

// 1x1: bytes of a staged row of 32 channels, filters and pixels alike; fragment reads of 16 rows start in different banks.
constexpr int kRow1 = 32 * 2 + 16;
// 3x3: a filter's 16 channels x 9 taps; a pixel's 16 channels.
constexpr int kFilter3 = 16 * 9 * 2, kRow3 = kFilter3 + 16, kPixel3 = 32;

struct SmallConvArgs {
    NchwConvArgs c;
    int nw;
    int tiles_px;  // per image
    int pairs;     // 3x3: pairs of pixels in a patch
    int wave_lds;
};

// SINGLE (1x1): pixels are loaded one by one, as planes of an odd size and strides above 1 ask for.
template <int TAPS, bool SINGLE>
__global__ __launch_bounds__(64 * MaxWaves(TAPS)) void SmallConvKernel(SmallConvArgs args) {
    const NchwConvArgs& p = args.c;
    constexpr int CK = TAPS == 1 ? 32 : 16;  // channels of a chunk
    extern __shared__ __align__(16) char lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 31, g = lane >> 5;
    int tile_px, tile_n;
    SmallDotTile(gridDim.x, blockIdx.x, args.tiles_px * p.N, tile_px, tile_n);
    const int img = tile_px / args.tiles_px;
    const int px0 = (tile_px - img * args.tiles_px) * 32;
    const int n0 = tile_n * 32;
    const int HW = p.H * p.W;
    const __amdgpu_buffer_rsrc_t xr = MakeRsrc(p.x, p.x_bytes), wr = MakeRsrc(p.wp, p.wp_bytes);
    char* const mine = lds + wave * args.wave_lds;

    float16_t acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.f;
    const int chunks = p.C / CK, per_wave = (chunks + args.nw - 1) / args.nw;
    const int begin = min(chunks, wave * per_wave), end = min(chunks, begin + per_wave);

    if constexpr (TAPS == 1) {
        char* const filters = mine;
        char* const pixels = mine + 32 * kRow1;
        // filters: 4 lanes to a row, 16 rows to a load; pixels: lane = a pair of pixels, 8 channels
        int w_off[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int n = n0 + i * 16 + (lane >> 2);
            w_off[i] = n < p.K ? (n * p.C + (lane & 3) * 8) * 2 : kOut;
        }
        const int pair = lane & 15, group = lane >> 4;
        int x_off[2];  // of the pair's pixels
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int px = px0 + pair * 2 + i;
            const int oh = px / p.OW, ow = px - oh * p.OW;
            const int at = SINGLE ? oh * p.stride * p.W + ow * p.stride : px;
            x_off[i] = px < p.P ? ((img * p.C + group * 8) * HW + at) * 2 : kOut;
        }
        Bytes16 wv[2][2];
        unsigned xv[2][8];
        auto load = [&](int st, int c) {
#pragma unroll
            for (int i = 0; i < 2; ++i) wv[st][i] = __builtin_amdgcn_raw_buffer_load_b128(wr, w_off[i], c * CK * 2, 0);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int so = (c * CK + e) * HW * 2;
                if constexpr (SINGLE) {
                    const unsigned lo = __builtin_amdgcn_raw_buffer_load_b16(xr, x_off[0], so, 0);
                    const unsigned hi = __builtin_amdgcn_raw_buffer_load_b16(xr, x_off[1], so, 0);
                    xv[st][e] = (lo & 0xffffu) | (hi << 16);
                } else {
                    xv[st][e] = __builtin_amdgcn_raw_buffer_load_b32(xr, x_off[0], so, 0);
                }
            }
        };
        auto multiply = [&](int st, auto&& next) {
#pragma unroll
            for (int i = 0; i < 2; ++i) *reinterpret_cast<Bytes16*>(filters + (i * 16 + (lane >> 2)) * kRow1 + (lane & 3) * 16) = wv[st][i];
            Bytes16 first, second;
            TurnPairs(xv[st], first, second);
            *reinterpret_cast<Bytes16*>(pixels + (pair * 2) * kRow1 + group * 16) = first;
            *reinterpret_cast<Bytes16*>(pixels + (pair * 2 + 1) * kRow1 + group * 16) = second;
            next();
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const Bytes16 wf = *reinterpret_cast<const Bytes16*>(filters + lr * kRow1 + (2 * q + g) * 16);
                const Bytes16 xf = *reinterpret_cast<const Bytes16*>(pixels + lr * kRow1 + (2 * q + g) * 16);
                MfmaTile<half_t>(wf, xf, acc);
            }
            __builtin_amdgcn_wave_barrier();
        };
        if (begin < end) {
            load(0, begin);
            if (begin + 1 < end) load(1, begin + 1);
            int c = begin;
            for (; c + 3 < end; c += 2) {
                multiply(0, [&] { load(0, c + 2); });
                multiply(1, [&] { load(1, c + 3); });
            }
            multiply(0, [&] {
                if (c + 2 < end) load(0, c + 2);
            });
            if (c + 1 < end) multiply(1, [] {});
            if (c + 2 < end) multiply(0, [] {});
        }
    } else {
        char* const filters = mine;
        char* const patch = mine + 32 * kRow3 + kPixel3;  // a pixel in front and one behind are read by masked taps
        // filters: pieces of 16 bytes, 18 to a row
        int w_off[9], w_to[9];
#pragma unroll
        for (int i = 0; i < 9; ++i) {
            const int id = i * 64 + lane, row = id / 18, piece = id - row * 18;
            w_off[i] = n0 + row < p.K ? (n0 + row) * p.C * 18 + piece * 16 : kOut;
            w_to[i] = row * kRow3 + piece * 16;
        }
        // the patch: whole rows from the one above the tile's first pixel on, contiguous in memory
        // (from an even pixel, so that no pair lies on both sides of the plane's beginning; what is negative is read by masked taps alone)
        const int first = (px0 / p.W - 1) * p.W & ~1;
        const int pairs = args.pairs;
        // this lane's pixel (MFMA column) and which of its taps lie inside the plane
        const int px = px0 + lr;
        const int y = px / p.W, x = px - y * p.W;
        unsigned inside = 0;
#pragma unroll
        for (int t = 0; t < 9; ++t) {
            const int yy = y + t / 3 - 1, xx = x + t % 3 - 1;
            inside |= static_cast<unsigned>(px < p.P && yy >= 0 && yy < p.H && xx >= 0 && xx < p.W) << t;
        }
        const int lin = min(px, p.P - 1) - first;
        constexpr int MAXP = 4;  // passes over the patch: 64 lanes, each a pair of pixels of 8 channels
        const int passes = (pairs * 2 + 63) / 64;
        for (int c = begin; c < end; ++c) {
            Bytes16 wv[9];
#pragma unroll
            for (int i = 0; i < 9; ++i) wv[i] = __builtin_amdgcn_raw_buffer_load_b128(wr, w_off[i], c * kFilter3, 0);
            unsigned xv[MAXP][8];
#pragma unroll
            for (int s = 0; s < MAXP; ++s) {
                if (s >= passes) continue;
                const int item = s * 64 + lane, group = item >= pairs ? 1 : 0, at = first + (item - group * pairs) * 2;
                const bool alone = at == HW - 1;  // the plane's last pixel: read with the one before
                const bool in = item < pairs * 2 && at >= 0 && at < HW;
                const int off = ((img * p.C + c * CK + group * 8) * HW + at - alone) * 2;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const unsigned v = __builtin_amdgcn_raw_buffer_load_b32(xr, in ? off + e * HW * 2 : kOut, 0, 0);
                    xv[s][e] = alone ? v >> 16 : v;
                }
            }
#pragma unroll
            for (int i = 0; i < 9; ++i) *reinterpret_cast<Bytes16*>(filters + w_to[i]) = wv[i];
#pragma unroll
            for (int s = 0; s < MAXP; ++s) {
                if (s >= passes) continue;
                const int item = s * 64 + lane, group = item >= pairs ? 1 : 0, at = item - group * pairs;
                Bytes16 a, b;
                TurnPairs(xv[s], a, b);
                if (item < pairs * 2) {
                    *reinterpret_cast<Bytes16*>(patch + at * 2 * kPixel3 + group * 16) = a;
                    *reinterpret_cast<Bytes16*>(patch + (at * 2 + 1) * kPixel3 + group * 16) = b;
                }
            }
            __builtin_amdgcn_wave_barrier();
            unsigned h[36];  // 8 channels x 9 taps of this lane's filter
#pragma unroll
            for (int i = 0; i < 9; ++i) {
                const Bytes16 v = *reinterpret_cast<const Bytes16*>(filters + lr * kRow3 + g * (kFilter3 / 2) + i * 16);
#pragma unroll
                for (int d = 0; d < 4; ++d) h[i * 4 + d] = v[d];
            }
            StaticFor<0, 9>([&](auto tap) {
                constexpr int t = decltype(tap)::value;
                Bytes16 wf;
                StaticFor<0, 4>([&](auto pair_of_channels) {
                    constexpr int d = decltype(pair_of_channels)::value, lo = 18 * d + t, hi = lo + 9;
                    wf[d] = PickHalves<(lo & 1) != 0, (hi & 1) != 0>(h[lo / 2], h[hi / 2]);
                });
                Bytes16 xf = *reinterpret_cast<const Bytes16*>(patch + (lin + (t / 3 - 1) * p.W + t % 3 - 1) * kPixel3 + g * 16);
                const unsigned keep = (inside >> t) & 1 ? ~0u : 0u;
#pragma unroll
                for (int d = 0; d < 4; ++d) xf[d] &= keep;
                MfmaTile<half_t>(wf, xf, acc);
            });
            __builtin_amdgcn_wave_barrier();
        }
    }
    __syncthreads();  // the staging areas become the sums
    // lane holds pixel lr, channels 8 * (v / 4) + 4 * g + v % 4
    float* const part = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int v = 0; v < 16; ++v) part[wave * kTilePart + (8 * (v / 4) + 4 * g + v % 4) * 33 + lr] = acc[v];
    __syncthreads();
    for (int e = tid; e < 32 * 32; e += 64 * args.nw) {
        const int row = e >> 5, col = e & 31;
        const int n = n0 + row, px = px0 + col;
        if (n >= p.K || px >= p.P) continue;
        float v = 0.f;
        for (int w = 0; w < args.nw; ++w) v += part[w * kTilePart + row * 33 + col];
        if (p.bias != nullptr) v += static_cast<float>(p.bias[n * p.bias_stride]);
        if (p.bn_gamma != nullptr) {  // as NchwConvKernel: the reference's association order, in float
            const float mean = static_cast<float>(p.bn_mean[n * p.bn_stride]);
            const float inv = 1.0f / sqrtf(static_cast<float>(p.bn_var[n * p.bn_stride]) + p.bn_eps);
            v = ((v - mean) * inv) * static_cast<float>(p.bn_gamma[n * p.bn_stride]) + static_cast<float>(p.bn_beta[n * p.bn_stride]);
        }
        const int64_t o = (static_cast<int64_t>(img) * p.K + n) * p.P + px;
        if (p.residual == nullptr) {
            if (p.relu) v = v < 0.f ? 0.f : v;  // NaN < 0 is false: NaN passes, like IfLessElse(x, 0, 0, x)
            p.out[o] = static_cast<half_t>(v);
        } else {
            float t = static_cast<float>(static_cast<half_t>(v)) + static_cast<float>(p.residual[o]);
            if (p.relu) t = t < 0.f ? 0.f : t;
            p.out[o] = static_cast<half_t>(t);
        }
    }
}

// Pairs of pixels in the rows that 32 consecutive pixels touch, at most, and the ones above and below, from an even pixel on.
int PatchPairs(const NchwConvArgs& a) { return ((std::min((32 + a.W - 2) / a.W + 1, a.H) + 2) * a.W + 2) / 2; }

// The waves of a workgroup: as many as there are chunks and LDS allows.
SmallConvArgs Plan(const NchwConvArgs& a, int taps) {
    SmallConvArgs p{};
    p.c = a;
    p.tiles_px = (a.P + 31) / 32;
    int chunks;
    if (taps == 1) {
        chunks = a.C / 32;
        p.wave_lds = 2 * 32 * kRow1;
    } else {
        chunks = a.C / 16;
        p.pairs = PatchPairs(a);
        p.wave_lds = 32 * kRow3 + (p.pairs * 2 + 2) * kPixel3;
    }
    p.nw = std::min({MaxWaves(taps), chunks, 160 * 1024 / p.wave_lds});
    const int per_wave = (chunks + p.nw - 1) / p.nw;
    p.nw = (chunks + per_wave - 1) / per_wave;
    return p;
}

}  // namespace

// Workgroups of SmallConv (its time is what a compute unit gets of them, times the reduction) against large tiles (which walk the reduction once at any
// batch this small): up to 1.5 + C / 300 to a compute unit for 3x3 filters, 1.6 for strides above 1, 2 for odd planes, 2 + 110 / C else.  us, large tiles
// and this kernel, around the lines: 3x3 64 channels at 56^2 392 workgroups 14.4 and 8.5, 784 14.5 and 15.2; 256 at 14^2 448 23.4 and 17.3, 672 23.8 and
// 24.9; 512 at 7^2 768 51 and 33; 1x1 1024 -> 256 at 14^2 448 14.2 and 10.1, 672 14.2 and 16.4; 64 -> 64 at 56^2 784 5.1 and 4.8, 1568 5.3 and 5.8;
// (for 3x3 the first figure is what NchwConvKernel takes; beyond one workgroup to a compute unit MidConvKernel is faster than both, us, this kernel and that:
// 512 channels at 7^2 256 12.8 and 18.1, 384 22.0 and 18.7; 256 at 14^2 224 10.0 and 13.0, 336 17.4 and 13.2; 128 at 28^2 200 7.9 and 10.4, 400 13.7 and
// 10.5; 64 at 56^2 392 8.9 and 9.7.)  1x1 2048 -> 512 at 7^2 512 33.5 and 23.8, 768 33.6 and 37.5; stride 2, 256 -> 512 at 56^2 400 7.5 and 5.9, 512 -> 256 at 28^2 448 10.7 and 13.9.
bool SmallConvTakes(const NchwConvArgs& a, int taps) {
    const double groups = static_cast<double>((a.P + 31) / 32) * a.N * ((a.K + 31) / 32) / NumCUs();
    if (taps == 9) {
        if (MidConvTakes(a, taps) && groups > (a.C < 128 ? 1.6 : 1.0)) return false;
        return groups <= 1.5 + a.C / 300.0 && PatchPairs(a) * 2 <= 4 * 64 && a.H * a.W >= 2;  // the patch of a tile is loaded in four passes at most
    }
    return groups <= (a.stride > 1 ? 1.6 : (a.P % 2 != 0 ? 2.0 : 2.0 + 110.0 / a.C));
}

void SmallConv(const NchwConvArgs& a, int taps, hipStream_t stream) {
    const SmallConvArgs p = Plan(a, taps);
    const int64_t grid = static_cast<int64_t>(p.tiles_px) * a.N * ((a.K + 31) / 32);
    HIPCX_REQUIRE(grid < (1LL << 22), HIPCX_NOT_IMPLEMENTED_ERROR, "problem too large for one launch");
    const int bytes = std::max<int>(p.nw * p.wave_lds, p.nw * kTilePart * sizeof(float));
    auto launch = [&](auto taps_tag, auto strided) {
        constexpr int T = decltype(taps_tag)::value;
        constexpr bool S = decltype(strided)::value;
        struct SmallConvTag {};
        EnsureDynamicLds<SmallConvTag>(reinterpret_cast<const void*>(SmallConvKernel<T, S>), bytes);
        hipLaunchKernelGGL((SmallConvKernel<T, S>), dim3(static_cast<unsigned>(grid)), dim3(64 * p.nw), bytes, stream, p);
    };
    if (taps == 9) launch(std::integral_constant<int, 9>{}, std::false_type{});
    else if (a.stride == 1 && a.P % 2 == 0) launch(std::integral_constant<int, 1>{}, std::false_type{});
    else launch(std::integral_constant<int, 1>{}, std::true_type{});
    CheckLaunch("small_conv");
}

}  // namespace hipcx
