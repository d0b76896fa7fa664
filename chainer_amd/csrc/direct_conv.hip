// float32 3x3 convolutions (stride 1, padding 1) of dense NCHW arrays with few enough output tiles that the chip waits for single ones.
//
// On the general kernel such a layer is a copy of x to channels-last, a copy of the filters, and 64 x 64 tiles of one wave each, on a fraction of the compute
// units, whose chunks of the reduction follow one another (1.3 us for 16 terms).  Here a wave owns 32 filters x 32 pixels, several waves share a tile's channels,
// and both operands are read as they lie: a lane's nine neighbours are dwords of the plane, 32 pixels in a row to an instruction, masked by their offsets,
// which are computed once (the channel is a scalar offset); the filters of eight channels, 288 bytes in a row, go through LDS, rows of 74 floats so that the
// 32 rows lie in the even banks and the next channel's terms in the odd ones.  A chunk of eight channels is in flight while the one before is multiplied:
// 36 v_mfma_f32_32x32x2_f32.  Sums of 36 terms are added up separately, which keeps the error of long sums below the split operands': 2-norm against 64 bits
// for 576, 1152 and 2304 terms 1.21e-7 to 1.24e-7, 1.23e-7 to 1.26e-7 and 1.29e-7 to 1.34e-7 (there 1.31e-7 to 1.33e-7, 1.85e-7 to 1.9e-7 and 2.7e-7), for 8, 24, 40 and
// 56 channels, which have no split operands there, 1.1e-7 to 1.2e-7 (1.5e-7 to 3.9e-7).  At 16, 32 and 48 channels the split operands are ahead of such sums, 6.7e-8,
// 9.3e-8 and 1.15e-7 against 1.13e-7 to 1.21e-7: chains of at most 10 terms, or of 18, are added up in double there, 6.2e-8, 8.1e-8 and 8.1e-8.
// Bound by the float pipe from a few hundred tiles on (0.74 of it at 4096), before by the latency of a wave's share.  us, general kernel with its copies and
// this one, 64 -> 64 at 32^2, 128 -> 128 at 16^2 and 256 -> 256 at 8^2: one image 53, 93, 174 and 6.7, 10.7, 16.0; 16 images 50, 95, 176 and 17.9, 17.2, 18.5; 64
// images 70, 79, 181 and 55, 56, 62.
#include "direct_conv.h"

#include <algorithm>
#include <cstdlib>

#include "igemm.h"
#include "launch_profile.h"
#include "nchw_conv.h"
#include "small_dot.h"

namespace hipcx {
namespace {

constexpr int kOut = 0x7fffffff;  // an offset beyond any buffer: loads give zeros, stores are dropped
constexpr int kTaps = 9;
constexpr int kChunk = 8;                   // channels
constexpr int kTerms = kChunk * kTaps;      // floats of a filter's chunk
constexpr int kPitch = kTerms + 2;          // in LDS
constexpr int kPieces = kTerms / 4;

struct DirectConvArgs {
    const float* x;
    const float* w;
    const float* bias;
    int64_t bias_stride;
    float* out;
    int C, K, W, P;  // P: pixels of a plane
    int M;           // images * P
    int tiles_f, tiles_p;
    int64_t x_bytes, out_bytes;
    unsigned w_bytes;
    FastDiv div_P, div_W;
};

// PW waves of a workgroup take 32 pixels each, with the same 32 filters; KS such groups share the channels.  CHAIN > 0: chains of that many taps of two
// channels, and of the rest of the nine, added up in double.
template <int PW, int KS, int CHAIN>
__global__ __launch_bounds__(64 * PW * KS) __attribute__((amdgpu_waves_per_eu(2))) void DirectConvKernel(DirectConvArgs p) {
    constexpr int kGroup = 64 * PW;  // threads that share filters
    constexpr int kStagePieces = 32 * kPieces;
    constexpr int SP = (kStagePieces + kGroup - 1) / kGroup;
    constexpr int kStage = 32 * kPitch;  // floats
    constexpr int kPairs = kChunk / 2;
    extern __shared__ __align__(16) float lds[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int pw = wave % PW, ks = wave / PW;
    const int r = lane & 31, g = lane >> 5;
    int tf, tp;
    SmallDotTile(p.tiles_f * p.tiles_p, blockIdx.x, p.tiles_f, tf, tp);
    const int n0 = tf * 32, m0 = tp * 32 * PW;
    const int img0 = p.div_P(m0);
    const int plane = p.P * 4;
    const int64_t skip_x = static_cast<int64_t>(img0) * p.C * plane, skip_out = static_cast<int64_t>(img0) * p.K * plane;
    auto rsrc = [](const float* base, int64_t skip, int64_t bytes) {
        return MakeRsrc(reinterpret_cast<const char*>(base) + skip, static_cast<unsigned>(min(bytes - skip, int64_t{0x7ffffffc})));
    };
    const __amdgpu_buffer_rsrc_t xr = rsrc(p.x, skip_x, p.x_bytes), outr = rsrc(p.out, skip_out, p.out_bytes), wr = MakeRsrc(p.w, p.w_bytes);

    // where this lane's pixel and its neighbours lie in the plane of channel g, and where its results go
    const int m = m0 + pw * 32 + r;
    const bool in = m < p.M;
    const int img = p.div_P(in ? m : m0), px = (in ? m : m0) - img * p.P;
    const int x = px - p.div_W(px) * p.W;
    int xoff[kTaps];
#pragma unroll
    for (int k = 0; k < kTaps; ++k) {
        const int dy = k / 3 - 1, dx = k % 3 - 1;
        const bool ok = in & (static_cast<unsigned>(x + dx) < static_cast<unsigned>(p.W)) & (static_cast<unsigned>(px + dy * p.W) < static_cast<unsigned>(p.P));
        xoff[k] = ok ? (img - img0) * p.C * plane + g * plane + (px + dy * p.W + dx) * 4 : kOut;
    }
    const int to = in ? (img - img0) * p.K * plane + (n0 + 4 * g) * plane + px * 4 : kOut;
    // the pieces of 16 bytes of a chunk of filters that this thread stages
    int woff[SP], wto[SP];
#pragma unroll
    for (int i = 0; i < SP; ++i) {
        const int q = pw * 64 + lane + i * kGroup, row = q / kPieces, col = q - row * kPieces;
        woff[i] = q < kStagePieces && n0 + row < p.K ? ((n0 + row) * p.C * kTaps + col * 4) * 4 : kOut;
        wto[i] = row * kPitch + col * 4;
    }
    float* const mine = lds + ks * 2 * kStage;
    const int frag = r * kPitch + g * kTaps;

    Bytes16 wreg[SP];
    float b[kPairs][kTaps];
    auto load_w = [&](int c) {
#pragma unroll
        for (int i = 0; i < SP; ++i) wreg[i] = __builtin_amdgcn_raw_buffer_load_b128(wr, woff[i], c * kTaps * 4, 0);
    };
    auto store_w = [&](int stage) {
#pragma unroll
        for (int i = 0; i < SP; ++i) {
            if ((i + 1) * kGroup <= kStagePieces || pw * 64 + lane + i * kGroup < kStagePieces) {
                Bytes8* const at = reinterpret_cast<Bytes8*>(mine + stage * kStage + wto[i]);
                at[0] = Bytes8{wreg[i].x, wreg[i].y};
                at[1] = Bytes8{wreg[i].z, wreg[i].w};
            }
        }
    };
    auto load_x = [&](int pair, int c) {
#pragma unroll
        for (int k = 0; k < kTaps; ++k) b[pair][k] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(xr, xoff[k], c * plane, 0));
    };
    auto sync = [&] {
        if constexpr (PW > 1) __syncthreads();
        else __builtin_amdgcn_wave_barrier();  // (filters of its own)
    };

    constexpr bool DOUBLE = CHAIN > 0;
    using Sum = std::conditional_t<DOUBLE, double, float>;
    using Sum16 = __attribute__((ext_vector_type(16))) Sum;
    Sum16 sum = {};
    float16_t acc[DOUBLE ? 2 : 1] = {};  // two chains in turn: one is added up while the other grows
    auto add_up = [&](int chain) {
#pragma unroll
        for (int v = 0; v < 16; ++v) sum[v] += static_cast<Sum>(acc[chain][v]);
    };
    const int chunks = p.C / kChunk, rounds = (chunks + KS - 1) / KS, own = (chunks - ks + KS - 1) / KS;
    auto multiply = [&](int i, auto next_tag) {
        const int c = (ks + i * KS) * kChunk;
        const float* const from = mine + (i & 1) * kStage + frag;
#pragma unroll
        for (int j = 0; j < kPairs; ++j) {
#pragma unroll
            for (int k = 0; k < kTaps; ++k) {
                const float16_t zero = {};
                const int chain = DOUBLE ? (CHAIN < kTaps ? k >= CHAIN : j % 2) : 0;
                const bool first = DOUBLE ? k == 0 || k == CHAIN : j % 2 == 0 && k == 0;
                acc[chain] = __builtin_amdgcn_mfma_f32_32x32x2f32(from[j * 2 * kTaps + k], b[j][k], first ? zero : acc[chain], 0, 0, 0);
                if (DOUBLE && first) add_up(1 - chain);
            }
            if constexpr (decltype(next_tag)::value) load_x(j, c + KS * kChunk + 2 * j);
            if (!DOUBLE && j % 2 == 1) add_up(0);
        }
    };
    if (own > 0) {
        load_w(ks * kChunk);
#pragma unroll
        for (int j = 0; j < kPairs; ++j) load_x(j, ks * kChunk + 2 * j);
        store_w(0);
        if (own > 1) load_w((ks + KS) * kChunk);
    }
    sync();
    for (int i = 0; i < rounds; ++i) {
        if (i + 1 < own) {
            store_w((i + 1) & 1);  // the stage that the round before read
            load_w((ks + min(i + 2, own - 1) * KS) * kChunk);
            multiply(i, std::true_type{});
        } else if (i < own) {
            multiply(i, std::false_type{});
        }
        sync();
    }

    // lane holds pixel r, filters 8 * (v / 4) + 4 * g + v % 4; each wave adds up its share of them
    if (DOUBLE) add_up(1);
    constexpr int kShare = 16 / KS;
    __syncthreads();  // the staging areas become partial sums
    Sum* const parts = reinterpret_cast<Sum*>(lds);
#pragma unroll
    for (int v = 0; v < 16; ++v) parts[(wave * 16 + v) * 64 + lane] = sum[v];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kShare; ++i) {
        const int v = ks * kShare + i, row = 8 * (v / 4) + v % 4, n = n0 + row + 4 * g;
        Sum total = 0;
#pragma unroll
        for (int k = 0; k < KS; ++k) total += parts[((k * PW + pw) * 16 + v) * 64 + lane];
        float s = static_cast<float>(total);
        if (p.bias != nullptr) s += n < p.K ? p.bias[n * p.bias_stride] : 0.f;
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(s), outr, (in & (n < p.K)) ? to + row * plane : kOut, 0, 0);
    }
}

template <int PW, int KS, int CHAIN>
void Launch(DirectConvArgs p, hipStream_t stream) {
    constexpr int kLds = std::max(KS * 2 * 32 * kPitch * 4, KS * PW * 16 * 64 * (CHAIN > 0 ? 8 : 4));
    p.tiles_f = (p.K + 31) / 32, p.tiles_p = (p.M + 32 * PW - 1) / (32 * PW);
    struct DirectConvTag {};
    EnsureDynamicLds<DirectConvTag>(reinterpret_cast<const void*>(DirectConvKernel<PW, KS, CHAIN>), kLds);
    hipLaunchKernelGGL((DirectConvKernel<PW, KS, CHAIN>), dim3(static_cast<unsigned>(p.tiles_f) * p.tiles_p), dim3(64 * PW * KS), kLds, stream, p);
    CheckLaunch("direct_conv");
}

// Where the split operands of the general kernel, which takes whole groups of 16 channels, have less error than chains of 36 terms.
bool SumsInDouble(int64_t channels) { return channels % 16 == 0 && channels < 64; }

int64_t Tiles(int64_t pixels, int64_t filters) { return ((pixels + 31) / 32) * ((filters + 31) / 32); }

}  // namespace

bool DirectConvTakes(const hipcx_array* x, const hipcx_array* w, const int64_t* stride, const int64_t* pad, const hipcx_array* out) {
    static const bool enabled = [] { const char* e = getenv("HIPCX_CONV_DIRECT"); return e == nullptr || e[0] != '0'; }();
    if (!enabled || out->dtype != HIPCX_FLOAT32 || !IsContiguous(x) || !IsContiguous(out)) return false;
    const int64_t N = x->shape[0], C = x->shape[1], P = x->shape[2] * x->shape[3], K = w->shape[0];
    // Beyond, the large tiles of the split operands (igemm_split.hip) catch up, copies of x and w included.  us there and here: 64 -> 64 at 32^2, 96 images 87 and 80,
    // 128 images (8192 tiles) 96 and 105; 128 -> 128 at 16^2, 96 images (3072) 88 and 82, 112 images 94 and 101; 256 -> 256 at 8^2, 160 images (2560) 145 and
    // 145, 200 images 152 and 185.
    // Half to two thirds of that where sums are in double, whose additions bound the kernel: 64 filters, 12 and 16 tiles to a compute unit, 16 channels 25.8 and 23.0,
    // 27.7 and 29.6, 32 channels 35.5 and 30.0, 40.6 and 38.7; 128 filters, 8 and 12, 21.8 and 17.0, 23.3 and 24.4, 48 channels 36.2 and 27.7, 38.3 and 39.5.
    const int most = SumsInDouble(C) ? (K <= 64 ? 12 : 8) : (K <= 64 ? 24 : 12);
    if (Tiles(N * P, K) > most * NumCUs()) return false;
    if (w->shape[2] != 3 || w->shape[3] != 3 || stride[0] != 1 || stride[1] != 1 || pad[0] != 1 || pad[1] != 1) return false;
    if (out->shape[2] != x->shape[2] || out->shape[3] != x->shape[3] || C % kChunk != 0 || C == 0) return false;
    // 32-bit offsets from a tile's first image
    const double limit = 2147483000.0 / 4, images = 256.0 / P + 3;
    return images * C * P < limit && images * (K + 64) * P < limit && static_cast<double>(K + 64) * C * kTaps < limit && static_cast<double>(N) * P < 2147483000.0;
}

void DirectConv(const hipcx_array* x, const hipcx_array* w, const hipcx_array* b, const hipcx_array* out, hipStream_t stream) {
    const int64_t N = x->shape[0], C = x->shape[1], P = x->shape[2] * x->shape[3], K = w->shape[0];
    DirectConvArgs p{};
    p.x = static_cast<const float*>(x->data), p.w = static_cast<const float*>(w->data), p.out = static_cast<float*>(out->data);
    p.bias = b != nullptr ? static_cast<const float*>(b->data) : nullptr;
    p.bias_stride = b != nullptr ? b->strides[0] / 4 : 0;
    p.C = static_cast<int>(C), p.K = static_cast<int>(K), p.W = static_cast<int>(x->shape[3]), p.P = static_cast<int>(P), p.M = static_cast<int>(N * P);
    p.x_bytes = N * C * P * 4, p.out_bytes = N * K * P * 4, p.w_bytes = static_cast<unsigned>(K * C * kTaps * 4);
    p.div_P = FastDiv(p.P), p.div_W = FastDiv(p.W);
    ProfileScope prof(stream, 2.0 * p.M * K * C * kTaps, 4.0 * (static_cast<double>(N) * C * P + static_cast<double>(K) * C * kTaps + static_cast<double>(p.M) * K));
    // The widest split of the channels while tiles leave compute units without a workgroup.  us, (PW, KS) = (1, 8), (2, 4) and (4, 2): 64 -> 64 at 32^2, 4
    // images (256 tiles) 7.4 10.3 16.2, 6 images 12.2 10.7 16.5, 12 images 18.1 19.2 17.4, 64 images 84 73 55; 256 -> 256 at 8^2, 16 images (256 tiles)
    // 18.5 26.9 57, 48 images 50 53 61, 80 images 81 78 96, 128 images 128 105 104.
    const int64_t tiles = Tiles(p.M, K), cus = NumCUs();
    auto run = [&](auto taps) {
        constexpr int CHAIN = decltype(taps)::value;
        if (tiles <= cus) Launch<1, 8, CHAIN>(p, stream);
        else if (tiles <= (C >= 128 ? 6 : 2) * cus) Launch<2, 4, CHAIN>(p, stream);
        else Launch<4, 2, CHAIN>(p, stream);
    };
    if (!SumsInDouble(C)) run(std::integral_constant<int, 0>{});
    else if (C == 16) run(std::integral_constant<int, 5>{});
    else run(std::integral_constant<int, kTaps>{});
}

}  // namespace hipcx
