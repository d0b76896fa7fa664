// float16 3x3 convolutions (stride 1, padding 1) of a few hundred output tiles: a handful of images in a network's deep layers.
//
// Such a layer has more work than SmallConvKernel's 32 x 32 tiles deliver operands for, and too few of NchwConvKernel's 256 x 64 tiles to occupy the chip (512 channels
// at 7^2, 32 images: 56 workgroups).  Here a workgroup owns 64 filters x 64 output positions and its four or eight waves share the channels, sixteen at a time.  The
// filters come packed, so that a wave's operands are whole lines straight from memory, one chunk ahead, tap by tap; the chunk's pixels, pairs of eight channel
// planes turned round in registers, lie in LDS that belongs to the wave, and its nine taps are reads at addresses computed once: no barrier before the sums,
// which meet in LDS.  Images follow one another without regard to tiles, planes of an odd size with a position that is none.  Bound by latency while tiles
// are few, then by what the waves read through L2 (9.4 TB/s of operands at 1568 tiles of 256 channels).  us with the filters' packing, before (the faster of the two
// kernels above) and now: 512 channels at 7^2, 12 images 22.0 -> 18.7, 32 images 54 -> 20.4, 64 images 55 -> 32.4; 256 at 14^2, 6 images 17.4 -> 13.2, 32
// images 25.5 -> 19.4; 128 at 28^2, 4 images 13.7 -> 10.5, 16 images 16.8 -> 14.2; 64 at 56^2, 4 images 14.8 -> 10.1.
#include <algorithm>

#include "mid_conv.h"
#include "pixel_pairs.h"
#include "small_dot.h"

namespace hipcx {
namespace {

constexpr int kOut = 0x7fffffff;  // an offset beyond any buffer: zeros
constexpr int kTile = 64;         // filters and positions of a workgroup
constexpr int kSumPitch = kTile + 8;
constexpr int kChunk = 16;        // channels
constexpr int kPixel = 2 * kChunk;

struct MidConvArgs {
    NchwConvArgs c;
    int plane;     // positions of an image: its pixels, and one more if they are odd
    int M;         // images * plane
    FastDiv div_plane;
    int pairs;     // of positions in a patch
    int wave_lds;  // bytes
};

// NP: passes of a wave over its patch.
template <int NP, int KS>
__global__ __launch_bounds__(64 * KS) __attribute__((amdgpu_waves_per_eu(2))) void MidConvKernel(MidConvArgs args) {
    const NchwConvArgs& p = args.c;
    extern __shared__ __align__(16) char lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int ks = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 31, g = lane >> 5;
    int tile_px, tile_n;
    SmallDotTile(gridDim.x, blockIdx.x, p.tiles_m, tile_px, tile_n);
    const int m0 = tile_px * kTile, n0 = tile_n * kTile;
    const __amdgpu_buffer_rsrc_t xr = MakeRsrc(p.x, p.x_bytes), wr = MakeRsrc(p.wp, p.wp_bytes);
    char* const mine = lds + ks * args.wave_lds;

    // lane i holds what is added to and multiplied with row i of this wave's share of the results
    constexpr int kRows = kTile / KS;
    float bias = 0.f, mean = 0.f, var = 0.f, gamma = 0.f, beta = 0.f;
    {
        const int n = min(n0 + ks * kRows + lane % kRows, p.K - 1);
        if (p.bias != nullptr) bias = static_cast<float>(p.bias[n * p.bias_stride]);
        if (p.bn_gamma != nullptr) {
            mean = static_cast<float>(p.bn_mean[n * p.bn_stride]);
            var = static_cast<float>(p.bn_var[n * p.bn_stride]);
            gamma = static_cast<float>(p.bn_gamma[n * p.bn_stride]);
            beta = static_cast<float>(p.bn_beta[n * p.bn_stride]);
        }
    }
    // the filters' groups of 8 channels that this lane multiplies
    int a_off[2];
#pragma unroll
    for (int f = 0; f < 2; ++f) {
        const int n = n0 + f * 32 + lr;
        a_off[f] = n < p.K ? (g * 9 * p.K + n) * 16 : kOut;
    }
    // The patch: positions of the images one behind another, from a row and a pixel before the tile's first on, from an even one on.  Neighbours that lie in
    // another row's end, another image or nowhere are never asked for: where a tap leaves the plane, a pixel of zeros is read.  A pair's second position may be
    // none; the last pixel of an odd plane is loaded with the one before (`shift`), so that nothing beyond the array is.
    const int pairs = args.pairs, first = (m0 - p.W - 1) & ~1, zeros = pairs * 2 * kPixel;
    int x_off[NP], x_to[NP], shift[NP];
#pragma unroll
    for (int s = 0; s < NP; ++s) {
        const int item = s * 64 + lane, group = item >= pairs ? 1 : 0, pr = item - group * pairs, q = first + 2 * pr;
        const bool in = (item < pairs * 2) & (q >= 0) & (q < args.M);
        const int img = args.div_plane(in ? q : 0), px = (in ? q : 0) - img * args.plane;
        const bool alone = px + 1 == p.P;
        x_off[s] = in ? ((img * p.C + group * 8) * p.P + px - alone) * 2 : kOut;
        shift[s] = alone ? 16 : 0;
        x_to[s] = item < pairs * 2 ? pr * 2 * kPixel + group * 16 : -1;
    }
    int at[9][2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int m = m0 + t * 32 + lr;
        const int px = m - args.div_plane(m) * args.plane, y = p.div_W(px), x = px - y * p.W;
        const bool in = (m < args.M) & (px < p.P);
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            const int dy = k / 3 - 1, dx = k % 3 - 1;
            const bool ok = in & (static_cast<unsigned>(y + dy) < static_cast<unsigned>(p.H)) & (static_cast<unsigned>(x + dx) < static_cast<unsigned>(p.W));
            at[k][t] = (ok ? (m - first + dy * p.W + dx) * kPixel : zeros) + g * 16;
        }
    }
    if (lane < 2) *reinterpret_cast<Bytes16*>(mine + zeros + lane * 16) = Bytes16{0u, 0u, 0u, 0u};

    float16_t acc[2][2];
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[f][t][v] = 0.f;
    const int chunks = p.C / kChunk, per_wave = (chunks + KS - 1) / KS;
    const int begin = min(chunks, ks * per_wave), end = min(chunks, begin + per_wave);
    Bytes16 av[9][2];
    unsigned xv[NP][8];
    auto load_a = [&](int k, int c) {
#pragma unroll
        for (int f = 0; f < 2; ++f) {
            av[k][f] = __builtin_amdgcn_raw_buffer_load_b128(wr, a_off[f], (c * 18 + k) * p.K * 16, 0);
            __builtin_amdgcn_sched_barrier(0);  // (in this order before the loop as well: the waits inside count on both)
        }
    };
    auto load_x = [&](int c) {
#pragma unroll
        for (int s = 0; s < NP; ++s)
#pragma unroll
            for (int e = 0; e < 8; ++e) xv[s][e] = __builtin_amdgcn_raw_buffer_load_b32(xr, x_off[s], (c * kChunk + e) * p.P * 2, 0);
    };
    auto multiply = [&](int c, auto next_tag) {
        constexpr bool kNext = decltype(next_tag)::value;
#pragma unroll
        for (int s = 0; s < NP; ++s) {
#pragma unroll
            for (int e = 0; e < 8; ++e) xv[s][e] >>= shift[s];
            Bytes16 even, odd;
            TurnPairs(xv[s], even, odd);
            if (x_to[s] >= 0) {
                *reinterpret_cast<Bytes16*>(mine + x_to[s]) = even;
                *reinterpret_cast<Bytes16*>(mine + x_to[s] + kPixel) = odd;
            }
        }
        if constexpr (kNext) load_x(c + 1);
        __builtin_amdgcn_wave_barrier();
        Bytes16 xf[2][2];
        auto fetch = [&](int k) {
#pragma unroll
            for (int t = 0; t < 2; ++t) xf[k & 1][t] = *reinterpret_cast<const Bytes16*>(mine + at[k][t]);
        };
        fetch(0);
        // (left to itself the compiler loads all of the next chunk's filters at the end of this one, and waits for them at the beginning of that)
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            if (k + 1 < 9) fetch(k + 1);
#pragma unroll
            for (int f = 0; f < 2; ++f)
#pragma unroll
                for (int t = 0; t < 2; ++t) MfmaTile<half_t>(av[k][f], xf[k & 1][t], acc[f][t]);
            if constexpr (kNext) load_a(k, c + 1);
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_wave_barrier();
    };
    if (begin < end) {
        load_x(begin);
#pragma unroll
        for (int k = 0; k < 9; ++k) load_a(k, begin);
        for (int c = begin; c + 1 < end; ++c) multiply(c, std::true_type{});
        multiply(end - 1, std::false_type{});
    }
    __syncthreads();  // the patches become the sums
    // lane holds position lr, channels 8 * (v / 4) + 4 * g + v % 4 of each block
    float* const part = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int v = 0; v < 16; ++v) part[(ks * kTile + f * 32 + 8 * (v / 4) + 4 * g + v % 4) * kSumPitch + t * 32 + lr] = acc[f][t][v];
    __syncthreads();
    const int m = m0 + lane, img = args.div_plane(m), px = m - img * args.plane;
    const bool in = (m < args.M) & (px < p.P);
    const int64_t at_out = static_cast<int64_t>(img) * p.K * p.P + px;
    half_t residual[kRows];
    if (p.residual != nullptr) {
#pragma unroll
        for (int i = 0; i < kRows; ++i) {
            const int n = n0 + ks * kRows + i;
            residual[i] = in & (n < p.K) ? p.residual[at_out + static_cast<int64_t>(n) * p.P] : half_t{0};
        }
    }
    // (all of a wave's rows are read before the first is added up)
    float sum[kRows];
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
        float v[KS];
#pragma unroll
        for (int k = 0; k < KS; ++k) v[k] = part[(k * kTile + ks * kRows + i) * kSumPitch + lane];
        sum[i] = v[0];
#pragma unroll
        for (int k = 1; k < KS; ++k) sum[i] += v[k];
    }
    const float inv = 1.0f / sqrtf(var + p.bn_eps);
    auto of_row = [](float v, int i) { return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), i)); };
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
        const int n = n0 + ks * kRows + i;
        if (n >= p.K) break;
        float v = sum[i];
        if (p.bias != nullptr) v += of_row(bias, i);
        // as NchwConvKernel: the reference's association order, in float
        if (p.bn_gamma != nullptr) v = ((v - of_row(mean, i)) * of_row(inv, i)) * of_row(gamma, i) + of_row(beta, i);
        if (p.residual != nullptr) v = static_cast<float>(static_cast<half_t>(v)) + static_cast<float>(residual[i]);
        if (p.relu) v = v < 0.f ? 0.f : v;  // NaN < 0 is false: NaN passes, like IfLessElse(x, 0, 0, x)
        if (in) p.out[at_out + static_cast<int64_t>(n) * p.P] = static_cast<half_t>(v);
    }
}

// Pairs of pixels that the taps of 64 consecutive ones reach, from an even one on.
int PatchPairs(const NchwConvArgs& a) { return (kTile + 2 * a.W + 4) / 2; }

template <int NP, int KS>
void Launch(const MidConvArgs& p, hipStream_t stream) {
    const int64_t grid = static_cast<int64_t>(p.c.tiles_m) * p.c.tiles_n;
    const int bytes = std::max<int>(KS * p.wave_lds, KS * kTile * kSumPitch * sizeof(float));
    struct MidConvTag {};
    EnsureDynamicLds<MidConvTag>(reinterpret_cast<const void*>(MidConvKernel<NP, KS>), bytes);
    hipLaunchKernelGGL((MidConvKernel<NP, KS>), dim3(static_cast<unsigned>(grid)), dim3(64 * KS), bytes, stream, p);
    CheckLaunch("mid_conv");
}

}  // namespace

namespace {
int64_t Positions(const NchwConvArgs& a) { return static_cast<int64_t>(a.N) * ((a.P + 1) / 2 * 2); }
int64_t Tiles(const NchwConvArgs& a) { return (Positions(a) + kTile - 1) / kTile * ((a.K + kTile - 1) / kTile); }
}  // namespace

// Up to two tiles to a compute unit, three for long reductions; beyond, what the tiles read through L2 takes longer than NchwConvKernel's larger ones.  us, that
// kernel and this, filters packed: 512 channels at 7^2 200 tiles 51 and 20.4, 600 53.7 and 43.2, 800 54.9 and 53.8; 256 at 14^2 392 24.5 and 19.4, 588 25.7
// and 26.1; 128 at 28^2 392 16.4 and 14.2, 588 17.3 and 19.0; 64 at 56^2 392 15.0 and 12.0, 588 15.5 and 16.4.
bool MidConvTakes(const NchwConvArgs& a, int taps) {
    if (taps != 9 || PatchPairs(a) * 2 > 3 * 64 || a.P < 2 || Positions(a) >= (1LL << 30)) return false;
    return Tiles(a) <= (a.C > 256 ? 3 : 2) * NumCUs();
}

void MidConv(const NchwConvArgs& a, hipStream_t stream) {
    MidConvArgs p{};
    p.c = a;
    p.plane = (a.P + 1) / 2 * 2;
    p.M = a.N * p.plane;
    p.div_plane = FastDiv(p.plane);
    p.pairs = PatchPairs(a);
    p.wave_lds = (p.pairs * 2 + 1) * kPixel;
    p.c.tiles_m = (p.M + kTile - 1) / kTile;
    p.c.tiles_n = (a.K + kTile - 1) / kTile;
    // eight waves to a tile while it has a compute unit to itself, else two tiles of four waves to each: 512 channels at 7^2 200 tiles 20.4 us and 20.8, 400 tiles
    // 35.8 and 32.4; 256 at 14^2 392 tiles 22.7 and 19.4
    const bool two = p.pairs * 2 <= 2 * 64;
    if (Tiles(a) <= NumCUs()) two ? Launch<2, 8>(p, stream) : Launch<3, 8>(p, stream);
    else two ? Launch<2, 4>(p, stream) : Launch<3, 4>(p, stream);
}

}  // namespace hipcx
