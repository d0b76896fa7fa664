// out[m][n] = sum over b < batch, k < depth of a[b][m][k] * bt[b][n][k] in float16: the weight gradients of convolutions, whose outputs are a few
// 128 x 128 tiles and whose reduction is every pixel of every image.
//
// The reduction is cut into chunks of 32 k of an image and split over `slices` workgroups per tile, whose float sums BatchedSumKernel adds up.
// Operands come from far away (a tile's rows are read once) and a slice is a few dozen chunks, so what counts is loads in flight: they go to LDS
// directly, three chunks ahead in a ring of four (64 KiB; two workgroups to a compute unit), and one barrier a
// chunk hands a stage over.  LDS layout, swizzle and counted waits as in gemm_pp.h.  An image's last chunk is masked in registers, in both operands: what
// follows a row may be Inf or NaN.  ResNet-50's 20 shapes of
// filters, us of the whole call, against 128 x 128 tiles two stages deep that read rows of 16 bytes only (odd planes and 14 x 14 ones came as
// copies): 567 -> 420 at batch 8, 1026 -> 738 at batch 32; 1x1 of 1024 channels on 14 x 14 at 32: 47 -> 22; 3x3 of 512 on 7 x 7: 102 -> 56.
#include <algorithm>

#include "batched_product.h"
#include "igemm.h"
#include "launch_profile.h"
#include "lds_load.h"

namespace hipcx {
namespace {

constexpr int kRing = 4;
constexpr int kTileBytes = 128 * 64;  // of one operand in a stage
constexpr int kStageBytes = 2 * kTileBytes;
constexpr int kOutRow = 64 * 4 + 16;  // bytes of a wave's row of sums on its way out
static_assert(4 * 32 * kOutRow <= kRing * kStageBytes, "the four waves' blocks fit the ring");

struct ProductArgs {
    BatchedOperands o;
    float* partial;  // [slices][M][N]
    int slices, chunks_per_image;
    int tiles_n;
    unsigned a_bytes, b_bytes;
};

__global__ __launch_bounds__(256) void BatchedProductKernel(ProductArgs p) {
    constexpr int LPO = 2, LPC = 2 * LPO;  // load instructions per operand / chunk and wave
    constexpr int kOut = 0x7fffffff;
    extern __shared__ __align__(16) char lds[];
    // the slices of a tile are neighbours: workgroup ids go round-robin to the XCDs, so that (with a multiple of eight slices) the tiles of a slice,
    // which read the same chunks, share an L2
    const int tile = blockIdx.x / p.slices, slice = blockIdx.x - tile * p.slices;
    const int tile_m = tile / p.tiles_n, tile_n = tile - tile_m * p.tiles_n;
    const int m0 = tile_m * 128, n0 = tile_n * 128;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave & 1, wn = wave >> 1;
    const int r = lane & 31, h = lane >> 5;
    const BatchedOperands& o = p.o;

    const auto ra = RawRsrc(o.a, p.a_bytes), rb = RawRsrc(o.b, p.b_bytes);
    int voa[LPO], vob[LPO];
#pragma unroll
    for (int i = 0; i < LPO; ++i) {
        const int row = (wave * LPO + i) * 16 + (lane >> 2);
        const int piece = (lane & 3) ^ ((lane >> 4) & 3);  // (row >> 2) & 3 = (lane >> 4) & 3
        const int m = m0 + row, n = n0 + row;
        int64_t b_row = static_cast<int64_t>(n) * o.b_row;
        if (o.taps_s > 0) {
            const int taps = o.taps_r * o.taps_s, c = n / taps, t = n - c * taps, tr = t / o.taps_s;
            const int ts = t - tr * o.taps_s;
            b_row = c * o.b_row + tr * o.r_stride + (ts & 1) * o.s_stride + (ts >> 1) * o.s_pair_stride;
        }
        voa[i] = m < o.M ? static_cast<int>(m * o.a_row * 2) + piece * 16 : kOut;
        vob[i] = n < o.N ? static_cast<int>(b_row * 2) + piece * 16 : kOut;
    }
    const int total = o.batch * p.chunks_per_image;
    const int begin = static_cast<int>(static_cast<int64_t>(total) * slice / p.slices), n = static_cast<int>(static_cast<int64_t>(total) * (slice + 1) / p.slices) - begin;

    const unsigned lds_base = static_cast<unsigned>(reinterpret_cast<uintptr_t>(lds));
    int issued = 0, image = begin / p.chunks_per_image, chunk = begin - image * p.chunks_per_image;  // of the next chunk to load
    auto issue = [&] {
        const unsigned st = lds_base + (issued % kRing) * kStageBytes + wave * LPO * 1024;
        const int so_a = static_cast<int>((image * o.a_slice + chunk * 32) * 2), so_b = static_cast<int>((image * o.b_slice + chunk * 32) * 2);
#pragma unroll
        for (int i = 0; i < LPO; ++i) LdsLoad16(ra, st + i * 1024, voa[i], so_a);
#pragma unroll
        for (int i = 0; i < LPO; ++i) LdsLoad16(rb, st + kTileBytes + i * 1024, vob[i], so_b);
        ++issued;
        const bool wrap = ++chunk == p.chunks_per_image;
        chunk = wrap ? 0 : chunk;
        image += wrap;
    };
    // 16-byte fragments: rows of a are the MFMA columns, rows of b its rows, so that a lane ends up with 4 consecutive n of one m
    int fa[2], fb[2];  // by half of the chunk
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int pos = (2 * t + h) ^ ((r >> 2) & 3);
        fa[t] = (wm * 64 + r) * 64 + pos * 16;
        fb[t] = kTileBytes + (wn * 64 + r) * 64 + pos * 16;
    }
    float16_t acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

    int at = begin % p.chunks_per_image;  // the current chunk's place in its image
    auto step = [&](int c, bool more) {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();  // every wave's share of chunk c has landed, and nobody reads the stage of chunk c - 1 any more
        asm volatile("" ::: "memory");
        if (more) issue();
        const char* const st = lds + (c % kRing) * kStageBytes;
        Bytes16 ma[2][2], mb[2][2];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                ma[t][i] = *reinterpret_cast<const Bytes16*>(st + fa[t] + i * 32 * 64);
                mb[t][i] = *reinterpret_cast<const Bytes16*>(st + fb[t] + i * 32 * 64);
            }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the reads are over before the next barrier
        const int valid = o.depth - at * 32;
        at = at + 1 == p.chunks_per_image ? 0 : at + 1;
        if (valid < 32) {
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    const int left = valid - (t * 16 + h * 8 + d * 2);
                    const unsigned mask = left >= 2 ? 0xffffffffu : (left == 1 ? 0xffffu : 0u);
#pragma unroll
                    for (int i = 0; i < 2; ++i) ma[t][i][d] &= mask, mb[t][i][d] &= mask;
                }
        }
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) MfmaTile<half_t>(mb[t][j], ma[t][i], acc[i][j]);
    };
    for (int c = 0; c < kRing - 1 && c < n; ++c) issue();
    int c = 0;
    for (; c + kRing - 1 < n; ++c) {
        WaitVmcnt<(kRing - 2) * LPC>();  // this wave's share of chunk c
        step(c, true);
    }
    for (; c < n; ++c) {
        WaitVmcnt<0>();
        step(c, false);
    }
    __syncthreads();  // the ring is free

    // lane holds m = r, n = 8 * (v / 4) + 4 * h + v % 4 of each 32 x 32 block; through LDS so that rows of 64 columns leave in whole lines
    char* const mine = lds + wave * 32 * kOutRow;
    auto store = [&](auto tag, auto* to, int64_t ld) {
        using T = decltype(tag);
        constexpr int E = 16 / static_cast<int>(sizeof(T)), LANES = 64 / E, ROWS = 64 / LANES;  // lanes of a row, rows of an instruction
        struct __attribute__((packed, aligned(2))) Piece {
            T e[E];
        };
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    T v[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = static_cast<T>(acc[i][j][q * 4 + e]);
                    __builtin_memcpy(mine + r * kOutRow + (j * 32 + q * 8 + h * 4) * sizeof(T), v, sizeof(v));
                }
            __builtin_amdgcn_wave_barrier();
            const int col = n0 + wn * 64 + (lane % LANES) * E;
#pragma unroll
            for (int s = 0; s < 32 / ROWS; ++s) {
                const int row = s * ROWS + lane / LANES, m = m0 + wm * 64 + i * 32 + row;
                Piece v;
                __builtin_memcpy(&v, mine + row * kOutRow + (lane % LANES) * 16, 16);
                if (m >= o.M) continue;
                T* const dst = to + m * ld + col;
                if (col + E <= o.N) {
                    *reinterpret_cast<Piece*>(dst) = v;
                } else {
#pragma unroll
                    for (int e = 0; e < E; ++e) {
                        if (col + e < o.N) dst[e] = v.e[e];
                    }
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
    };
    if (p.slices > 1) store(float{}, p.partial + static_cast<int64_t>(slice) * o.M * o.N, o.N);
    else store(half_t{}, o.out, o.N);
}

// out = the sum of the slices, rounded once.  Bound by the latency of its loads: the four waves of a workgroup share 256 outputs, 4 of a lane, and take
// every fourth slice, eight loads in flight each.
__global__ __launch_bounds__(256) void BatchedSumKernel(const float* partial, half_t* out, int64_t total, int slices) {
    __shared__ float others[3][64][5];
    struct __attribute__((packed, aligned(4))) Piece {
        float e[4];
    };
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t i = (static_cast<int64_t>(blockIdx.x) * 64 + lane) * 4;
    const int64_t from = i + 4 <= total ? i : (total >= 4 ? total - 4 : 0);  // the last outputs are summed by two lanes
    float sum[4] = {};
    if (total >= 4) {
#pragma unroll 8
        for (int s = wave; s < slices; s += 4) {
            const Piece v = *reinterpret_cast<const Piece*>(partial + s * total + from);
#pragma unroll
            for (int e = 0; e < 4; ++e) sum[e] += v.e[e];
        }
    } else {
        for (int s = wave; s < slices; s += 4) {
            for (int e = 0; e < total; ++e) sum[e] += partial[s * total + e];
        }
    }
    if (wave > 0) {
#pragma unroll
        for (int e = 0; e < 4; ++e) others[wave - 1][lane][e] = sum[e];
    }
    __syncthreads();
    if (wave > 0 || i >= total) return;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float all = sum[e] + others[0][lane][e] + others[1][lane][e] + others[2][lane][e];
        if (from + e < total) out[from + e] = static_cast<half_t>(all);
    }
}

// Where the last window of a row begins.
double LastTap(const BatchedOperands& o) {
    if (o.taps_s <= 0) return 0.0;
    const int last = o.taps_s - 1;
    const double even = static_cast<double>(last / 2) * o.s_pair_stride, odd = last > 0 ? static_cast<double>(o.s_stride) + (last - 1) / 2 * static_cast<double>(o.s_pair_stride) : 0.0;
    return (o.taps_r - 1.0) * o.r_stride + std::max(even, odd);
}

double Bytes(int64_t rows, int64_t row, int64_t slice, const BatchedOperands& o) { return 2.0 * ((rows - 1.0) * row + (o.batch - 1.0) * slice + o.depth); }

}  // namespace

// One workgroup to a compute unit (its ring then has the unit's whole bandwidth; two: 4 % slower, three: 8 %), two where one each would leave more than a
// quarter of the chip idle (144 tiles of 3x3 of 512 channels on 7 x 7: 73 -> 56 us).  Slices of 8 chunks at least: of 4, the sum outweighs the
// shorter loops (458 against 426 us over ResNet-50's shapes at batch 8); 16 is the same.  Multiples of 8, for the L2s.  Windows of a larger array make eight
// slices or more of 6 chunks already, which their tight rows of 14 would otherwise turn into half as many of the double length (24 images of 11 x 11, 50
// filters, 15 slices of 8: 11.3 us in 8, 9.0 in 16; 1x1 filters of 970 channels on 16 x 16 gain nothing, 16.1 and 18.3).
int HalfProductSlices(const BatchedOperands& o) {
    const int64_t tiles = std::max<int64_t>(1, ((int64_t{o.M} + 127) / 128) * ((int64_t{o.N} + 127) / 128)), chunks = (int64_t{o.depth} + 31) / 32 * o.batch;
    const int64_t cus = NumCUs();
    int64_t s = cus / tiles;
    if (s * tiles < cus * 3 / 4) s = 2 * cus / tiles;
    s = std::min(s, o.taps_s > 0 && chunks / 6 >= 8 ? chunks / 6 : chunks / 8);
    if (s >= 8) s = s / 8 * 8;
    return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(s, 256)));
}

bool HalfProductApplies(const BatchedOperands& o) {
    const double last_b = LastTap(o);
    const int64_t b_rows = o.taps_s > 0 ? o.N / (o.taps_r * o.taps_s) : o.N;
    const double limit = 2147483000.0;
    const int64_t tiles = ((static_cast<int64_t>(o.M) + 127) / 128) * ((static_cast<int64_t>(o.N) + 127) / 128);
    const int64_t odd = static_cast<int64_t>(reinterpret_cast<uintptr_t>(o.a) | reinterpret_cast<uintptr_t>(o.b)) / 2 | o.depth | o.a_row | o.a_slice | o.b_row |
                        o.b_slice | o.r_stride | o.s_stride | o.s_pair_stride;
    return o.depth >= 32 && odd % 2 == 0 && tiles < (1 << 14) && Bytes(o.M, o.a_row, o.a_slice, o) < limit && Bytes(b_rows, o.b_row, o.b_slice, o) + 2 * last_b < limit &&
           static_cast<double>(o.M) * o.N < limit;
}

void HalfProduct(const BatchedOperands& o, float* partial, int slices, hipStream_t stream) {
    ProductArgs p{};
    p.o = o;
    p.partial = partial;
    p.slices = slices;
    p.chunks_per_image = (o.depth + 31) / 32;
    p.tiles_n = (o.N + 127) / 128;
    const int64_t b_rows = o.taps_s > 0 ? o.N / (o.taps_r * o.taps_s) : o.N;
    const double last_b = LastTap(o);
    p.a_bytes = static_cast<unsigned>(Bytes(o.M, o.a_row, o.a_slice, o));
    p.b_bytes = static_cast<unsigned>(Bytes(b_rows, o.b_row, o.b_slice, o) + 2 * last_b);
    const int64_t tiles = static_cast<int64_t>((o.M + 127) / 128) * p.tiles_n;
    const double terms = static_cast<double>(o.depth) * o.batch;
    ProfileScope prof(stream, 2.0 * o.M * o.N * terms, 2.0 * (o.M * terms + o.N * terms + static_cast<double>(o.M) * o.N));
    struct BatchedProductTag {};
    EnsureDynamicLds<BatchedProductTag>(reinterpret_cast<const void*>(BatchedProductKernel), kRing * kStageBytes);
    hipLaunchKernelGGL(BatchedProductKernel, dim3(static_cast<unsigned>(tiles * slices)), dim3(256), kRing * kStageBytes, stream, p);
    CheckLaunch("batched_product");
    if (slices > 1) {
        const int64_t total = static_cast<int64_t>(o.M) * o.N;
        hipLaunchKernelGGL(BatchedSumKernel, dim3(static_cast<unsigned>((total + 255) / 256)), dim3(256), 0, stream, partial, o.out, total, slices);
        CheckLaunch("batched_product sum");
    }
}

}  // namespace hipcx
