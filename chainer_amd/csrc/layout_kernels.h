// Gather of an NCHW-shaped activation (any strides) into dense channels-last memory
// [N][H'][W'][Cpad], optionally sub-sampling the spatial axes (for strided 1x1 convolutions) and
// zero-padding the channel axis up to Cpad.  A 64(c) x 64(pixel) tile goes through LDS so that both
// the global reads (along pixels) and the global writes (along channels) are coalesced.
#pragma once

#include "common.h"

namespace hipcx {

struct ToChannelsLastArgs {
    const void* x;
    void* out;
    int N, C, Cpad;
    int Ho, Wo;          // output plane extents
    int step_h, step_w;  // input pixel = (h * step_h, w * step_w)
    int64_t xsN, xsC, xsH, xsW;  // elements
    int64_t first_tile;  // of 64 pixels
    int vec_in;          // 1: plane is dense along pixels (xsW == 1, xsH == Wo, steps 1) and 16-byte loads are aligned
};

template <typename T>
__global__ __launch_bounds__(256) void ToChannelsLastKernel(ToChannelsLastArgs a) {
    constexpr int TILE = 64;
    constexpr int EPV = 16 / sizeof(T);  // elements per 16 bytes
    constexpr int ROW = TILE + EPV;      // padded LDS row, elements
    __shared__ __align__(16) T tile[TILE * ROW];  // [pixel][channel]
    const T* x = static_cast<const T*>(a.x);
    T* out = static_cast<T*>(a.out);
    const int tid = threadIdx.x;
    const int64_t plane = static_cast<int64_t>(a.Ho) * a.Wo;
    const int64_t p0 = (a.first_tile + blockIdx.x) * TILE;
    const int c0 = blockIdx.y * TILE;
    const int n = blockIdx.z;
    const T* xn = x + n * a.xsN;

    if (a.vec_in) {
        // thread: channel row = tid / (TILE/EPV) + i * rows_per_pass, pixel chunk = tid % (TILE/EPV)
        constexpr int CHUNKS = TILE / EPV;
        constexpr int ROWS_PER_PASS = 256 / CHUNKS;
        struct alignas(16) V {
            T e[EPV];
        };
        const int pc = tid % CHUNKS;
#pragma unroll
        for (int i = 0; i < TILE / ROWS_PER_PASS; ++i) {
            int cl = tid / CHUNKS + i * ROWS_PER_PASS;
            int c = c0 + cl;
            int64_t p = p0 + pc * EPV;
            V v = {};
            if (c < a.C && p < plane) v = *reinterpret_cast<const V*>(xn + c * a.xsC + p);  // plane % EPV == 0: no partial chunk
#pragma unroll
            for (int e = 0; e < EPV; ++e) tile[(pc * EPV + e) * ROW + cl] = v.e[e];
        }
    } else {
        for (int e = tid; e < TILE * TILE; e += 256) {
            int pl = e % TILE;
            int cl = e / TILE;
            int c = c0 + cl;
            int64_t p = p0 + pl;
            T v = T(0);
            if (c < a.C && p < plane) {
                int w = static_cast<int>(p % a.Wo);
                int h = static_cast<int>(p / a.Wo);
                v = xn[c * a.xsC + static_cast<int64_t>(h) * a.step_h * a.xsH + static_cast<int64_t>(w) * a.step_w * a.xsW];
            }
            tile[pl * ROW + cl] = v;
        }
    }
    __syncthreads();
    {
        constexpr int CHUNKS = TILE / EPV;
        constexpr int ROWS_PER_PASS = 256 / CHUNKS;
        struct alignas(16) V {
            T e[EPV];
        };
        const int cc = tid % CHUNKS;
#pragma unroll
        for (int i = 0; i < TILE / ROWS_PER_PASS; ++i) {
            int pl = tid / CHUNKS + i * ROWS_PER_PASS;
            int64_t p = p0 + pl;
            int c = c0 + cc * EPV;
            if (p < plane && c < a.Cpad) {  // Cpad % EPV == 0
                V v = *reinterpret_cast<const V*>(&tile[pl * ROW + cc * EPV]);
                *reinterpret_cast<V*>(out + (static_cast<int64_t>(n) * plane + p) * a.Cpad + c) = v;
            }
        }
    }
}

template <typename T>
inline void LaunchToChannelsLast(ToChannelsLastArgs a, hipStream_t stream) {
    int64_t plane = static_cast<int64_t>(a.Ho) * a.Wo;
    if (plane == 0 || a.N == 0 || a.Cpad == 0) return;
    dim3 grid(1, static_cast<unsigned>((a.Cpad + 63) / 64), static_cast<unsigned>(a.N));
    HIPCX_REQUIRE(grid.y <= 65535 && grid.z <= 65535, HIPCX_NOT_IMPLEMENTED_ERROR, "too many channels or images for the layout kernel");
    const int64_t tiles = (plane + 63) / 64;
    for (a.first_tile = 0; a.first_tile < tiles; a.first_tile += kBlocksPerLaunch) {
        const int64_t left = tiles - a.first_tile;
        grid.x = static_cast<unsigned>(left < kBlocksPerLaunch ? left : kBlocksPerLaunch);
        hipLaunchKernelGGL((ToChannelsLastKernel<T>), grid, dim3(256), 0, stream, a);
    }
    CheckLaunch("to_channels_last");
}

// dst[r][c] (dense, row pitch dst_pitch elements, a multiple of 16 bytes; columns c >= cols zero-filled up to dst_pitch) = src[r * sr + c * sc]:
// brings a matrix operand whose reduction axis is not the unit-stride one into the layout the MFMA kernels read.
// Bound by memory.  A thread moves a block of E x E elements (E = 16 bytes' worth) by 16-byte accesses at any address and turns it
// round in registers; 8 x 8 threads make a wave's block, so that reads and writes both cover whole 128-byte lines without a detour
// through LDS.  [4480,10000] float16 transposed: 55 -> 40 us, against 64 x 64 tiles of single elements in LDS.
enum StageRead { kStageColumns, kStageRows, kStageElements };  // src's unit-stride axis: c, r, neither

template <typename T>
struct __attribute__((packed, aligned(1))) StagePiece {
    T e[16 / sizeof(T)];
};

template <typename T, int READ>
__global__ __launch_bounds__(256) void StageMatrixKernel(const T* src, int64_t sr, int64_t sc, T* dst, int64_t dst_pitch, int rows, int cols) {
    constexpr int E = 16 / static_cast<int>(sizeof(T)), TILE = 8 * E;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r0 = blockIdx.y * TILE + (lane & 7) * E;
    const int64_t c0 = (static_cast<int64_t>(blockIdx.x) * 4 + wave) * TILE + (lane >> 3) * E;
    if (r0 >= rows || c0 >= dst_pitch) return;
    StagePiece<T> in[E], out[E];  // in: by column where the source's rows are the unit-stride axis
    if (r0 + E <= rows && c0 + E <= cols && READ != kStageElements) {
#pragma unroll
        for (int i = 0; i < E; ++i) in[i] = *reinterpret_cast<const StagePiece<T>*>(READ == kStageRows ? src + r0 + (c0 + i) * sc : src + (r0 + i) * sr + c0);
    } else {
#pragma unroll
        for (int i = 0; i < E; ++i)
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int r = r0 + (READ == kStageRows ? e : i);
                const int64_t c = c0 + (READ == kStageRows ? i : e);
                in[i].e[e] = r < rows && c < cols ? src[r * sr + c * sc] : T(0);
            }
    }
#pragma unroll
    for (int i = 0; i < E; ++i)
#pragma unroll
        for (int e = 0; e < E; ++e) out[i].e[e] = READ == kStageRows ? in[e].e[i] : in[i].e[e];
#pragma unroll
    for (int i = 0; i < E; ++i) {
        if (r0 + i < rows) *reinterpret_cast<StagePiece<T>*>(dst + (r0 + i) * dst_pitch + c0) = out[i];
    }
}

template <typename T>
void StageMatrix(const T* src, int64_t sr, int64_t sc, T* dst, int64_t dst_pitch, int64_t rows, int64_t cols, hipStream_t stream) {
    constexpr int TILE = 128 / static_cast<int>(sizeof(T));
    // row tiles lie along the grid's y axis; more rows than it holds take several launches
    constexpr int64_t kMaxRows = int64_t{65535} * TILE;
    auto launch = [&](auto read) {
        for (int64_t r0 = 0; r0 < rows; r0 += kMaxRows) {
            const int64_t count = rows - r0 < kMaxRows ? rows - r0 : kMaxRows;
            const dim3 grid(static_cast<unsigned>((dst_pitch + 4 * TILE - 1) / (4 * TILE)), static_cast<unsigned>((count + TILE - 1) / TILE));
            hipLaunchKernelGGL((StageMatrixKernel<T, decltype(read)::value>), grid, dim3(256), 0, stream, src + r0 * sr, sr, sc, dst + r0 * dst_pitch,
                               dst_pitch, static_cast<int>(count), static_cast<int>(cols));
        }
    };
    if (sc == 1) launch(std::integral_constant<int, kStageColumns>{});
    else if (sr == 1) launch(std::integral_constant<int, kStageRows>{});
    else launch(std::integral_constant<int, kStageElements>{});
    CheckLaunch("stage_matrix");
}

}  // namespace hipcx
