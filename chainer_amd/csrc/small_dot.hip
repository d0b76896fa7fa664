// The small matrix product: which kernel of small_dot.h takes it, in how many parts, and the launches.
#include <algorithm>
#include <cstdlib>

#include "dot_parts.h"
#include "launch_profile.h"
#include "small_dot.h"

namespace hipcx {

// Fewer tiles of 128 x 128 than keep the chip busy; up to 256 for fewer than 64 terms, where larger tiles are bound by copying operands into their layout.  us,
// without and with these kernels: [64,33] . [33,64] float32 35 and 4.1, [20,50] . [50,8789] 33 and 4.2, float16 30 and 3.9, [128,63] . [63,2600] 41 and 4.6 (one
// element after another, or a wave to a tile); [352,35] . [35,8653], 204 tiles, float16 23 and 17 (float32 of that size is staged, see PlanDotStaging); beyond, 288
// tiles of [3000,33] . [33,1500], 18.2 and 18.9, float16 17.3 and 23.7.
bool SmallDotShape(int64_t m, int64_t n, int64_t k) { return ((m + 127) / 128) * ((n + 127) / 128) < (k >= 64 ? 128 : 256); }

namespace {

// Workgroups that share a tile's reduction: while tiles leave compute units without one, but at least 896 bytes of a row each.
int PlanSmallDotSplit(int64_t m, int64_t n, int64_t k, int dtype) {
    const int64_t tiles = ((m + 31) / 32) * ((n + 31) / 32), lines = (k * ItemSize(dtype) + 127) / 128;
    const int64_t s = std::min<int64_t>({NumCUs() / tiles, lines / 7, 32});
    return s > 1 ? static_cast<int>(s) : 1;
}

// Splitting pays for the extra pass over the partial sums (3-4 us) once a tile's reduction takes longer than that on one compute unit:
// 0.11 us per 128 bytes of its rows in float32 (16 MFMAs), 0.065 us in float16 (fetching the lines).  Against 1 to 32 parts on 206 products of
// 650 to 10007 terms the choice is within 10 % of the best for 162.  Not so for float16 operands read element by element, 0.27 us per 128 bytes:
// [20,3500] . [3500,650] row-major takes 17.6 us in one part and 8.1 in eight.
int SmallDotSplit(int64_t m, int64_t n, int64_t k, int dtype) {
    const int64_t lines = (k * ItemSize(dtype) + 127) / 128;
    return lines >= (dtype == HIPCX_FLOAT32 ? 48 : 80) ? PlanSmallDotSplit(m, n, k, dtype) : 1;
}

size_t SmallDotPartialBytes(int64_t m, int64_t n, int64_t k, int dtype) {
    const int split = SmallDotSplit(m, n, k, dtype);
    return split > 1 ? static_cast<size_t>(split) * m * n * sizeof(float) : 0;
}

// Fills in the operands; false when their strides or spans rule the kernels out.
template <typename T>
bool SmallDotOperands(const hipcx_array* a, const hipcx_array* b, SmallDotArgs* p, int* a_mode, int* b_mode) {
    const int64_t M = a->shape[0], K = a->shape[1], N = b->shape[1];
    const int64_t it = sizeof(T);
    for (const hipcx_array* x : {a, b}) {
        if (x->strides[0] < 0 || x->strides[1] < 0 || x->strides[0] % it || x->strides[1] % it) return false;
    }
    p->a = a->data;
    p->b = b->data;
    p->M = static_cast<int>(M);
    p->N = static_cast<int>(N);
    p->K = static_cast<int>(K);
    p->a_row = a->strides[0] / it;
    p->a_k = a->strides[1] / it;
    p->b_k = b->strides[0] / it;
    p->b_col = b->strides[1] / it;
    int64_t a_span = ((M - 1) * p->a_row + (K - 1) * p->a_k + 1) * it, b_span = ((K - 1) * p->b_k + (N - 1) * p->b_col + 1) * it;
    if (a_span >= (1LL << 31) - 256 || b_span >= (1LL << 31) - 256) return false;
    // (the stride of an axis of length one says nothing: a reshaped row may have any)
    auto mode = [&](const void* ptr, int64_t k_stride, int64_t lines, int64_t line_stride, int64_t* span) {
        if (k_stride != 1 && K > 1) return static_cast<int>(kElements);
        if (reinterpret_cast<uintptr_t>(ptr) % 4 == 0 && (lines == 1 || line_stride * it % 4 == 0)) {
            *span = (*span + 3) / 4 * 4;  // a last half element shares its (aligned) dword with the two bytes behind it
            return static_cast<int>(kPieces);
        }
        return static_cast<int>(kOddPieces);
    };
    *a_mode = mode(a->data, p->a_k, M, p->a_row, &a_span);
    *b_mode = mode(b->data, p->b_k, N, p->b_col, &b_span);
    p->a_bytes = static_cast<unsigned>(a_span);
    p->b_bytes = static_cast<unsigned>(b_span);
    p->tiles_m = static_cast<int>((M + 31) / 32);
    p->tiles_n = static_cast<int>((N + 31) / 32);
    return true;
}

// Elements come as they are used: chunks of 32 bytes, six of them in flight, beat whole lines ([32,1000] . [1000,2048] float16 14.3 -> 5.5 us,
// [200,4000] . [4000,4000] 174 -> 51, [20,2600] . [2600,650] float32 13.4 -> 9.3); rows of odd pitch gain from whole lines at any size.
template <typename T, int AM, int BM>
void LaunchSmallDotMixed(const SmallDotArgs& p, dim3 grid, hipStream_t stream) {
    constexpr int kWaveBytes = std::max<int>(AM == kOddPieces || BM == kOddPieces ? kSmallDotStage : 0, kSmallDotPart * sizeof(float));
    struct SmallDotTag {};
    EnsureDynamicLds<SmallDotTag>(reinterpret_cast<const void*>(SmallDotMixedKernel<T, AM, BM>), kSmallDotMaxWaves * kWaveBytes);
    hipLaunchKernelGGL((SmallDotMixedKernel<T, AM, BM>), grid, dim3(64 * p.nw), p.nw * kWaveBytes, stream, p);
    CheckLaunch("small_dot_mixed");
}

// Columns, in 16s, of the tiles of whole lines regrouped through LDS (SmallDotLinesKernel); 0: loads straight into the MFMA layout (SmallDotKernel) are
// faster.  `rows` tiles of 32 rows, each of whose reductions of `k` terms `parts` workgroups share.  Tiles take the narrowest width that finds each of
// them a compute unit, and long enough reductions: below, the detour through LDS outweighs the lines.  us, SmallDotKernel, then tiles of 16, 32, 48 and 64
// columns (more of them: profiles/matrix_product_plans.txt): float32 [100,1000] . [1000,1000] 8.5 7.4 9.1 11.3, [128,650] . [650,2600] 12.2 12.0 12.4 11.1
// 12.7, [100,300] . [300,1000] 4.7 5.0 6.2; float16 [37,2048] . [2048,1000] 9.7 5.1 6.1 7.3, [500,1000] . [1000,1000] 9.5 8.8 10.3 11.3 8.3.  No width that
// pads the columns by a tenth more than 32 does ([2122,442] . [442,106] in float16 5.2 us, 6.0 by 48 columns).
template <typename T>
int LinesBlocks(int64_t rows, int64_t n, int64_t parts, int64_t k) {
    constexpr bool kHalf = sizeof(T) == 2;
    const int64_t cus = NumCUs(), bytes = k * static_cast<int64_t>(sizeof(T)), least = kHalf ? 800 : 1600;
    auto groups = [&](int blocks) { return rows * ((n + 16 * blocks - 1) / (16 * blocks)) * parts; };
    if (groups(1) <= cus) return bytes >= 1600 ? 1 : 0;
    if (groups(2) <= cus) {
        if (kHalf) return bytes >= 1600 ? 2 : 0;
        return bytes >= 6144 || (bytes >= 4096 && groups(2) > cus * 3 / 4) ? 2 : 0;
    }
    auto fits = [&](int blocks) { return groups(blocks) <= cus && 10 * blocks * groups(blocks) <= 11 * 2 * groups(2); };
    if (fits(3)) return bytes >= least ? 3 : 0;
    if (kHalf && fits(4)) return bytes >= least ? 4 : 0;
    if (bytes <= (groups(2) > 2 * cus ? 7 * 128 : least)) return 0;
    return kHalf && 10 * 3 * groups(3) <= 11 * 2 * groups(2) ? 3 : 2;
}

// Their waves: eight keep most loads in flight while a compute unit has one or two tiles (328 float32 tiles of 21 chunks: 12.3 us, 12.8 with four, 16.6
// with two), or four for the lighter float16 ones beyond one ([150,1024] . [1024,4096] by 48 columns 9.6 -> 8.6 us); beyond, what leaves the busiest SIMD
// the fewest chunks, fewer waves on near terms (626 tiles of 21 chunks: 17.6 us with two, 18.2 with three, 16.5 with four; 1252 of 21: 26.9, 26.5, 29.0;
// 1504 of 25: 34.1, 37.9, 35.3).
int LinesWaves(int64_t groups, int chunks, bool half) {
    if (groups <= 2 * NumCUs()) return std::min(half && groups > NumCUs() ? 4 : kSmallDotMaxWaves, chunks);
    const int64_t per_unit = (groups + NumCUs() - 1) / NumCUs();
    auto cost = [&](int nw) { return (per_unit * nw + 3) / 4 * ((chunks + nw - 1) / nw); };
    int best = 2;
    for (int nw : {3, 4}) {
        if (10 * cost(nw) < 9 * cost(best)) best = nw;
    }
    return std::min(best, chunks);
}

// Columns, in 16s, of the tiles of 64 rows (SmallDotSquaresKernel); 0: other tiles are faster.  They read each operand half as often as 32 rows do, but one of them
// occupies a compute unit, so it takes outputs that fill one round of them (float32: or two) and enough terms for the kernel's slow start.  Of 128 products of 66 to
// 4084 terms these are the 42 that gain 1 to 52 %, 12 in the middle; us, without and with them: float32 [128,650] . [650,10000] (0.98 of a round) 28.1 24.8,
// [512,1000] . [1000,1000] (0.98) 17.8 15.6, [143,1682] . [1682,3773] (0.69) 34.1 31.6, [670,3324] . [3324,2007] (0.86 of two) 126 107; float16
// [1782,2632] . [2632,471] (0.80) 30.3 19.9, [99,1654] . [1654,5651] (0.71) 15.6 12.5.  Beside the lines: float32 [135,932] . [932,3209] (0.55) 17.4 20.2,
// [308,262] . [262,1617] 8.2 8.7, [467,788] . [788,3290] (0.73 of two) 40.4 41.2, float16 [994,424] . [424,807] (0.77) 8.4 8.8, [814,378] . [378,1580] (0.82 of two)
// 10.1 13.2.
template <typename T>
int SquaresBlocks(int64_t m, int64_t n, int64_t k) {
    if (k < (sizeof(T) == 4 ? 300 : 470)) return 0;
    int best = 0;
    double most = 0;
    for (int rounds = 1; rounds <= (sizeof(T) == 4 ? 2 : 1); ++rounds) {
        for (int blocks = 2; blocks <= 5; ++blocks) {
            const int64_t groups = (m + 63) / 64 * ((n + 16 * blocks - 1) / (16 * blocks));
            if (groups > rounds * NumCUs()) continue;
            const double filled = static_cast<double>(m) * n / (64.0 * 16 * blocks * rounds * NumCUs());
            if (filled >= (rounds == 1 ? 0.65 : 0.8) && filled > most) best = blocks, most = filled;
            break;  // wider tiles only leave more idle
        }
        if (best > 0) return best;
    }
    return 0;
}

// `batch` products (SmallDotArgs::outs) of p.ksplit workgroups per tile.
template <typename T>
void LaunchSmallDot(SmallDotArgs p, int a_mode, int b_mode, int batch, hipStream_t stream) {
    const int64_t tiles = static_cast<int64_t>(p.tiles_m) * p.tiles_n;
    const dim3 grid(static_cast<unsigned>(tiles * p.ksplit), static_cast<unsigned>(batch));
    // nine terms stay in one chain: a second wave's only product would be rounded once more (5.67e-8 of the norm and 5.78e-8)
    const bool one_chain = sizeof(T) == 4 && p.K == 9;
    if (a_mode != kElements && b_mode != kElements && p.K >= 16 / static_cast<int>(sizeof(T))) {
        const int chunks = ((p.K * static_cast<int>(sizeof(T)) + 127) / 128 + p.ksplit - 1) / p.ksplit;
        auto lines = [&](auto blocks_tag) {
            constexpr int NB = decltype(blocks_tag)::value, kWaveBytes = (32 + 16 * NB) * kSmallDotPitch;
            p.tiles_n = (p.N + 16 * NB - 1) / (16 * NB);
            const int64_t groups = static_cast<int64_t>(p.tiles_m) * p.tiles_n * p.ksplit;
            p.nw = LinesWaves(groups * batch, chunks, sizeof(T) == 2);
            struct LinesTag {};
            EnsureDynamicLds<LinesTag>(reinterpret_cast<const void*>(SmallDotLinesKernel<T, NB>), kSmallDotMaxWaves * kWaveBytes);
            hipLaunchKernelGGL((SmallDotLinesKernel<T, NB>), dim3(static_cast<unsigned>(groups), static_cast<unsigned>(batch)), dim3(64 * p.nw), p.nw * kWaveBytes,
                               stream, p);
            CheckLaunch("small_dot_lines");
        };
        const int square_blocks = p.ksplit == 1 && batch == 1 ? SquaresBlocks<T>(p.M, p.N, p.K) : 0;
        auto squares = [&](auto blocks_tag) {
            constexpr int NB = decltype(blocks_tag)::value, kLds = std::max(2 * (64 + (NB + 1) / 2 * 32) * kSquaresPitch, 4 * 64 * (16 * NB + 1) * 4);
            p.tiles_m = (p.M + 63) / 64, p.tiles_n = (p.N + 16 * NB - 1) / (16 * NB);
            struct SquaresTag {};
            EnsureDynamicLds<SquaresTag>(reinterpret_cast<const void*>(SmallDotSquaresKernel<T, NB>), kLds);
            hipLaunchKernelGGL((SmallDotSquaresKernel<T, NB>), dim3(static_cast<unsigned>(p.tiles_m * p.tiles_n)), dim3(512), kLds, stream, p);
            CheckLaunch("small_dot_squares");
        };
        switch (square_blocks) {
            case 2: return squares(std::integral_constant<int, 2>{});
            case 3: return squares(std::integral_constant<int, 3>{});
            case 4: return squares(std::integral_constant<int, 4>{});
            case 5: return squares(std::integral_constant<int, 5>{});
        }
        int blocks = LinesBlocks<T>(p.tiles_m, p.N, static_cast<int64_t>(p.ksplit) * batch, p.K / p.ksplit);
        // SmallDotKernel reads beyond the end of a row, which does not do for the last one of an odd pitch.  us, by elements where a piece does not fit, and so:
        // [20,651] . [651,2600] 6.3 4.8, [64,33] . [33,500] 7.7 5.5, [128,101] . [101,3000] 7.5 5.4; in tiles of 32 columns 5.7, 7.3, 6.7.  Other widths take these
        // rows as well: [1000,785] . [785,1000] 26.1 12.1 (784 terms 10.9), [37,801] . [801,1000] 7.3 5.2.
        if (blocks == 0 && (a_mode == kOddPieces || b_mode == kOddPieces)) blocks = 1;
        switch (blocks) {
            case 1: return lines(std::integral_constant<int, 1>{});
            case 2: return lines(std::integral_constant<int, 2>{});
            case 3: return lines(std::integral_constant<int, 3>{});
            case 4:
                if constexpr (sizeof(T) == 2) return lines(std::integral_constant<int, 4>{});
        }
        if (a_mode == kPieces && b_mode == kPieces && !one_chain) {
            hipLaunchKernelGGL((SmallDotKernel<T>), grid, dim3(512), 0, stream, p);
            CheckLaunch("small_dot");
            return;
        }
    } else if (a_mode == kPieces && b_mode == kPieces) {
        hipLaunchKernelGGL((SmallDotKernel<T>), grid, dim3(512), 0, stream, p);
        CheckLaunch("small_dot");
        return;
    }
    if constexpr (sizeof(T) == 4) {
        // Once 64 x 64 tiles occupy three quarters of the compute units; us, elements in 32 x 32 tiles and these: [700,650]^T . [700,650], 121 tiles, 15.0
        // and 19.4, [100,784]^T . [100,1000], 208, 8.8 and 7.9, [64,1300]^T . [64,1300], 441, 11.3 and 10.6.  Not for fewer than 64
        // terms, these and elements: [20,2000]^T . [20,1900] 18.5 and 16.4, [12,1000]^T . [12,1000] 7.5 and 5.5, [35,650]^T . [35,1300] 7.5 and 6.0.
        const int64_t squares = static_cast<int64_t>((p.M + 63) / 64) * ((p.N + 63) / 64) * p.ksplit * batch;
        if (p.K >= 64 && a_mode == kElements && b_mode == kElements && p.a_row == 1 && p.b_col == 1 && 4 * squares >= 3 * NumCUs()) {
            constexpr int kLds = 4 * 64 * (64 + 4) * 4;
            p.tiles_m = (p.M + 63) / 64, p.tiles_n = (p.N + 63) / 64;
            struct ColumnsTag {};
            EnsureDynamicLds<ColumnsTag>(reinterpret_cast<const void*>(SmallDotColumnsKernel<float>), kLds);
            hipLaunchKernelGGL((SmallDotColumnsKernel<float>), dim3(static_cast<unsigned>(static_cast<int64_t>(p.tiles_m) * p.tiles_n * p.ksplit), static_cast<unsigned>(batch)),
                               dim3(256), kLds, stream, p);
            CheckLaunch("small_dot_columns");
            return;
        }
    }
    if (a_mode != kElements && b_mode != kElements) a_mode = b_mode = kElements;  // (fewer terms than a piece holds)
    // eight waves keep more loads in flight; four, one per SIMD, once there is a workgroup for every compute unit
    const int chunk = a_mode == kOddPieces || b_mode == kOddPieces ? 128 : 32, chunks = (p.K * static_cast<int>(sizeof(T)) + chunk - 1) / chunk;
    const int per_split = (chunks + p.ksplit - 1) / p.ksplit;
    const int most = static_cast<int>(grid.x) * batch <= NumCUs() ? kSmallDotMaxWaves : 4;
    const int per_wave = one_chain ? per_split : (per_split + most - 1) / most;
    p.nw = (per_split + per_wave - 1) / per_wave;
    if (a_mode == kPieces) return LaunchSmallDotMixed<T, kPieces, kElements>(p, grid, stream);
    if (b_mode == kPieces) return LaunchSmallDotMixed<T, kElements, kPieces>(p, grid, stream);
    if constexpr (sizeof(T) == 2) {
        if (a_mode == kOddPieces) return LaunchSmallDotMixed<T, kOddPieces, kElements>(p, grid, stream);
        if (b_mode == kOddPieces) return LaunchSmallDotMixed<T, kElements, kOddPieces>(p, grid, stream);
    }
    LaunchSmallDotMixed<T, kElements, kElements>(p, grid, stream);
}

// Rows of a and columns of b of whole 8-byte granules, k dense: what IGemmFastKernel and IGemmSplitKernel read.
template <typename T>
bool LiesForTiles(const hipcx_array* a, const hipcx_array* b) {
    const int64_t it = sizeof(T), k = a->shape[1];
    auto lies = [&](const void* ptr, int64_t line, int64_t k_stride) {
        return k_stride == it && line % 8 == 0 && k * it % 8 == 0 && reinterpret_cast<uintptr_t>(ptr) % 8 == 0;
    };
    return lies(a->data, a->strides[0], a->strides[1]) && lies(b->data, b->strides[1], b->strides[0]);
}

// Which kernel of small_dot.h takes a product.
enum SmallDotPath { kNoSmallDot, kSmallDotVector, kSmallDotTiles, kSmallDotWhole };  // (whole: tiles whose reduction is not split)

template <typename T>
SmallDotPath PlanSmallDot(const hipcx_array* a, const hipcx_array* b, SmallDotArgs* p, int* a_mode, int* b_mode) {
    static const bool enabled = [] { const char* e = getenv("HIPCX_SMALL_DOT"); return e == nullptr || e[0] != '0'; }();
    const int64_t M = a->shape[0], K = a->shape[1], N = b->shape[1];
    if (!enabled || !SmallDotShape(M, N, K) || !SmallDotOperands<T>(a, b, p, a_mode, b_mode)) return kNoSmallDot;
    if (K < 64 && LiesForTiles<T>(a, b)) {
        // The tiles of 128 x 128 read these operands as they lie.  float16: [1000,32] . [32,1000] 7.9 us there and 5.0 here, [8192,8] . [8,512] (256 of them) 8.7 and
        // 13.2.  float32: 6 to 10 us there and 3 to 6 here, but with errors of 2.8e-8 to 4.6e-8 (2-norm, 8 to 50 terms; bfloat16 parts) and 5.4e-8 to 7.7e-8; a
        // single tile is summed term by term there, which recurrent networks that amplify rounding are held to.
        if (sizeof(T) == 4 || ((M + 127) / 128) * ((N + 127) / 128) >= 128) return kNoSmallDot;
    }
    if (*a_mode != kPieces || *b_mode != kPieces) return kSmallDotTiles;
    if (M <= 4) {
        // A wave to a column.  float32 whatever its size, whose lanes' sums are short, but not few terms: a product is rounded before it is added there, 4.4e-8 of the norm
        // for three terms where a chain of the matrix pipe has 3.7e-8.  float16, whose products cost two conversions each there and which the tiles take as fast for ten
        // thousand columns as for one thousand, where the columns are few or the terms many.  us, tiles and waves, one row: [1,512] . [512,3000] 3.8 3.8, [1,1000] . [1000,5000]
        // 4.7 4.5, 6000 columns 4.7 4.8, 10000 5.5 6.4, [1,2048] . [2048,10000] 9.2 8.6; two: [2,1000] . [1000,2561] 4.3 4.6, [2,2048] . [2048,4000] 5.3 5.2, 6000 6.1 6.5;
        // four: [4,1000] . [1000,1000] 4.2 4.2, [4,2048] . [2048,1000] 5.1 4.2, 2000 5.2 5.3, [4,3000] . [3000,500] 5.9 5.6, 2000 6.0 7.7, [4,332] . [332,3333] 3.3 7.1.
        const int64_t most = sizeof(T) == 4 ? (K >= 64 ? N : 0) : M > 2 ? (K >= 2048 ? 1280 : 0) : std::max<int64_t>(2560, M == 1 ? 28 * K / 5 : 5 * K / 2);
        if (N <= most) return kSmallDotVector;
    }
    return 2.0 * M * N * K >= 1e9 ? kSmallDotWhole : kSmallDotTiles;  // enough tiles, or enough of them long, to keep the chip busy
}

template <typename T>
bool TryTyped(const hipcx_array* a, const hipcx_array* b, const hipcx_array* bias, const hipcx_array* out, float* partial, hipStream_t stream) {
    const int64_t M = a->shape[0], K = a->shape[1], N = b->shape[1];
    const int64_t it = sizeof(T);
    if (out->strides[0] < 0 || out->strides[1] < 0 || out->strides[0] % it || out->strides[1] % it) return false;
    SmallDotArgs p{};
    int a_mode = 0, b_mode = 0;
    const SmallDotPath path = PlanSmallDot<T>(a, b, &p, &a_mode, &b_mode);
    if (path == kNoSmallDot) return false;
    p.out = out->data;
    p.o_row = out->strides[0] / it;
    p.o_col = out->strides[1] / it;
    if (bias != nullptr) {
        p.bias = bias->data;
        p.bias_stride = bias->strides[0] / it;
    }
    ProfileScope prof(stream, 2.0 * M * N * K, static_cast<double>(it) * (M * K + K * N + M * N));
    if (path == kSmallDotVector) {
        const dim3 grid(static_cast<unsigned>((N + 3) / 4));
        if (M == 1) hipLaunchKernelGGL((SmallDotVectorKernel<T, 1>), grid, dim3(256), 0, stream, p);
        else if (M == 2) hipLaunchKernelGGL((SmallDotVectorKernel<T, 2>), grid, dim3(256), 0, stream, p);
        else hipLaunchKernelGGL((SmallDotVectorKernel<T, 4>), grid, dim3(256), 0, stream, p);
        CheckLaunch("small_dot_vector");
        return true;
    }
    p.ksplit = partial != nullptr && path == kSmallDotTiles ? SmallDotSplit(M, N, K, DtypeOf<T>::value) : 1;
    p.partial = p.ksplit > 1 ? partial : nullptr;
    LaunchSmallDot<T>(p, a_mode, b_mode, 1, stream);
    if (p.ksplit > 1) {
        hipLaunchKernelGGL((SmallDotSumKernel<T>), dim3(static_cast<unsigned>((M * N + 255) / 256)), dim3(256), 0, stream, p);
        CheckLaunch("small_dot_sum");
    }
    return true;
}

}  // namespace

size_t SmallDotWorkspace(const hipcx_array* a, const hipcx_array* b, int dtype) {
    if (dtype != HIPCX_FLOAT16 && dtype != HIPCX_FLOAT32) return 0;
    const size_t bytes = SmallDotPartialBytes(a->shape[0], b->shape[1], a->shape[1], dtype);
    if (bytes == 0) return 0;  // most products
    SmallDotArgs p{};
    int a_mode = 0, b_mode = 0;
    const SmallDotPath path = dtype == HIPCX_FLOAT16 ? PlanSmallDot<half_t>(a, b, &p, &a_mode, &b_mode) : PlanSmallDot<float>(a, b, &p, &a_mode, &b_mode);
    return path == kSmallDotTiles ? bytes : 0;
}

bool TrySmallDot(const hipcx_array* a, const hipcx_array* b, const hipcx_array* bias, const hipcx_array* out, float* partial, hipStream_t stream) {
    return out->dtype == HIPCX_FLOAT16 ? TryTyped<half_t>(a, b, bias, out, partial, stream) : TryTyped<float>(a, b, bias, out, partial, stream);
}

bool DotSeveral(const hipcx_array* a0, int64_t a_distance, const hipcx_array* b, const hipcx_array* const* outs, int n, hipStream_t stream) {
    const int64_t M = a0->shape[0], K = a0->shape[1], N = b->shape[1];
    SmallDotArgs p{};
    int a_mode = 0, b_mode = 0;
    if (n > kSmallDotMaxBatch || !SmallDotShape(M, N, K) || SmallDotSplit(M, N, K, HIPCX_FLOAT32) > 1) return false;
    if (K < 64 && 2.0 * M * N * K >= 2e8) return false;  // one by one they run on the bfloat16 parts, with half the error (PlanDotStaging)
    if (!SmallDotOperands<float>(a0, b, &p, &a_mode, &b_mode)) return false;
    for (int i = 0; i < n; ++i) {
        if (outs[i]->strides[0] != outs[0]->strides[0] || outs[i]->strides[1] != outs[0]->strides[1]) return false;
        p.outs[i] = outs[i]->data;
    }
    if (outs[0]->strides[0] < 0 || outs[0]->strides[1] < 0 || outs[0]->strides[0] % 4 || outs[0]->strides[1] % 4) return false;
    p.out = outs[0]->data;
    p.o_row = outs[0]->strides[0] / 4;
    p.o_col = outs[0]->strides[1] / 4;
    p.a_batch = a_distance;
    p.ksplit = 1;
    ProfileScope prof(stream, 2.0 * M * N * K * n, 4.0 * n * (M * K + K * N + M * N));
    LaunchSmallDot<float>(p, a_mode, b_mode, n, stream);
    return true;
}

}  // namespace hipcx
