// float16 matrix product on the matrix pipes of gfx950 for large problems whose operands both have the reduction index as
// their unit-stride axis:
//
//   c[m][n] = sum_k a[m][k] * b[n][k]          (float accumulation, one rounding to float16)
//
// A workgroup of eight wavefronts owns a 256 x 256 tile of c and walks k in chunks of 32.  Operands reach LDS without passing
// through registers (buffer loads with the LDS modifier: 16 bytes per lane, 1 KiB per instruction) into a ring of three
// stages: stage[row][4 pieces of 8 halves], piece g of row r at position g ^ ((r >> 2) & 3) (the loading lane picks the
// global piece that belongs at its LDS position), so that the 16-byte fragment reads of consecutive rows use all banks.
// A wave multiplies 128 rows of a by 64 rows of b (4 x 2 MFMA 32x32x16 blocks, 128 accumulator registers).  The waves form
// two groups of four (one of each on every SIMD) that alternate between a memory phase (issue the loads of the chunk two
// ahead, read the 12 fragments of the current chunk) and an MFMA phase (16 MFMAs on registers), half a period apart and
// separated by workgroup barriers: while one wave of a SIMD multiplies, the other one feeds.
// k may be any number: the last chunk is masked in registers; rows need dword alignment only.  Where tiles leave compute units idle the
// reduction is split over `slices` workgroups, whose float sums GemmSumKernel adds up.  An operand that lies k by k (the weights of a gradient, both
// operands of a weight gradient) is loaded as it lies and turned round by transposing LDS reads.
// Bound by the matrix pipes and, in short reductions, by writing c.  us, against 128 x 128 tiles over padded copies of the operands:
// [4480,650] . [650,10000] 126 -> 95, [4480,10000] . [10000,650] 188 -> 115, [10000,4480] . [4480,650] with a and b transposed 198 -> 130;
// [4096,4096]^2 126 (1089 TFLOP/s).  Against copies with the reduction axis dense: [4480,10000] . [10000,650], b k by k, 104 -> 86; [10000,4480] .
// [4480,650], a and b, 130 -> 85; [4096,4480] . [4480,1024], a and b, 116 -> 57; [4096,4096]^2 152 -> 125.
// Tiles are ordered so that the 32 workgroups an XCD runs at a time cover `band` tile rows x 32 / band tile columns: they
// share operand rows in that XCD's L2.
#pragma once

#include "common.h"
#include "igemm.h"
#include "lds_load.h"
#include "nchw_conv.h"

namespace hipcx {
namespace gemm_pp {

struct GemmArgs {
    const half_t* a;
    const half_t* b;
    half_t* c;
    int M, N, K;
    int lda, ldb, ldc;  // elements; rows of a and b (their columns, where those are what is dense) start at multiples of 4 bytes
    int tiles_m, tiles_n;
    int slices;         // workgroups per tile along k
    int slice_chunks;   // chunks of 32 k of a slice (the last one may have fewer), at least kMinK / 32
    float* partial;     // slices > 1: [slices][M][N] sums go there, GemmSumKernel makes c of them
    int band;  // tile rows per band of the tile order
    const half_t* bias;  // one element per column of c, added before the rounding; may be null
    int64_t bias_stride;
};

constexpr int kStages = 3;
constexpr int kLdsBytes = kStages * 2 * 256 * 64, kPairLdsBytes = kStages * (256 + 128) * 64;
constexpr int kMinK = 32 * (kStages - 1);  // the pipeline's prologue issues kStages - 1 chunks
// Rows of a wave's 32 x 64 block on its way out, a float for partial sums: 16 bytes of padding keep the banks apart.
constexpr int kOutPitch = 64 * 4 + 16;
static_assert(8 * 32 * kOutPitch <= kLdsBytes, "the eight waves' blocks fit the ring");

template <typename T>
struct __attribute__((packed, aligned(2))) OutPiece {  // 16 bytes of c, whose rows may start anywhere
    T e[16 / sizeof(T)];
};

// A_COLS, B_COLS: the operand lies k by k, a[k][m] or b[k][n] with m or n dense (transposing LDS reads, ds_read_b64_tr_b16, turn it round).
// PAIR: tiles of 256 x 128 by four waves, two workgroups to a compute unit: one's start and end run under the other's products, which in short reductions
// is most of the time.  us, against one workgroup of eight waves (with the stores straight from the registers) and the 128 x 128 kernel: [8192,128] .
// [128,8192] 125, 109, 54; [4480,256] . [256,10000] 98, 91, 54; [1500,64] . [64,3000] 28, 19, 10; [10000,300] . [300,5000] 86, 154, 82.
template <bool A_COLS, bool B_COLS, bool PAIR>
__global__ __launch_bounds__(PAIR ? 256 : 512, 2) void GemmPpKernel(GemmArgs p) {
    static_assert(!PAIR || !(A_COLS || B_COLS), "pairs read rows");
    constexpr int NSTAGE = kStages, AHEAD = NSTAGE - 1;
    constexpr int WAVES = PAIR ? 4 : 8, COLS = WAVES * 32;
    constexpr int TILE_B = 256 * 64;  // bytes of a's tile in a stage
    constexpr int STAGE_B = TILE_B + COLS * 64;
    constexpr int LPA = 16 / WAVES, LPB = COLS / 16 / WAVES;  // load instructions per operand, wave and chunk
    constexpr int LPC = LPA + LPB;
    extern __shared__ __align__(16) char lds[];

    // ---- tile of this workgroup: XCD x (workgroup ids go round-robin to the 8 XCDs) walks a contiguous range of the tile
    // order; inside it bands of `band` tile rows are walked column by column ----
    const int tiles = p.tiles_m * p.tiles_n;
    const int total = tiles * p.slices;
    const int per = (total + 7) / 8;
    int logical = (static_cast<int>(blockIdx.x) % 8) * per + static_cast<int>(blockIdx.x) / 8;
    if (logical >= total) return;
    const int slice = logical / tiles;
    logical -= slice * tiles;
    const int k0 = slice * p.slice_chunks * 32;
    const int k_left = p.K - k0;
    int tile_m, tile_n;
    {
        const int band_tiles = p.band * p.tiles_n;
        const int bi = logical / band_tiles;
        const int rem = logical - bi * band_tiles;
        const int rows = min(p.band, p.tiles_m - bi * p.band);
        tile_m = bi * p.band + rem % rows;
        tile_n = rem / rows;
    }
    const int m0 = tile_m * 256, n0 = tile_n * COLS;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = wave >> 2;
    const int wm = wave & 1, wn = wave >> 1;
    const int r = lane & 31, h = lane >> 5;

    // ---- global -> LDS loads.  Rows: a wave instruction covers 16 rows x 64 bytes; lane = 4 * row + position.  Columns: two k of 256 elements, kept
    // as they lie (stage[k][32 pieces of 8 elements]), 16-byte piece i of k at position i ^ (4 * (k & 3)): the four k that a transposing read
    // combines then fall into four different 64-byte bank groups ----
    // what lies behind the last element of the last row is out of the buffers' bounds (an odd end shares its dword with 2 more bytes)
    auto span = [&](int rows, int ld, int cols) { return ((static_cast<unsigned>(rows - 1) * static_cast<unsigned>(ld) + cols) * 2u + 3u) & ~3u; };
    const int rows_a = min(p.M - m0, 256), rows_b = min(p.N - n0, COLS);
    const int4_t ra = A_COLS ? RawRsrc(p.a + static_cast<int64_t>(k0) * p.lda + m0, span(k_left, p.lda, rows_a))
                             : RawRsrc(p.a + static_cast<int64_t>(m0) * p.lda + k0, span(rows_a, p.lda, k_left));
    const int4_t rb = B_COLS ? RawRsrc(p.b + static_cast<int64_t>(k0) * p.ldb + n0, span(k_left, p.ldb, rows_b))
                             : RawRsrc(p.b + static_cast<int64_t>(n0) * p.ldb + k0, span(rows_b, p.ldb, k_left));
    int voa[LPA], vob[LPB];
    // beyond the buffer: zeros (rows of k from K on are beyond it too)
    auto offsets = [&](auto cols_tag, auto& vo, int rows, int ld) {
        constexpr int LPO = sizeof(vo) / sizeof(int);
#pragma unroll
        for (int i = 0; i < LPO; ++i) {
            const int row = (wave * LPO + i) * 16 + (lane >> 2);
            const int piece = (lane & 3) ^ ((lane >> 4) & 3);  // (row >> 2) & 3 = (lane >> 4) & 3
            const int k = (wave * LPO + i) * 2 + (lane >> 5), col = ((lane & 31) ^ (4 * (k & 3))) * 8;
            if constexpr (decltype(cols_tag)::value) vo[i] = col < rows ? (k * ld + col) * 2 : 0x7fffffff;
            else vo[i] = row < rows ? row * ld * 2 + piece * 16 : 0x7fffffff;
        }
    };
    offsets(std::integral_constant<bool, A_COLS>{}, voa, rows_a, p.lda);
    offsets(std::integral_constant<bool, B_COLS>{}, vob, rows_b, p.ldb);
    const unsigned lds_base = static_cast<unsigned>(reinterpret_cast<uintptr_t>(lds));
    const int step_a = A_COLS ? p.lda * 64 : 64, step_b = B_COLS ? p.ldb * 64 : 64;  // bytes of a chunk
    auto issue = [&](int c) {
        const unsigned st = lds_base + (c % NSTAGE) * STAGE_B;
#pragma unroll
        for (int i = 0; i < LPA; ++i) LdsLoad16(ra, st + (wave * LPA + i) * 1024, voa[i], c * step_a);
#pragma unroll
        for (int i = 0; i < LPB; ++i) LdsLoad16(rb, st + TILE_B + (wave * LPB + i) * 1024, vob[i], c * step_b);
    };

    // ---- fragment addresses: rows of a are the MFMA column operand, rows of b the row operand, so that a lane ends up with
    // 4 consecutive n of one m: an 8-byte store into row-major c ----
    const int pos0 = h ^ ((r >> 2) & 3), pos1 = (2 + h) ^ ((r >> 2) & 3);
    const unsigned fa0 = lds_base + (wm * 128 + r) * 64 + pos0 * 16, fa1 = lds_base + (wm * 128 + r) * 64 + pos1 * 16;
    const unsigned fb0 = lds_base + TILE_B + (wn * 64 + r) * 64 + pos0 * 16, fb1 = lds_base + TILE_B + (wn * 64 + r) * 64 + pos1 * 16;

    // columns: lane = 16 g + 4 q + s addresses elements 16 (g & 1) + 4 s .. + 3 of k = 8 (g >> 1) + q and receives element 16 (g & 1) + 4 q + s of four k
    const int fg = lane >> 4, fq = (lane >> 2) & 3, fs = lane & 3;
    const unsigned col0 = (8 * (fg >> 1) + fq) * 512 + (fs & 1) * 8;
    const unsigned ca0 = col0 + ((16 * wm + 2 * (fg & 1) + (fs >> 1)) ^ (4 * fq)) * 16, cb0 = col0 + TILE_B + ((8 * wn + 2 * (fg & 1) + (fs >> 1)) ^ (4 * fq)) * 16;

    float16_t acc[4][2];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

    Bytes16 fm[2][4], fn[2][2];
    // All fragment reads of a chunk and the wait for them in one statement: nothing touches the registers before the
    // data has landed.
    auto read_frags = [&](int c) {
        const unsigned so = (c % NSTAGE) * STAGE_B;
        Bytes8 am[2][4][2], bn[2][2][2];
        const unsigned at = lds_base + so, a0 = A_COLS ? at + ca0 : fa0 + so, a1 = A_COLS ? at + (ca0 ^ 64) : fa1 + so, a2 = at + (ca0 ^ 128), a3 = at + (ca0 ^ 192);
        const unsigned b0 = B_COLS ? at + cb0 : fb0 + so, b1 = B_COLS ? at + (cb0 ^ 64) : fb1 + so;
        if constexpr (A_COLS && B_COLS) {
            asm volatile(
                "ds_read_b64_tr_b16 %0, %24\n\t"
                "ds_read_b64_tr_b16 %1, %24 offset:2048\n\t"
                "ds_read_b64_tr_b16 %2, %25\n\t"
                "ds_read_b64_tr_b16 %3, %25 offset:2048\n\t"
                "ds_read_b64_tr_b16 %4, %26\n\t"
                "ds_read_b64_tr_b16 %5, %26 offset:2048\n\t"
                "ds_read_b64_tr_b16 %6, %27\n\t"
                "ds_read_b64_tr_b16 %7, %27 offset:2048\n\t"
                "ds_read_b64_tr_b16 %8, %28\n\t"
                "ds_read_b64_tr_b16 %9, %28 offset:2048\n\t"
                "ds_read_b64_tr_b16 %10, %29\n\t"
                "ds_read_b64_tr_b16 %11, %29 offset:2048\n\t"
                "ds_read_b64_tr_b16 %12, %24 offset:8192\n\t"
                "ds_read_b64_tr_b16 %13, %24 offset:10240\n\t"
                "ds_read_b64_tr_b16 %14, %25 offset:8192\n\t"
                "ds_read_b64_tr_b16 %15, %25 offset:10240\n\t"
                "ds_read_b64_tr_b16 %16, %26 offset:8192\n\t"
                "ds_read_b64_tr_b16 %17, %26 offset:10240\n\t"
                "ds_read_b64_tr_b16 %18, %27 offset:8192\n\t"
                "ds_read_b64_tr_b16 %19, %27 offset:10240\n\t"
                "ds_read_b64_tr_b16 %20, %28 offset:8192\n\t"
                "ds_read_b64_tr_b16 %21, %28 offset:10240\n\t"
                "ds_read_b64_tr_b16 %22, %29 offset:8192\n\t"
                "ds_read_b64_tr_b16 %23, %29 offset:10240\n\t"
                "s_waitcnt lgkmcnt(0)"
                : "=&v"(am[0][0][0]), "=&v"(am[0][0][1]), "=&v"(am[0][1][0]), "=&v"(am[0][1][1]), "=&v"(am[0][2][0]), "=&v"(am[0][2][1]),
                  "=&v"(am[0][3][0]), "=&v"(am[0][3][1]), "=&v"(bn[0][0][0]), "=&v"(bn[0][0][1]), "=&v"(bn[0][1][0]), "=&v"(bn[0][1][1]),
                  "=&v"(am[1][0][0]), "=&v"(am[1][0][1]), "=&v"(am[1][1][0]), "=&v"(am[1][1][1]), "=&v"(am[1][2][0]), "=&v"(am[1][2][1]),
                  "=&v"(am[1][3][0]), "=&v"(am[1][3][1]), "=&v"(bn[1][0][0]), "=&v"(bn[1][0][1]), "=&v"(bn[1][1][0]), "=&v"(bn[1][1][1])
                : "v"(a0), "v"(a1), "v"(a2), "v"(a3), "v"(b0), "v"(b1)
                : "memory");
        } else if constexpr (A_COLS) {
            asm volatile(
                "ds_read_b64_tr_b16 %0, %20\n\t"
                "ds_read_b64_tr_b16 %1, %20 offset:2048\n\t"
                "ds_read_b64_tr_b16 %2, %21\n\t"
                "ds_read_b64_tr_b16 %3, %21 offset:2048\n\t"
                "ds_read_b64_tr_b16 %4, %22\n\t"
                "ds_read_b64_tr_b16 %5, %22 offset:2048\n\t"
                "ds_read_b64_tr_b16 %6, %23\n\t"
                "ds_read_b64_tr_b16 %7, %23 offset:2048\n\t"
                "ds_read_b128 %8, %24\n\t"
                "ds_read_b128 %9, %24 offset:2048\n\t"
                "ds_read_b64_tr_b16 %10, %20 offset:8192\n\t"
                "ds_read_b64_tr_b16 %11, %20 offset:10240\n\t"
                "ds_read_b64_tr_b16 %12, %21 offset:8192\n\t"
                "ds_read_b64_tr_b16 %13, %21 offset:10240\n\t"
                "ds_read_b64_tr_b16 %14, %22 offset:8192\n\t"
                "ds_read_b64_tr_b16 %15, %22 offset:10240\n\t"
                "ds_read_b64_tr_b16 %16, %23 offset:8192\n\t"
                "ds_read_b64_tr_b16 %17, %23 offset:10240\n\t"
                "ds_read_b128 %18, %25\n\t"
                "ds_read_b128 %19, %25 offset:2048\n\t"
                "s_waitcnt lgkmcnt(0)"
                : "=&v"(am[0][0][0]), "=&v"(am[0][0][1]), "=&v"(am[0][1][0]), "=&v"(am[0][1][1]), "=&v"(am[0][2][0]), "=&v"(am[0][2][1]),
                  "=&v"(am[0][3][0]), "=&v"(am[0][3][1]), "=&v"(fn[0][0]), "=&v"(fn[0][1]), "=&v"(am[1][0][0]), "=&v"(am[1][0][1]),
                  "=&v"(am[1][1][0]), "=&v"(am[1][1][1]), "=&v"(am[1][2][0]), "=&v"(am[1][2][1]), "=&v"(am[1][3][0]), "=&v"(am[1][3][1]),
                  "=&v"(fn[1][0]), "=&v"(fn[1][1])
                : "v"(a0), "v"(a1), "v"(a2), "v"(a3), "v"(b0), "v"(b1)
                : "memory");
        } else if constexpr (B_COLS) {
            asm volatile(
                "ds_read_b128 %0, %16\n\t"
                "ds_read_b128 %1, %16 offset:2048\n\t"
                "ds_read_b128 %2, %16 offset:4096\n\t"
                "ds_read_b128 %3, %16 offset:6144\n\t"
                "ds_read_b64_tr_b16 %4, %18\n\t"
                "ds_read_b64_tr_b16 %5, %18 offset:2048\n\t"
                "ds_read_b64_tr_b16 %6, %19\n\t"
                "ds_read_b64_tr_b16 %7, %19 offset:2048\n\t"
                "ds_read_b128 %8, %17\n\t"
                "ds_read_b128 %9, %17 offset:2048\n\t"
                "ds_read_b128 %10, %17 offset:4096\n\t"
                "ds_read_b128 %11, %17 offset:6144\n\t"
                "ds_read_b64_tr_b16 %12, %18 offset:8192\n\t"
                "ds_read_b64_tr_b16 %13, %18 offset:10240\n\t"
                "ds_read_b64_tr_b16 %14, %19 offset:8192\n\t"
                "ds_read_b64_tr_b16 %15, %19 offset:10240\n\t"
                "s_waitcnt lgkmcnt(0)"
                : "=&v"(fm[0][0]), "=&v"(fm[0][1]), "=&v"(fm[0][2]), "=&v"(fm[0][3]), "=&v"(bn[0][0][0]), "=&v"(bn[0][0][1]),
                  "=&v"(bn[0][1][0]), "=&v"(bn[0][1][1]), "=&v"(fm[1][0]), "=&v"(fm[1][1]), "=&v"(fm[1][2]), "=&v"(fm[1][3]),
                  "=&v"(bn[1][0][0]), "=&v"(bn[1][0][1]), "=&v"(bn[1][1][0]), "=&v"(bn[1][1][1])
                : "v"(a0), "v"(a1), "v"(b0), "v"(b1)
                : "memory");
        } else {
            asm volatile(
                "ds_read_b128 %0, %12\n\t"
                "ds_read_b128 %1, %12 offset:2048\n\t"
                "ds_read_b128 %2, %12 offset:4096\n\t"
                "ds_read_b128 %3, %12 offset:6144\n\t"
                "ds_read_b128 %4, %14\n\t"
                "ds_read_b128 %5, %14 offset:2048\n\t"
                "ds_read_b128 %6, %13\n\t"
                "ds_read_b128 %7, %13 offset:2048\n\t"
                "ds_read_b128 %8, %13 offset:4096\n\t"
                "ds_read_b128 %9, %13 offset:6144\n\t"
                "ds_read_b128 %10, %15\n\t"
                "ds_read_b128 %11, %15 offset:2048\n\t"
                "s_waitcnt lgkmcnt(0)"
                : "=&v"(fm[0][0]), "=&v"(fm[0][1]), "=&v"(fm[0][2]), "=&v"(fm[0][3]), "=&v"(fn[0][0]), "=&v"(fn[0][1]), "=&v"(fm[1][0]),
                  "=&v"(fm[1][1]), "=&v"(fm[1][2]), "=&v"(fm[1][3]), "=&v"(fn[1][0]), "=&v"(fn[1][1])
                : "v"(a0), "v"(a1), "v"(b0), "v"(b1)
                : "memory");
        }
#pragma unroll
        for (int t = 0; t < 2; ++t) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if constexpr (A_COLS) fm[t][i] = Bytes16{am[t][i][0].x, am[t][i][0].y, am[t][i][1].x, am[t][i][1].y};
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                if constexpr (B_COLS) fn[t][j] = Bytes16{bn[t][j][0].x, bn[t][j][0].y, bn[t][j][1].x, bn[t][j][1].y};
            }
        }
    };
    auto compute = [&]() {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, fn[t][j]), __builtin_bit_cast(half8_t, fm[t][i]), acc[i][j], 0, 0, 0);
    };

    // The last chunk's elements from k = K on are the next row's: zeros instead, in both operands (they may be NaN or Inf).
    auto mask_tail = [&](int valid) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                const int left = valid - (t * 16 + h * 8 + d * 2);
                const unsigned mask = left >= 2 ? 0xffffffffu : (left == 1 ? 0xffffu : 0u);
#pragma unroll
                for (int i = 0; i < 4; ++i) fm[t][i][d] &= mask;
#pragma unroll
                for (int j = 0; j < 2; ++j) fn[t][j][d] &= mask;
            }
    };

    // ---- pipeline (the host guarantees nc >= AHEAD) ----
    const int nc = min(p.slice_chunks, (k_left + 31) / 32);
#pragma unroll
    for (int c = 0; c < AHEAD; ++c) issue(c);
    WaitVmcnt<(AHEAD - 1) * LPC>();  // this wave's share of chunk 0 has landed
    __builtin_amdgcn_s_barrier();
    if (!PAIR && grp == 1) __builtin_amdgcn_s_barrier();  // the second group runs half a period behind
    auto iteration = [&](int c, auto issue_tag, auto wait_tag) {
        constexpr bool ISSUE = decltype(issue_tag)::value;
        constexpr int WAIT = decltype(wait_tag)::value;
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (ISSUE) issue(c + AHEAD);  // into the stage that everyone finished reading a phase ago
        read_frags(c);
        if constexpr (!ISSUE && WAIT == 0) {
            if (c * 32 + 32 > k_left) mask_tail(k_left - c * 32);
        }
        WaitVmcnt<WAIT>();  // chunk c + 1 (this wave's share) must have landed before the barrier behind which it is read
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        compute();
        if constexpr (!PAIR) {
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    int c = 0;
    for (; c + AHEAD < nc; ++c) iteration(c, std::true_type{}, std::integral_constant<int, (AHEAD - 1) * LPC>{});
    // tail: nothing left to issue; with tt chunks behind c in flight, chunk c + 1 has landed when tt - 1 are outstanding
    StaticFor<0, AHEAD>([&](auto i_tag) {
        constexpr int tt = AHEAD - 1 - decltype(i_tag)::value;
        iteration(c, std::false_type{}, std::integral_constant<int, (tt >= 1 ? tt - 1 : 0) * LPC>{});
        ++c;
    });
    if (!PAIR && grp == 0) __builtin_amdgcn_s_barrier();

    // ---- epilogue: lane holds m = r, n = 8 * (v / 4) + 4 * h + v % 4 of each 32 x 32 block.  The blocks pass through LDS (a piece per wave, free now),
    // so that a row of 64 columns leaves in whole lines at any address: [4480,650] . [650,10000] 100 -> 94 us against 8-byte stores ----
    char* const mine = lds + wave * 32 * kOutPitch;
    float bias[2][16];
    if (p.bias != nullptr && p.slices == 1) {  // one load for the wave's 64 columns, then to where the lanes need them
        const int n = n0 + wn * 64 + lane;
        const float v = n < p.N ? static_cast<float>(p.bias[n * p.bias_stride]) : 0.f;
        __builtin_memcpy(mine + lane * 4, &v, 4);
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) __builtin_memcpy(&bias[j][q * 4], mine + (j * 32 + 8 * q + 4 * h) * 4, 16);
        __builtin_amdgcn_wave_barrier();
    }
    auto store = [&](auto tag, auto* c, int64_t ld) {
        using T = decltype(tag);
        constexpr int E = 16 / static_cast<int>(sizeof(T)), LANES = 64 / E, ROWS = 64 / LANES;  // lanes of a row, rows of an instruction
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    T o[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        float v = acc[i][j][q * 4 + e];
                        if constexpr (sizeof(T) == 2) {
                            if (p.bias != nullptr) v += bias[j][q * 4 + e];
                        }
                        o[e] = static_cast<T>(v);
                    }
                    __builtin_memcpy(mine + r * kOutPitch + (j * 32 + q * 8 + h * 4) * sizeof(T), o, sizeof(o));
                }
            __builtin_amdgcn_wave_barrier();
            const int n = n0 + wn * 64 + (lane % LANES) * E;
#pragma unroll
            for (int s = 0; s < 32 / ROWS; ++s) {
                const int row = s * ROWS + lane / LANES;
                const int m = m0 + wm * 128 + i * 32 + row;
                OutPiece<T> o;
                __builtin_memcpy(&o, mine + row * kOutPitch + (lane % LANES) * 16, 16);
                if (m < p.M) {
                    T* const to = c + static_cast<int64_t>(m) * ld + n;
                    if (n + E <= p.N) {
                        *reinterpret_cast<OutPiece<T>*>(to) = o;
                    } else {
#pragma unroll
                        for (int e = 0; e < E; ++e) {
                            if (n + e < p.N) to[e] = o.e[e];
                        }
                    }
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
    };
    if (p.slices > 1) store(float{}, p.partial + static_cast<int64_t>(slice) * p.M * p.N, p.N);
    else store(half_t{}, p.c, p.ldc);
}

// c = the sum of the slices (from the first on), plus the bias, rounded once.  Bound by memory: 8 columns of a row per thread.
__global__ __launch_bounds__(256) void GemmSumKernel(GemmArgs p) {
    const int groups = (p.N + 7) / 8;
    const int64_t g = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    const int64_t m = g / groups;
    const int n = static_cast<int>(g - m * groups) * 8;
    if (m >= p.M) return;
    const float* from = p.partial + m * p.N + n;
    const int64_t slice = static_cast<int64_t>(p.M) * p.N;
    half_t* const to = p.c + m * p.ldc + n;
    if (n + 8 <= p.N) {
        float sum[8] = {};
        for (int s = 0; s < p.slices; ++s, from += slice) {
            const OutPiece<float> lo = *reinterpret_cast<const OutPiece<float>*>(from), hi = *reinterpret_cast<const OutPiece<float>*>(from + 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) sum[e] += lo.e[e], sum[4 + e] += hi.e[e];
        }
        OutPiece<half_t> o;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (p.bias != nullptr) sum[e] += static_cast<float>(p.bias[(n + e) * p.bias_stride]);
            o.e[e] = static_cast<half_t>(sum[e]);
        }
        *reinterpret_cast<OutPiece<half_t>*>(to) = o;
    } else {
        for (int e = 0; n + e < p.N; ++e) {
            float sum = 0.f;
            for (int s = 0; s < p.slices; ++s) sum += from[s * slice + e];
            if (p.bias != nullptr) sum += static_cast<float>(p.bias[(n + e) * p.bias_stride]);
            to[e] = static_cast<half_t>(sum);
        }
    }
}
}  // namespace gemm_pp
}  // namespace hipcx
