// Matrix products with small outputs (batch-sized Linear layers, recurrent steps, weight gradients of small layers):
// out[M,N] = a[M,K] . b[K,N] with so few elements that 128x128 tiles would occupy a handful of compute units.
//
// A workgroup owns one 32x32 tile of `out` (SmallDotLinesKernel: 16 to 64 columns, SmallDotSquaresKernel: 64 x 32 to 64 x 80, SmallDotColumnsKernel: 64x64); its waves split the reduction
// axis -- and, with ksplit > 1, so do several workgroups, whose sums another kernel adds up -- each feeding the MFMA from global memory on its own
// (operands this small live in the caches), and the partial tiles are summed through LDS.  Six kernels, by where the operands lie (chosen in
// LaunchSmallDot, the last one in PlanSmallDot):
//   SmallDotKernel        k is the unit-stride axis of both operands (Linear's x and W^T): straight from global memory, bound by the
//                         latency of a few loads.
//   SmallDotLinesKernel   the same for more or longer tiles: whole 128-byte lines regrouped through LDS.
//   SmallDotSquaresKernel the same once 64 rows to a tile fill the chip: whole lines into LDS that the waves share.
//   SmallDotMixedKernel   an operand whose k axis is not the unit-stride one (dG . Wh of a recurrent network, x^T . gy).
//   SmallDotColumnsKernel float32, both operands with m and n as the unit-stride axes, of outputs that make a 64 x 64 tile per compute unit.
//   SmallDotVectorKernel  M <= 4 (one image, one sentence): a wave per output column, K across the lanes, where the MFMA would work on
//                         32 rows (float16: of few columns or many terms).
// For float the reduction index is dealt to the v_mfma_f32_32x32x2_f32 steps so that a lane's four steps use four consecutive k (one
// 16-byte load when k is the contiguous axis of the operand); for float16 a lane's v_mfma_f32_32x32x16_f16 operand is 8 consecutive k.
// Rows / columns beyond M / N and the tail of K are served as zeros by the buffer bounds check or explicit masks.
#pragma once

#include "igemm.h"

namespace hipcx {

constexpr int kSmallDotMaxBatch = 4;

struct SmallDotArgs {
    const void* a;
    const void* b;
    void* out;
    int M, N, K;
    int64_t a_row, a_k;  // element strides of a along m and k
    int64_t b_k, b_col;  // element strides of b along k and n
    int64_t o_row, o_col;
    unsigned a_bytes, b_bytes;  // spans, for the buffer descriptors
    int tiles_m, tiles_n;
    const void* bias;     // one element per column of out, added to the rounded product (Dot, then Add); may be null
    int64_t bias_stride;  // elements
    int nw;               // waves per workgroup = ways a workgroup's share of the reduction is split (SmallDotKernel: 8)
    int ksplit;           // workgroups per tile along the reduction
    float* partial;       // not null: [ksplit][M][N] sums go there instead of to out
    // blockIdx.y: products of one b that share their shapes and strides, left operands at a constant distance (elements), outputs
    // anywhere
    int64_t a_batch;
    void* outs[kSmallDotMaxBatch];
};

// Workgroups are dealt to the 8 XCDs round-robin, and each XCD has its own L2: give every XCD one contiguous range of
// tiles, row tiles fastest, so that the workgroups sharing a slice of b (the weights) share an L2 and the whole of b is
// fetched into the L2s once instead of once per XCD.
__device__ __forceinline__ void SmallDotTile(int nblk, int bid, int tiles_m, int& tm, int& tn) {
    const int xcd = bid & 7, loc = bid >> 3;
    const int q = nblk >> 3, r = nblk & 7;
    const int tile = xcd * q + min(xcd, r) + loc;
    tn = tile / tiles_m;
    tm = tile - tn * tiles_m;
}

// One element of the product, with the bias of a Linear layer: Dot rounds its result, then Add adds the bias and rounds again.
template <typename T>
__device__ __forceinline__ void StoreDot(const SmallDotArgs& p, T* out, int m, int n, float s) {
    T v = static_cast<T>(s);
    if (p.bias != nullptr) v = static_cast<T>(static_cast<float>(v) + static_cast<float>(static_cast<const T*>(p.bias)[n * p.bias_stride]));
    out[m * p.o_row + n * p.o_col] = v;
}

// Where an element of a tile goes.
template <typename T>
__device__ __forceinline__ void StoreTileElement(const SmallDotArgs& p, int split, T* out, int m, int n, float s) {
    if (p.partial != nullptr) {
        p.partial[(static_cast<int64_t>(split) * p.M + m) * p.N + n] = s;
    } else {
        StoreDot<T>(p, out, m, n, s);
    }
}

template <typename T>
struct SmallDotTraits;
template <>
struct SmallDotTraits<float> {
    static constexpr int KG = 8;  // k values one "group step" of a wave consumes (4 MFMAs x 2)
    static constexpr int PER_LANE = 4;
    static constexpr int STEPS_IN_FLIGHT = 3;  // per register stage (two stages)
};
template <>
struct SmallDotTraits<half_t> {
    static constexpr int KG = 16;  // one MFMA
    static constexpr int PER_LANE = 8;
    static constexpr int STEPS_IN_FLIGHT = 2;  // per register stage (two stages)
};

// The same run when k is the unit-stride axis, without a branch: lines beyond the operand come back as zeros from the
// buffer bounds check, elements beyond kend (they belong to the next line) are masked.  Loads written this way can all be
// issued before the first one is waited for.
template <typename T>
__device__ __forceinline__ Bytes16 LoadRunContig(__amdgpu_buffer_rsrc_t r, int64_t line_off, int k, int kend, bool line_ok) {
    constexpr int PL = SmallDotTraits<T>::PER_LANE;
    const int off = line_ok && k < kend ? static_cast<int>((line_off + k) * static_cast<int64_t>(sizeof(T))) : 0x7fffffff;
    Bytes16 v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
    const int c = kend - k;  // valid elements of the run (>= PL for all but the last run of a line)
    if constexpr (sizeof(T) == 4) {
        v.y = c > 1 ? v.y : 0u;
        v.z = c > 2 ? v.z : 0u;
        v.w = c > 3 ? v.w : 0u;
    } else {
        auto m = [c](int d) { return c > 2 * d + 1 ? 0xffffffffu : (c > 2 * d ? 0x0000ffffu : 0u); };
        v.x &= m(0);
        v.y &= m(1);
        v.z &= m(2);
        v.w &= m(3);
    }
    return v;
}

template <typename T>
__global__ __launch_bounds__(512) void SmallDotKernel(SmallDotArgs p) {
    constexpr int NW = 8;
    constexpr int KG = SmallDotTraits<T>::KG;
    constexpr int PL = SmallDotTraits<T>::PER_LANE;
    __shared__ float part[NW][32 * 33];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: the K loop below runs on scalar control flow
    const int lr = lane & 31;
    const int g = lane >> 5;
    int tm, tn;
    const int tiles = p.tiles_m * p.tiles_n;
    const int split = blockIdx.x / tiles;
    SmallDotTile(tiles, blockIdx.x - split * tiles, p.tiles_m, tm, tn);
    const int m = tm * 32 + lr;
    const int n = tn * 32 + lr;
    const int batch = blockIdx.y;
    const __amdgpu_buffer_rsrc_t ar = MakeRsrc(static_cast<const T*>(p.a) + batch * p.a_batch, p.a_bytes);
    const __amdgpu_buffer_rsrc_t br = MakeRsrc(p.b, p.b_bytes);
    const bool m_ok = m < p.M, n_ok = n < p.N;
    const int64_t a_off = static_cast<int64_t>(m) * p.a_row;
    const int64_t b_off = static_cast<int64_t>(n) * p.b_col;

    // this wave's share of K, in whole group steps
    const int groups = (p.K + KG - 1) / KG;
    const int per_split = (groups + p.ksplit - 1) / p.ksplit;
    const int split_end = min(groups, (split + 1) * per_split);
    const int per_wave = (per_split + NW - 1) / NW;
    const int k_begin = (split * per_split + wave * per_wave) * KG;
    const int k_end = min(p.K, min(split_end, split * per_split + (wave + 1) * per_wave) * KG);

    float16_t acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.f;
    constexpr int U = SmallDotTraits<T>::STEPS_IN_FLIGHT;
    {
        // Two register stages of U group steps: the loads of the next stage are issued before the MFMAs of the current one,
        // so that a wave's matrix work overlaps its own loads (all waves of a workgroup run in lockstep otherwise).
        // Stages made of whole runs inside K need no masking, so nothing but the MFMAs depends on a load and the waits
        // land where the data is consumed; the (masked) remainder of a wave's share is done afterwards.
        Bytes16 av[2][U], bv[2][U];
        const int a_base = m_ok ? static_cast<int>(a_off * static_cast<int64_t>(sizeof(T))) : 0x7fffffff;
        const int b_base = n_ok ? static_cast<int>(b_off * static_cast<int64_t>(sizeof(T))) : 0x7fffffff;
        auto load_stage = [&](int st, int k) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int koff = (k + u * KG + g * PL) * static_cast<int>(sizeof(T));
                av[st][u] = __builtin_amdgcn_raw_buffer_load_b128(ar, m_ok ? a_base + koff : 0x7fffffff, 0, 0);
                bv[st][u] = __builtin_amdgcn_raw_buffer_load_b128(br, n_ok ? b_base + koff : 0x7fffffff, 0, 0);
            }
        };
        auto mfma_stage = [&](int st) {
#pragma unroll
            for (int u = 0; u < U; ++u) MfmaTile<T>(av[st][u], bv[st][u], acc);
        };
        constexpr int STEP = U * KG;
        const int nfull = k_end > k_begin ? (k_end - k_begin) / STEP : 0;  // stages whose every run ends inside K
        int k = k_begin;
        if (nfull > 0) {
            // The steady-state body has no conditional loads: the wait in front of a stage's MFMAs then only covers that
            // stage (the other stage's loads, issued later, stay in flight).  One or two stages are left for after the loop.
            load_stage(0, k);
            int i = 0;
            for (; i + 2 <= nfull - 1; i += 2) {
                load_stage(1, k + STEP);
                mfma_stage(0);
                load_stage(0, k + 2 * STEP);
                mfma_stage(1);
                k += 2 * STEP;
            }
            if (nfull - i == 2) {
                load_stage(1, k + STEP);
                mfma_stage(0);
                mfma_stage(1);
            } else {
                mfma_stage(0);
            }
            k = k_begin + nfull * STEP;
        }
        for (; k < k_end; k += KG) {
            const int kk = k + g * PL;
            Bytes16 ta = LoadRunContig<T>(ar, a_off, kk, k_end, m_ok);
            Bytes16 tb = LoadRunContig<T>(br, b_off, kk, k_end, n_ok);
            MfmaTile<T>(ta, tb, acc);
        }
    }
    // lane holds column lr, rows 8*(v/4) + 4*g + v%4
#pragma unroll
    for (int v = 0; v < 16; ++v) part[wave][(8 * (v / 4) + 4 * g + (v % 4)) * 33 + lr] = acc[v];
    __syncthreads();
    T* out = static_cast<T*>(gridDim.y > 1 ? p.outs[batch] : p.out);
    for (int e = tid; e < 32 * 32; e += 512) {
        int row = e >> 5, col = e & 31;
        float s = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) s += part[w][row * 33 + col];
        int om = tm * 32 + row, on = tn * 32 + col;
        if (om < p.M && on < p.N) StoreTileElement<T>(p, split, out, om, on, s);
    }
}

// How SmallDotMixedKernel reads an operand.  kPieces: rows of contiguous k as 16-byte pieces; kElements: another axis is the unit-stride
// one, element by element with that axis across the lanes -- whole lines too, already in the MFMA layout; kOddPieces: float16 rows of odd
// pitch, whose last elements share a dword with what lies behind the array: pieces, but the chunk that holds the end of K by elements.
enum SmallDotMode { kPieces, kElements, kOddPieces };

constexpr int kSmallDotMaxWaves = 8;
constexpr int kSmallDotPart = 32 * 33;  // floats of a wave's partial tile

constexpr int kSmallDotPitch = 144;  // bytes of a row staged in LDS: the 16-byte reads of 8 consecutive rows start in different banks
constexpr int kSmallDotStage = 32 * kSmallDotPitch;

// One lane's share of a chunk of an operand: P pieces of 16 bytes.
template <int P>
struct SmallDotShare {
    Bytes16 v[P];
};

// PL consecutive elements of k at byte `line` (negative: a row beyond the operand).  WHOLE: as one load, which may reach beyond K.
template <typename T, bool WHOLE>
__device__ __forceinline__ Bytes16 LoadPiece(__amdgpu_buffer_rsrc_t r, int line, int k_stride_bytes, int k, int K) {
    constexpr int PL = 16 / sizeof(T);
    constexpr int kOut = 0x7fffffff;
    if constexpr (WHOLE) {
        return __builtin_amdgcn_raw_buffer_load_b128(r, line >= 0 && k < K ? line + k * static_cast<int>(sizeof(T)) : kOut, 0, 0);
    } else {
        Bytes16 v;
        if constexpr (sizeof(T) == 4) {
#pragma unroll
            for (int e = 0; e < PL; ++e) v[e] = __builtin_amdgcn_raw_buffer_load_b32(r, line >= 0 && k + e < K ? line + (k + e) * k_stride_bytes : kOut, 0, 0);
        } else {
            unsigned short s[PL];
#pragma unroll
            for (int e = 0; e < PL; ++e) s[e] = __builtin_amdgcn_raw_buffer_load_b16(r, line >= 0 && k + e < K ? line + (k + e) * k_stride_bytes : kOut, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = s[2 * e] | (static_cast<unsigned>(s[2 * e + 1]) << 16);
        }
        return v;
    }
}

// The first K - k elements of a piece, zeros in place of what follows K in the memory of a row.
template <typename T>
__device__ __forceinline__ Bytes16 MaskPiece(Bytes16 v, int k, int K) {
    constexpr int PD = 4 / sizeof(T);  // elements per dword
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        const int left = K - (k + d * PD);
        v[d] = left >= PD ? v[d] : (left == 1 && PD == 2 ? v[d] & 0xffffu : 0u);
    }
    return v;
}

// A piece that reaches beyond the end of its row is read from the row's last 16 bytes instead: rows may then start and end anywhere, as long as they are 16
// bytes long.  Elements by which that is early, of the piece at `k`; they are another piece's.
template <typename T>
__device__ __forceinline__ int PieceEarly(int k, int K) {
    return max(0, k - (K - static_cast<int>(16 / sizeof(T))));
}
// The piece without them.
template <typename T>
__device__ __forceinline__ Bytes16 KeepPiece(Bytes16 v, int early) {
    constexpr int PL = 16 / sizeof(T);
    using Piece = __attribute__((ext_vector_type(PL))) std::conditional_t<sizeof(T) == 4, unsigned, unsigned short>;
    Piece e = __builtin_bit_cast(Piece, v);
#pragma unroll
    for (int i = 0; i < PL; ++i) e[i] = i < early ? 0 : e[i];
    return __builtin_bit_cast(Bytes16, e);
}

// 16 x 16 outputs from 16 bytes of 16 rows of a and b, the k of a piece in any order as long as both operands keep to it.
template <typename T>
__device__ __forceinline__ void MfmaBlock(const Bytes16& a, const Bytes16& b, float4_t& acc) {
    if constexpr (sizeof(T) == 2) {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, a), __builtin_bit_cast(half8_t, b), acc, 0, 0, 0);
    } else {
        const float4_t af = __builtin_bit_cast(float4_t, a), bf = __builtin_bit_cast(float4_t, b);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(af[e], bf[e], acc, 0, 0, 0);
    }
}

// Both operands in pieces; tiles of 32 rows and 16 * NB columns.  A wave takes chunks of 128 bytes per row: whole lines (8 lanes to a row, 8 rows to an
// instruction), turned round in LDS of its own.  Two chunks are in flight while a third is multiplied; the loads' offsets are constants plus a scalar, and
// only the chunk that holds the end of K looks at it.  Bound by the matrix pipe and by the delivery of operands (64 rows for 1024 outputs) in about equal
// parts, and by tiles that are not dealt out evenly: hence the widths.  us, against one chunk in flight and three or more waves to a tile: float32
// [1024,1024]^2 33.4 -> 26.7, [1000,784] . [784,1000] 27.4 -> 22.5, [256,1024] . [1024,1024] 11.4 -> 9.4 (against SmallDotKernel); float16 15.4 -> 10.7,
// 13.3 -> 11.2, 6.6 -> 5.0, [37,2048] . [2048,1000] 9.8 -> 5.1.
template <typename T, int NB>
__global__ __launch_bounds__(64 * kSmallDotMaxWaves) __attribute__((amdgpu_waves_per_eu(2, 8))) void SmallDotLinesKernel(SmallDotArgs p) {
    constexpr int PL = 16 / sizeof(T);
    constexpr int KC = 8 * PL;  // k per chunk
    constexpr int kOut = 0x7fffffff;
    constexpr int BL = 2 * NB;  // loads of b per chunk, 8 rows each
    constexpr int kStage = (32 + 16 * NB) * kSmallDotPitch, kPitch = 16 * NB + 1;
    extern __shared__ __align__(16) char lds[];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: the loop below runs on scalar control flow
    const int lr = lane & 15;
    const int g = lane >> 4;
    const int piece = lane & 7, sub = lane >> 3;
    const int tiles = p.tiles_m * p.tiles_n;
    const int split = blockIdx.x / tiles;
    int tm, tn;
    SmallDotTile(tiles, blockIdx.x - split * tiles, p.tiles_m, tm, tn);
    const int batch = blockIdx.y;
    const __amdgpu_buffer_rsrc_t ar = MakeRsrc(static_cast<const T*>(p.a) + batch * p.a_batch, p.a_bytes);
    const __amdgpu_buffer_rsrc_t br = MakeRsrc(p.b, p.b_bytes);
    int a_line[4], b_line[BL];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int m = tm * 32 + j * 8 + sub;
        a_line[j] = m < p.M ? static_cast<int>((m * p.a_row + piece * PL) * static_cast<int64_t>(sizeof(T))) : kOut;
    }
#pragma unroll
    for (int j = 0; j < BL; ++j) {
        const int n = tn * 16 * NB + j * 8 + sub;
        b_line[j] = n < p.N ? static_cast<int>((n * p.b_col + piece * PL) * static_cast<int64_t>(sizeof(T))) : kOut;
    }
    char* const a_stage = lds + wave * kStage;
    char* const to = a_stage + sub * kSmallDotPitch + piece * 16;
    const char* const from = a_stage + lr * kSmallDotPitch + g * 16;

    // this wave's chunks
    const int chunks = (p.K + KC - 1) / KC;
    const int per_split = (chunks + p.ksplit - 1) / p.ksplit;
    const int s_begin = split * per_split, s_end = min(chunks, s_begin + per_split);
    const int per_wave = (max(s_end - s_begin, 0) + p.nw - 1) / p.nw;
    const int begin = s_begin + wave * per_wave, end = min(s_end, begin + per_wave);

    float4_t acc[2][NB];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
    Bytes16 av[2][4], bv[2][BL];
    auto load = [&](int st, int c) {
        if ((c + 1) * KC <= p.K) {
#pragma unroll
            for (int j = 0; j < 4; ++j) av[st][j] = __builtin_amdgcn_raw_buffer_load_b128(ar, a_line[j], c * 128, 0);
#pragma unroll
            for (int j = 0; j < BL; ++j) bv[st][j] = __builtin_amdgcn_raw_buffer_load_b128(br, b_line[j], c * 128, 0);
        } else {
            int at = c * 128;
            bool in = true;
            if constexpr (sizeof(T) == 2) at -= PieceEarly<T>(c * KC + piece * PL, p.K) * static_cast<int>(sizeof(T));
            else in = c * KC + piece * PL < p.K;  // (rows of whole dwords: pieces beyond K are not read, what lies behind it in one is masked)
#pragma unroll
            for (int j = 0; j < 4; ++j) av[st][j] = __builtin_amdgcn_raw_buffer_load_b128(ar, (in & (a_line[j] != kOut)) ? a_line[j] + at : kOut, 0, 0);
#pragma unroll
            for (int j = 0; j < BL; ++j) bv[st][j] = __builtin_amdgcn_raw_buffer_load_b128(br, (in & (b_line[j] != kOut)) ? b_line[j] + at : kOut, 0, 0);
        }
    };
    auto multiply = [&](int st, int c, auto&& next) {
        if ((c + 1) * KC > p.K) {
            auto keep = [&](Bytes16 v) {
                // float32 by masks: by early pieces it takes 146 registers with two blocks, not 128, and a compute unit has no room for a second workgroup of eight waves
                // ([135,896] . [896,3209] 13.8 us, 16.3)
                if constexpr (sizeof(T) == 2) return KeepPiece<T>(v, PieceEarly<T>(c * KC + piece * PL, p.K));
                else return MaskPiece<T>(v, c * KC + piece * PL, p.K);
            };
#pragma unroll
            for (int j = 0; j < 4; ++j) av[st][j] = keep(av[st][j]);
#pragma unroll
            for (int j = 0; j < BL; ++j) bv[st][j] = keep(bv[st][j]);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) *reinterpret_cast<Bytes16*>(to + j * 8 * kSmallDotPitch) = av[st][j];
#pragma unroll
        for (int j = 0; j < BL; ++j) *reinterpret_cast<Bytes16*>(to + kSmallDotStage + j * 8 * kSmallDotPitch) = bv[st][j];
        next();
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int q = 0; q < 2; ++q) {  // pieces g and g + 4 of each row
            Bytes16 fa[2], fb[NB];
#pragma unroll
            for (int i = 0; i < 2; ++i) fa[i] = *reinterpret_cast<const Bytes16*>(from + i * 16 * kSmallDotPitch + q * 64);
#pragma unroll
            for (int j = 0; j < NB; ++j) fb[j] = *reinterpret_cast<const Bytes16*>(from + kSmallDotStage + j * 16 * kSmallDotPitch + q * 64);
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < NB; ++j) MfmaBlock<T>(fa[i], fb[j], acc[i][j]);
        }
        __builtin_amdgcn_wave_barrier();
    };
    if (begin < end) {
        load(0, begin);
        if (begin + 1 < end) load(1, begin + 1);
        int c = begin;
        for (; c + 3 < end; c += 2) {
            multiply(0, c, [&] { load(0, c + 2); });
            multiply(1, c + 1, [&] { load(1, c + 3); });
        }
        // one, two or three are left
        multiply(0, c, [&] {
            if (c + 2 < end) load(0, c + 2);
        });
        if (c + 1 < end) multiply(1, c + 1, [] {});
        if (c + 2 < end) multiply(0, c + 2, [] {});
    }
    __syncthreads();  // the staging areas become the partial tiles
    // lane holds column lr, rows 4 * g + v of each block
    constexpr int kPart = 32 * kPitch;
    float* const part = reinterpret_cast<float*>(lds);
    float* const mine = part + wave * kPart;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) mine[(i * 16 + 4 * g + v) * kPitch + j * 16 + lr] = acc[i][j][v];
    __syncthreads();
    T* out = static_cast<T*>(gridDim.y > 1 ? p.outs[batch] : p.out);
    for (int e = tid; e < 32 * 16 * NB; e += 64 * p.nw) {
        const int row = e / (16 * NB), col = e - row * (16 * NB);
        const int om = tm * 32 + row, on = tn * 16 * NB + col;
        if (om >= p.M || on >= p.N) continue;
        float s = 0.f;
        for (int w = 0; w < p.nw; ++w) s += part[w * kPart + row * kPitch + col];
        StoreTileElement<T>(p, split, out, om, on, s);
    }
}

// Tiles of 64 rows and 16 * NB columns, both operands in pieces.  The eight waves take 32 rows each of a quarter of a chunk's k; chunks of 256 bytes per
// row go through LDS that they share (two buffers, one barrier a chunk): while one is multiplied, the fragments of the next come out of LDS, the one after
// goes there, and one more is on its way.  A chunk's products start from zero and are
// added up by chunk, so that a chain is 16 terms: the error is half of that of tiles whose waves add up all of their terms ([128,650] . [650,10000] 1.07e-7 of the
// norm, 2.68e-7; [670,3324] . [3324,2007] 1.6e-7, 7.3e-7).  Bound by the matrix pipe, 1.2 us of a chunk's 1.5 at five blocks, and by 5 us of launch, first loads
// and sums; fragments read twice as often (16 rows to a wave) or what is not a product after the products, instead of between them, cost 3 us of 25.
// Against SmallDotLinesKernel: float32 [128,650] . [650,10000] 28.1 -> 24.8 us (11.5 of matrix work), [1000,784] . [784,1000] 24.2 -> 22.3, float16
// [1903,2408] . [2408,452] 28.6 -> 19.7.
constexpr int kSquaresPitch = 256 + 16;  // bytes of a row in LDS: 16 rows' pieces start in different banks
template <typename T, int NB>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void SmallDotSquaresKernel(SmallDotArgs p) {
    constexpr int PL = 16 / sizeof(T);
    constexpr int KC = 16 * PL;  // k per chunk
    constexpr int kOut = 0x7fffffff;
    constexpr int BL = (NB + 1) / 2;  // loads of b per chunk and thread, 32 rows each in all
    constexpr int kStage = (64 + 32 * BL) * kSquaresPitch, kPitch = 16 * NB + 1;
    extern __shared__ __align__(16) char lds[];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, g = lane >> 4;
    int tm, tn;
    SmallDotTile(p.tiles_m * p.tiles_n, blockIdx.x, p.tiles_m, tm, tn);
    const __amdgpu_buffer_rsrc_t ar = MakeRsrc(static_cast<const T*>(p.a), p.a_bytes);
    const __amdgpu_buffer_rsrc_t br = MakeRsrc(p.b, p.b_bytes);
    const int row_in = tid >> 4, k_in = (tid & 15) * PL;  // of this thread's loads
    int a_line[2], b_line[BL];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int m = tm * 64 + j * 32 + row_in;
        a_line[j] = m < p.M ? static_cast<int>((m * p.a_row + k_in) * static_cast<int64_t>(sizeof(T))) : kOut;
    }
#pragma unroll
    for (int j = 0; j < BL; ++j) {
        const int row = j * 32 + row_in, n = tn * 16 * NB + row;
        b_line[j] = row < 16 * NB && n < p.N ? static_cast<int>((n * p.b_col + k_in) * static_cast<int64_t>(sizeof(T))) : kOut;
    }
    char* const to = lds + row_in * kSquaresPitch + (tid & 15) * 16;
    const int rows = wave & 1, quarter = wave >> 1;
    const char* const from = lds + lr * kSquaresPitch + quarter * 64 + g * 16;

    float4_t acc[2][NB], terms[2][NB];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = terms[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
    const int chunks = (p.K + KC - 1) / KC;
    Bytes16 av[2], bv[BL], fa[2][2], fb[2][NB];
    auto load = [&](int c) {
        int at = c * 256;
        bool in = true;
        if constexpr (sizeof(T) == 2) at -= PieceEarly<T>(c * KC + k_in, p.K) * static_cast<int>(sizeof(T));
        else in = c * KC + k_in < p.K;  // (their rows are whole dwords: what lies behind them is masked, what is behind the array reads as zeros)
#pragma unroll
        for (int j = 0; j < 2; ++j) av[j] = __builtin_amdgcn_raw_buffer_load_b128(ar, (in & (a_line[j] != kOut)) ? a_line[j] + at : kOut, 0, 0);
#pragma unroll
        for (int j = 0; j < BL; ++j) bv[j] = __builtin_amdgcn_raw_buffer_load_b128(br, (in & (b_line[j] != kOut)) ? b_line[j] + at : kOut, 0, 0);
    };
    auto store = [&](int c, auto whole) {
        if (!decltype(whole)::value && (c + 1) * KC > p.K) {
            auto keep = [&](Bytes16 v) {
                if constexpr (sizeof(T) == 2) return KeepPiece<T>(v, PieceEarly<T>(c * KC + k_in, p.K));
                else return MaskPiece<T>(v, c * KC + k_in, p.K);
            };
#pragma unroll
            for (int j = 0; j < 2; ++j) av[j] = keep(av[j]);
#pragma unroll
            for (int j = 0; j < BL; ++j) bv[j] = keep(bv[j]);
        }
        char* const at = to + (c & 1) * kStage;
#pragma unroll
        for (int j = 0; j < 2; ++j) *reinterpret_cast<Bytes16*>(at + j * 32 * kSquaresPitch) = av[j];
#pragma unroll
        for (int j = 0; j < BL; ++j) *reinterpret_cast<Bytes16*>(at + (64 + j * 32) * kSquaresPitch) = bv[j];
    };
    auto read = [&](int st, int c) {
        const char* const at = from + (c & 1) * kStage;
#pragma unroll
        for (int i = 0; i < 2; ++i) fa[st][i] = *reinterpret_cast<const Bytes16*>(at + (rows * 32 + i * 16) * kSquaresPitch);
#pragma unroll
        for (int j = 0; j < NB; ++j) fb[st][j] = *reinterpret_cast<const Bytes16*>(at + (64 + j * 16) * kSquaresPitch);
    };
    // `whole`: c + 2 lies inside K
    auto step = [&](auto parity, int c, auto whole) {
        constexpr int S = decltype(parity)::value;
        constexpr bool kWhole = decltype(whole)::value;
        read(S ^ 1, c + 1);
        store(c + 2, whole);
        load(c + 3);
        if (kWhole || c * KC + quarter * (KC / 4) < p.K) {
#pragma unroll
            for (int e = 0; e < (sizeof(T) == 4 ? 4 : 1); ++e)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < NB; ++j) {
                        if (e == 0) {  // the chunk before's
                            acc[i][j] += terms[i][j];
                            terms[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
                        }
                        if constexpr (sizeof(T) == 4) {
                            terms[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(fa[S][i][e]), __uint_as_float(fb[S][j][e]), terms[i][j], 0, 0, 0);
                        } else {
                            MfmaBlock<T>(fa[S][i], fb[S][j], terms[i][j]);
                        }
                    }
        }
        if constexpr (kWhole) {  // what is not a product goes between them, under the matrix pipe
            constexpr int kProducts = sizeof(T) == 4 && NB >= 4 ? 2 : 1;
#pragma unroll
            for (int i = 0; i < 2 + NB; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x8, kProducts, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
#pragma unroll
            for (int i = 0; i < 2 + BL; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x8, kProducts, 0);
                __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
            }
#pragma unroll
            for (int i = 0; i < 2 + BL; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x8, kProducts, 0);
                __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);
            }
        }
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
    };
    load(0);
    store(0, std::false_type{});
    load(1);
    __syncthreads();
    read(0, 0);
    store(1, std::false_type{});
    load(2);
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    int c = 0;
    for (; (c + 4) * KC <= p.K; c += 2) {
        step(std::integral_constant<int, 0>{}, c, std::true_type{});
        step(std::integral_constant<int, 1>{}, c + 1, std::true_type{});
    }
    for (; c < chunks; c += 2) {
        step(std::integral_constant<int, 0>{}, c, std::false_type{});
        if (c + 1 < chunks) step(std::integral_constant<int, 1>{}, c + 1, std::false_type{});
    }
    // lane holds column lr, rows 4 * g + v of each block
    constexpr int kPart = 64 * kPitch;
    float* const part = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) part[quarter * kPart + (rows * 32 + i * 16 + 4 * g + v) * kPitch + j * 16 + lr] = acc[i][j][v] + terms[i][j][v];
    __syncthreads();
    T* const out = static_cast<T*>(p.out);
    for (int e = tid; e < 64 * 16 * NB; e += 512) {
        const int row = e / (16 * NB), col = e - row * (16 * NB);
        const int om = tm * 64 + row, on = tn * 16 * NB + col;
        if (om >= p.M || on >= p.N) continue;
        const float* const s = part + row * kPitch + col;
        StoreDot<T>(p, out, om, on, (s[0] + s[kPart]) + (s[2 * kPart] + s[3 * kPart]));
    }
}

// At least one operand element by element.  The reduction is dealt out in chunks of 32 bytes per row, which come as they are used, six of them in flight, or, where
// the other operand's are float16 rows of odd pitch, of 128 bytes, two in flight: these are loaded as whole lines and turned round through a piece of LDS that
// belongs to the wave (no barrier).  [20,2600] . [2600,650] float32, row-major b: 34 -> 9.3 us (several workgroups per tile and the pass over their sums included).
template <typename T, int AM, int BM>
__global__ __launch_bounds__(64 * kSmallDotMaxWaves) __attribute__((amdgpu_waves_per_eu(3, 8))) void SmallDotMixedKernel(SmallDotArgs p) {
    static_assert(AM == kElements || BM == kElements);
    constexpr int PL = 16 / sizeof(T);
    constexpr bool A_LDS = AM == kOddPieces, B_LDS = BM == kOddPieces;
    constexpr int P = A_LDS || B_LDS ? 4 : 1;
    constexpr int KC = 2 * P * PL;      // k per chunk
    constexpr int D = P == 1 ? 6 : 2;   // chunks in flight
    extern __shared__ __align__(16) char lds[];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: the loop below runs on scalar control flow
    const int lr = lane & 31;
    const int g = lane >> 5;
    const int piece = lane & 7, sub = lane >> 3;
    const int tiles = p.tiles_m * p.tiles_n;
    const int split = blockIdx.x / tiles;
    int tm, tn;
    SmallDotTile(tiles, blockIdx.x - split * tiles, p.tiles_m, tm, tn);
    const int batch = blockIdx.y;
    const __amdgpu_buffer_rsrc_t ar = MakeRsrc(static_cast<const T*>(p.a) + batch * p.a_batch, p.a_bytes);
    const __amdgpu_buffer_rsrc_t br = MakeRsrc(p.b, p.b_bytes);
    const int a_ks = static_cast<int>(p.a_k * sizeof(T)), b_ks = static_cast<int>(p.b_k * sizeof(T));
    // rows this lane reads: in the MFMA layout its own (lr), as whole lines every eighth one
    auto line_of = [](int row, int rows, int64_t stride) { return row < rows ? static_cast<int>(row * stride * static_cast<int64_t>(sizeof(T))) : -1; };
    int a_line[4], b_line[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        a_line[j] = line_of(tm * 32 + (A_LDS ? j * 8 + sub : lr), p.M, p.a_row);
        b_line[j] = line_of(tn * 32 + (B_LDS ? j * 8 + sub : lr), p.N, p.b_col);
    }
    char* const stage = lds + wave * kSmallDotStage;

    // this wave's chunks
    const int chunks = (p.K + KC - 1) / KC;
    const int per_split = (chunks + p.ksplit - 1) / p.ksplit;
    const int s_begin = split * per_split, s_end = min(chunks, s_begin + per_split);
    const int per_wave = (max(s_end - s_begin, 0) + p.nw - 1) / p.nw;
    const int begin = s_begin + wave * per_wave, end = min(s_end, begin + per_wave);

    float16_t acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.f;
    SmallDotShare<P> av[D], bv[D];
    auto load_operand = [&](auto mode_tag, SmallDotShare<P>& x, __amdgpu_buffer_rsrc_t r, const int (&line)[4], int ks, int c) {
        constexpr int MODE = decltype(mode_tag)::value;
        constexpr bool LDS = MODE == kOddPieces;
        const int k0 = c * KC + (LDS ? piece * PL : g * P * PL);
        if (MODE == kPieces || (MODE == kOddPieces && (c + 1) * KC <= p.K)) {
#pragma unroll
            for (int j = 0; j < P; ++j) x.v[j] = LoadPiece<T, true>(r, line[LDS ? j : 0], ks, k0 + (LDS ? 0 : j * PL), p.K);
        } else {
#pragma unroll
            for (int j = 0; j < P; ++j) x.v[j] = LoadPiece<T, false>(r, line[LDS ? j : 0], ks, k0 + (LDS ? 0 : j * PL), p.K);
        }
    };
    auto load = [&](int i, int c) {
        load_operand(std::integral_constant<int, AM>{}, av[i], ar, a_line, a_ks, c);
        load_operand(std::integral_constant<int, BM>{}, bv[i], br, b_line, b_ks, c);
    };
    // the chunk in the MFMA layout: lane (lr, g) holds pieces g * P .. of its row
    auto arrange = [&](auto mode_tag, SmallDotShare<P>& x, int c) {
        constexpr int MODE = decltype(mode_tag)::value;
        if (MODE == kPieces && (c + 1) * KC > p.K) x.v[0] = MaskPiece<T>(x.v[0], c * KC + g * PL, p.K);
        if constexpr (MODE == kOddPieces) {
#pragma unroll
            for (int j = 0; j < P; ++j) *reinterpret_cast<Bytes16*>(stage + (j * 8 + sub) * kSmallDotPitch + piece * 16) = x.v[j];
        }
    };
    auto fragment = [&](bool in_lds, const SmallDotShare<P>& x, int j) {
        return in_lds ? *reinterpret_cast<const Bytes16*>(stage + lr * kSmallDotPitch + (g * P + j) * 16) : x.v[j];
    };
    auto multiply = [&](int i, int c, auto&& next) {
        arrange(std::integral_constant<int, AM>{}, av[i], c);
        arrange(std::integral_constant<int, BM>{}, bv[i], c);
        if constexpr (A_LDS || B_LDS) __builtin_amdgcn_wave_barrier();
        Bytes16 fa[P], fb[P];
#pragma unroll
        for (int j = 0; j < P; ++j) {
            fa[j] = fragment(A_LDS, av[i], j);
            fb[j] = fragment(B_LDS, bv[i], j);
        }
        if constexpr (A_LDS || B_LDS) __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int j = 0; j < P; ++j) MfmaTile<T>(fa[j], fb[j], acc);
        next();  // (into the registers that were this chunk's fragments)
    };
    if (begin < end) {
#pragma unroll
        for (int i = 0; i < D; ++i) {
            if (begin + i < end) load(i, begin + i);
        }
        int c = begin;
        // no conditional loads while a whole round of them is left: the waits then cover one chunk, not what was issued behind it
        for (; c + 2 * D <= end; c += D) {
#pragma unroll
            for (int i = 0; i < D; ++i) multiply(i, c + i, [&] { load(i, c + i + D); });
        }
        if (c + D < end) {
#pragma unroll
            for (int i = 0; i < D; ++i) {
                multiply(i, c + i, [&] {
                    if (c + i + D < end) load(i, c + i + D);
                });
            }
            c += D;
        }
#pragma unroll
        for (int i = 0; i < D; ++i) {
            if (c + i < end) multiply(i, c + i, [] {});
        }
    }
    if constexpr (A_LDS || B_LDS) __syncthreads();  // the staging areas become the partial tiles
    // lane holds column lr, rows 8*(v/4) + 4*g + v%4
    float* const part = reinterpret_cast<float*>(lds);
    float* const mine = part + wave * kSmallDotPart;
#pragma unroll
    for (int v = 0; v < 16; ++v) mine[(8 * (v / 4) + 4 * g + (v % 4)) * 33 + lr] = acc[v];
    __syncthreads();
    T* out = static_cast<T*>(gridDim.y > 1 ? p.outs[batch] : p.out);
    for (int e = tid; e < 32 * 32; e += 64 * p.nw) {
        const int row = e >> 5, col = e & 31;
        const int om = tm * 32 + row, on = tn * 32 + col;
        if (om >= p.M || on >= p.N) continue;
        float s = 0.f;
        for (int w = 0; w < p.nw; ++w) s += part[w * kSmallDotPart + row * 33 + col];
        StoreTileElement<T>(p, split, out, om, on, s);
    }
}

// float32, both operands k by k with m and n dense (weight gradients x^T . gy): tiles of 64 x 64 by four waves that split the reduction.  A lane's 16 bytes of
// one k are a term each of four v_mfma_f32_16x16x4_f32 operands whose rows are every fourth one: lines arrive whole, in the order the MFMA takes them,
// without LDS.  Bound by the float pipe.  us, against elements in tiles of
// 32 x 32: [700,2600]^T . [700,650] 43 -> 34, [1000,1000]^T . [1000,1000] 34 -> 30, [100,1000]^T . [100,1000] 10.0 -> 8.1.
template <typename T>
__global__ __launch_bounds__(256, 2) void SmallDotColumnsKernel(SmallDotArgs p) {
    static_assert(sizeof(T) == 4);
    constexpr int U = 4, KC = 4 * U;  // loads of an operand and k per stage
    constexpr int kOut = 0x7fffffff;
    constexpr int kPitch = 64 + 4, kPart = 64 * kPitch;
    extern __shared__ __align__(16) char lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int tiles = p.tiles_m * p.tiles_n;
    const int split = blockIdx.x / tiles;
    int tm, tn;
    SmallDotTile(tiles, blockIdx.x - split * tiles, p.tiles_m, tm, tn);
    const int batch = blockIdx.y;
    const __amdgpu_buffer_rsrc_t ar = MakeRsrc(static_cast<const float*>(p.a) + batch * p.a_batch, p.a_bytes);
    const __amdgpu_buffer_rsrc_t br = MakeRsrc(p.b, p.b_bytes);
    const int m = tm * 64 + 4 * r, n = tn * 64 + 4 * r;
    const unsigned a_step = static_cast<unsigned>(p.a_k * 4), b_step = static_cast<unsigned>(p.b_k * 4);

    const int chunks = (p.K + KC - 1) / KC;
    const int per_split = (chunks + p.ksplit - 1) / p.ksplit;
    const int end = min(chunks, (split + 1) * per_split);
    float4_t acc[4][4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int f = 0; f < 4; ++f) acc[e][f] = float4_t{0.f, 0.f, 0.f, 0.f};
    Bytes16 av[2][U], bv[2][U];
    auto load = [&](int st, int c) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = c * KC + u * 4 + g;
            const bool in = (k < p.K) & (c < end);
            av[st][u] = __builtin_amdgcn_raw_buffer_load_b128(ar, (in & (m < p.M)) ? static_cast<int>(k * a_step + m * 4) : kOut, 0, 0);
            bv[st][u] = __builtin_amdgcn_raw_buffer_load_b128(br, (in & (n < p.N)) ? static_cast<int>(k * b_step + n * 4) : kOut, 0, 0);
        }
    };
    auto multiply = [&](int st) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int f = 0; f < 4; ++f)
                    acc[e][f] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(av[st][u][e]), __uint_as_float(bv[st][u][f]), acc[e][f], 0, 0, 0);
    };
    // the waves take every fourth chunk; what lies beyond the last one is loaded as zeros
    int c = split * per_split + wave;
    load(0, c);
    for (; c < end; c += 8) {
        load(1, c + 4);
        multiply(0);
        load(0, c + 8);
        multiply(1);
    }
    // lane holds rows 4 * (4 * g + v) + e, columns 4 * r + f
    float* const mine = reinterpret_cast<float*>(lds) + wave * kPart;
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int v = 0; v < 4; ++v)
            *reinterpret_cast<float4_t*>(mine + (16 * g + 4 * v + e) * kPitch + 4 * r) = float4_t{acc[e][0][v], acc[e][1][v], acc[e][2][v], acc[e][3][v]};
    __syncthreads();
    float* out = static_cast<float*>(gridDim.y > 1 ? p.outs[batch] : p.out);
    const float* const part = reinterpret_cast<const float*>(lds);
    for (int e = tid; e < 64 * 64; e += 256) {
        const int row = e >> 6, col = e & 63, om = tm * 64 + row, on = tn * 64 + col;
        if (om >= p.M || on >= p.N) continue;
        float s = 0.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) s += part[w * kPart + row * kPitch + col];
        StoreTileElement<float>(p, split, out, om, on, s);
    }
}

// Sums the partial products of ksplit > 1.
template <typename T>
__global__ __launch_bounds__(256) void SmallDotSumKernel(SmallDotArgs p) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    const int64_t total = static_cast<int64_t>(p.M) * p.N;
    if (i >= total) return;
    float s = 0.f;
#pragma unroll 4
    for (int k = 0; k < p.ksplit; ++k) s += p.partial[k * total + i];
    const int m = static_cast<int>(i / p.N);
    StoreDot<T>(p, static_cast<T*>(p.out), m, static_cast<int>(i - static_cast<int64_t>(m) * p.N), s);
}

// M <= 4 rows against rows of K contiguous elements (b_k == 1, a_k == 1): a wave per output column, 64 x 16 bytes of K per step, the
// rows of `a` out of L1.  Bound by one pass over b: [1,784] . [784,1000] float32 7.7 -> 3 us.
template <typename T, int MR>
__global__ __launch_bounds__(256) void SmallDotVectorKernel(SmallDotArgs p) {
    constexpr int PL = 16 / sizeof(T);
    constexpr int U = 4;  // steps in flight
    const int lane = threadIdx.x & 63;
    const int n = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (n >= p.N) return;
    const __amdgpu_buffer_rsrc_t ar = MakeRsrc(p.a, p.a_bytes);
    const __amdgpu_buffer_rsrc_t br = MakeRsrc(p.b, p.b_bytes);
    const int b_line = static_cast<int>(n * p.b_col * static_cast<int64_t>(sizeof(T)));
    float acc[MR];
#pragma unroll
    for (int r = 0; r < MR; ++r) acc[r] = 0.f;
    for (int k0 = lane * PL; k0 - lane * PL < p.K; k0 += U * 64 * PL) {  // (uniform trip count)
        Bytes16 bv[U], av[U][MR];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + u * 64 * PL;
            const bool in = k < p.K;
            bv[u] = __builtin_amdgcn_raw_buffer_load_b128(br, in ? b_line + k * static_cast<int>(sizeof(T)) : 0x7fffffff, 0, 0);
#pragma unroll
            for (int r = 0; r < MR; ++r) {
                const int line = static_cast<int>(r * p.a_row * static_cast<int64_t>(sizeof(T)));
                av[u][r] = __builtin_amdgcn_raw_buffer_load_b128(ar, in && r < p.M ? line + k * static_cast<int>(sizeof(T)) : 0x7fffffff, 0, 0);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + u * 64 * PL;
            struct Piece {
                T e[PL];
            };
            const Piece bp = __builtin_bit_cast(Piece, bv[u]);
#pragma unroll
            for (int r = 0; r < MR; ++r) {
                const Piece ap = __builtin_bit_cast(Piece, av[u][r]);
#pragma unroll
                for (int e = 0; e < PL; ++e) {
                    const float product = static_cast<float>(ap.e[e]) * static_cast<float>(bp.e[e]);
                    acc[r] += k + e < p.K ? product : 0.f;  // (what follows K may be anything)
                }
            }
        }
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
#pragma unroll
        for (int r = 0; r < MR; ++r) acc[r] += __shfl_xor(acc[r], d, 64);
    }
    if (lane == 0) {
#pragma unroll
        for (int r = 0; r < MR; ++r) {
            if (r < p.M) StoreDot<T>(p, static_cast<T*>(p.out), r, n, acc[r]);
        }
    }
}

}  // namespace hipcx
