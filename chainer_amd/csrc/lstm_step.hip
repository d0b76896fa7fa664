// A step of an LSTM whose gates are Linear(x) + Linear(h), cell by cell: the two products, their sum and the cells in one launch.
#include <algorithm>

#include "lstm_cell.h"
#include "small_dot.h"

namespace hipcx {
namespace {

using double4_t = __attribute__((ext_vector_type(4))) double;

// The products of 16 bytes of 16 rows of a and b: in one chain of additions, in two, and in double.
template <typename T>
__device__ __forceinline__ void Terms(const Bytes16& a, const Bytes16& b, float4_t (&t)[1]) {
    t[0] = float4_t{0.f, 0.f, 0.f, 0.f};
    MfmaBlock<T>(a, b, t[0]);
}
template <typename T>
__device__ __forceinline__ void Terms(const Bytes16& a, const Bytes16& b, float4_t (&t)[2]) {
    const float4_t af = __builtin_bit_cast(float4_t, a), bf = __builtin_bit_cast(float4_t, b);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        t[i] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 2 * i; e < 2 * i + 2; ++e) t[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[e], bf[e], t[i], 0, 0, 0);
    }
}
template <typename T>
__device__ __forceinline__ void Terms(const Bytes16& a, const Bytes16& b, double4_t (&t)[1]) {
    const float4_t af = __builtin_bit_cast(float4_t, a), bf = __builtin_bit_cast(float4_t, b);
    t[0] = double4_t{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int e = 0; e < 4; ++e) t[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>(af[e]), static_cast<double>(bf[e]), t[0], 0, 0, 0);
}

struct LstmStepSide {
    const void* a;  // [M][K]
    const void* w;  // [4H][K]: gate k of unit j is row 4 j + k
    int K;
    unsigned a_row, w_row;  // bytes
};

struct LstmStepArgs {
    LstmStepSide side[2];  // x, h
    int x_waves;           // of the eight, those that take the x side
    int M, H;
    const void* bias;  // of the x side; may be null
    int64_t bias_stride;
    const void* c;
    void *h_out, *c_out;
    int64_t c_row, h_out_row, c_out_row;  // (elements)
    int tiles_m, tiles_n;
};

// Tiles of 16 * RB rows and the gates of 4 * NB units.  Eight waves split the reductions of the two products, each of which belongs to some of them; their sums
// meet in LDS, where the cells run on them: pre-activations never reach memory, and are rounded once.  A wave takes chunks of 128 bytes per row, whole
// lines turned round in LDS of its own, two of them in flight while a third is multiplied (three and four: equal or slower, [512,650] float32 78 us
// against 62).  Rows beyond M and columns beyond 4H repeat the last one (nobody reads what comes of them); the pieces that reach beyond the end of K
// are read from its last 16 bytes, without what the one before them holds.  Loads take any address, so odd pitches of float16 need no kernel of their own.
// Sums: 16 (8 for few rows or few terms) products to a chain, the chains of a chunk, the chunks, the waves, so that no case has a larger error than the separate calls
// (2-norm of the error of h and c, against 64 bits, separate calls and this: 128 x 650 units 1.06e-7, 6.8e-8, 1 x 650 5.2e-8, 5.1e-8, 2 x 77 of 129 inputs
// 4.57e-8, 4.56e-8); Acc = double for reductions of fewer than 64 terms, whose separate products are exact but for a rounding.
// Bound by the matrix pipe and by the delivery of operands at 128 rows, by the latency of launch, first loads and sums below.  us, the four calls and this,
// back to back on the device: 128 x 650 units float32 27.7, 18.6 (7.1 of MFMA on 220 compute units), float16 17.3, 8.9; 20 x 650 15.6, 8.8; 1 x 650 9.7, 6.8; 1 x 50
// 22.5, 4.3; float16 of an odd number of units, 37 x 77 of 129 inputs 15.2, 4.6.
template <typename T, typename Acc, int NB, int RB, int CH>
__global__ __launch_bounds__(512) void LstmStepKernel(LstmStepArgs p) {
    constexpr int PL = 16 / sizeof(T);
    constexpr int KC = 8 * PL;  // k per chunk
    using Acc4 = std::conditional_t<sizeof(Acc) == 8, double4_t, float4_t>;
    constexpr bool kExact = sizeof(Acc) == 8;
    static_assert(CH == 2 || (CH == 4 && sizeof(T) == 4 && !kExact));  // chains of additions that a chunk makes
    constexpr bool kHalves = CH == 4 && RB == 2;  // whose chains are added up by half a chunk: there are no registers for all of them
    constexpr int kKept = kHalves ? 2 : CH;
    constexpr int AL = 2 * RB, BL = 2 * NB;  // loads of a and w per chunk, 8 rows each
    constexpr int kRowsOfW = 16 * RB * kSmallDotPitch, kStage = kRowsOfW + 16 * NB * kSmallDotPitch, kPitch = 16 * NB + 4;
    extern __shared__ __align__(16) char lds[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, g = lane >> 4;
    const int piece = lane & 7, sub = lane >> 3;
    int tm, tn;
    SmallDotTile(p.tiles_m * p.tiles_n, blockIdx.x, p.tiles_m, tm, tn);
    const int of_h = wave >= p.x_waves;
    const char* const a = static_cast<const char*>(p.side[of_h].a);
    const char* const w = static_cast<const char*>(p.side[of_h].w);
    const int K = p.side[of_h].K;

    // what this thread's cell reads
    const int row = tid / (4 * NB), unit = tid % (4 * NB), m = tm * 16 * RB + row, u = tn * 4 * NB + unit;
    const bool has_cell = row < 16 * RB && m < p.M && u < p.H;
    float c_old = 0.f, bias[4] = {0.f, 0.f, 0.f, 0.f};
    if (has_cell) {
        c_old = static_cast<float>(static_cast<const T*>(p.c)[m * p.c_row + u]);
        if (p.bias != nullptr) {
#pragma unroll
            for (int k = 0; k < 4; ++k) bias[k] = static_cast<float>(static_cast<const T*>(p.bias)[(4 * u + k) * p.bias_stride]);
        }
    }

    unsigned a_line[AL], w_line[BL];
#pragma unroll
    for (int j = 0; j < AL; ++j) a_line[j] = static_cast<unsigned>(min(tm * 16 * RB + j * 8 + sub, p.M - 1)) * p.side[of_h].a_row;
#pragma unroll
    for (int j = 0; j < BL; ++j) w_line[j] = static_cast<unsigned>(min(tn * 16 * NB + j * 8 + sub, 4 * p.H - 1)) * p.side[of_h].w_row;
    char* const stage = lds + wave * kStage;
    char* const to = stage + sub * kSmallDotPitch + piece * 16;
    const char* const from = stage + lr * kSmallDotPitch + g * 16;

    const int chunks = (K + KC - 1) / KC, waves = of_h ? 8 - p.x_waves : p.x_waves;
    const int per_wave = (chunks + waves - 1) / waves;
    const int begin = (of_h ? wave - p.x_waves : wave) * per_wave, end = min(chunks, begin + per_wave);

    Acc4 acc[RB][NB];
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = Acc4{};
    Bytes16 av[2][AL], wv[2][BL];
    auto load = [&](int st, int c) {
        const unsigned at = static_cast<unsigned>(min(c * KC + piece * PL, K - PL)) * static_cast<unsigned>(sizeof(T));
#pragma unroll
        for (int j = 0; j < AL; ++j) __builtin_memcpy(&av[st][j], a + (a_line[j] + at), 16);
#pragma unroll
        for (int j = 0; j < BL; ++j) __builtin_memcpy(&wv[st][j], w + (w_line[j] + at), 16);
    };
    auto multiply = [&](int st, int c, auto&& next) {
        if ((c + 1) * KC > K) {
            const int early = PieceEarly<T>(c * KC + piece * PL, K);
#pragma unroll
            for (int j = 0; j < AL; ++j) av[st][j] = KeepPiece<T>(av[st][j], early);
#pragma unroll
            for (int j = 0; j < BL; ++j) wv[st][j] = KeepPiece<T>(wv[st][j], early);
        }
#pragma unroll
        for (int j = 0; j < AL; ++j) *reinterpret_cast<Bytes16*>(to + j * 8 * kSmallDotPitch) = av[st][j];
#pragma unroll
        for (int j = 0; j < BL; ++j) *reinterpret_cast<Bytes16*>(to + kRowsOfW + j * 8 * kSmallDotPitch) = wv[st][j];
        next();
        __builtin_amdgcn_wave_barrier();
        Acc4 terms[kKept][RB][NB];
#pragma unroll
        for (int q = 0; q < 2; ++q) {  // pieces g and g + 4 of each row
            Bytes16 fa[RB], fb[NB];
#pragma unroll
            for (int i = 0; i < RB; ++i) fa[i] = *reinterpret_cast<const Bytes16*>(from + i * 16 * kSmallDotPitch + q * 64);
#pragma unroll
            for (int j = 0; j < NB; ++j) fb[j] = *reinterpret_cast<const Bytes16*>(from + kRowsOfW + j * 16 * kSmallDotPitch + q * 64);
#pragma unroll
            for (int i = 0; i < RB; ++i)
#pragma unroll
                for (int j = 0; j < NB; ++j) {
                    Acc4 t[CH / 2];
                    Terms<T>(fa[i], fb[j], t);
#pragma unroll
                    for (int e = 0; e < CH / 2; ++e) terms[(kHalves ? 0 : q * CH / 2) + e][i][j] = t[e];
                }
            if (!kHalves && q == 0) continue;
#pragma unroll
            for (int i = 0; i < RB; ++i)
#pragma unroll
                for (int j = 0; j < NB; ++j) {
                    if constexpr (kKept == 2) acc[i][j] += terms[0][i][j] + terms[1][i][j];
                    else acc[i][j] += (terms[0][i][j] + terms[1][i][j]) + (terms[2][i][j] + terms[3][i][j]);
                }
        }
        __builtin_amdgcn_wave_barrier();
    };
    if (begin < end) {
        load(0, begin);
        if (begin + 1 < end) load(1, begin + 1);
        for (int c = begin; c < end; c += 2) {
            multiply(0, c, [&] {
                if (c + 2 < end) load(0, c + 2);
            });
            if (c + 1 < end) {
                multiply(1, c + 1, [&] {
                    if (c + 3 < end) load(1, c + 3);
                });
            }
        }
    }
    __syncthreads();  // the staging areas become the sums
    // lane holds column lr, rows 4 * g + v of each block (in double g + 4 * v)
    constexpr int kPart = 16 * RB * kPitch;
    Acc* const part = reinterpret_cast<Acc*>(lds);
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) part[wave * kPart + (i * 16 + (kExact ? g + 4 * v : 4 * g + v)) * kPitch + j * 16 + lr] = acc[i][j][v];
    __syncthreads();
    if (!has_cell) return;
    Acc4 sum[2] = {Acc4{}, Acc4{}};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const Acc4 s = *reinterpret_cast<const Acc4*>(part + i * kPart + row * kPitch + unit * 4);
        if (i < p.x_waves) sum[0] += s;
        else sum[1] += s;
    }
    float gate[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) gate[k] = static_cast<float>((sum[0][k] + static_cast<Acc>(bias[k])) + sum[1][k]);
    float c_new;
    const float h = LstmCell<float>(gate, c_old, c_new);
    static_cast<T*>(p.c_out)[m * p.c_out_row + u] = static_cast<T>(c_new);
    static_cast<T*>(p.h_out)[m * p.h_out_row + u] = static_cast<T>(h);
}

constexpr int kExactTerms = 64;  // float32 reductions of fewer terms are summed in double

int64_t StepTiles(int64_t rows, int64_t units, int blocks) { return (rows + 31) / 32 * ((units + 4 * blocks - 1) / (4 * blocks)); }

// Up to four (float16: six) tiles of 32 rows and 16 units to a compute unit: beyond, the tiles of a large product read each operand less often.  us, the four
// calls and one, float32: 768 x 650 units, 3.8 tiles, 90.7, 85.5; 4096 x 128, 4, 50.9, 25.6; 1024 x 650, 5.1, 116, 123; 512 x 2048, 8, 282, 336.  float16: 1024 x 650
// 64.7, 49.9; 2048 x 300, 4.8, 41.0, 28.7; 1024 x 1024, 8, 69.4, 75.1; 512 x 2048 94.4, 111.
// And up to a number of terms, over the rounds of tiles that a compute unit takes: the separate products split theirs over workgroups, or run in larger tiles.
// float32 (rounds x terms): 445 x 567 of 594 inputs (2322) 43.1, 37.6; 57 x 79 of 3388 (3467) 15.3, 15.0; 52 x 168 of 5347 (5515) 22.3, 21.3; 886 x 419 of 2576
// (8985) 112, 114; 107 x 112 of 9223 (9335) 30.2, 35.7; 169 x 1537 of 7891 (28284) 217, 285.  float16: 245 x 1465 of 238 (5109) 40.7, 31.3; 144 x 948 of 2967 (7830)
// 35.3, 37.5; 606 x 9 of 9241 (9250) 19.5, 22.0; 3003 x 184 of 7054 (36190) 83, 149.  In double, in tiles of 4 units: 8192 x 16 (128) 23.8, 10.5; 4096 x 50 (700) 37.8,
// 15.8; 32 x 15 of 940 (955) 12.3, 10.1; 3 x 27 of 975 (1002) 9.8, 10.2; 508 x 319 of 23 (1710) 20.9, 22.2; 128 x 2048 of 50 (16784) 66, 116.
bool StepTakes(int64_t rows, int64_t units, int64_t inputs, int dtype) {
    if (StepTiles(rows, units, 4) > (dtype == HIPCX_FLOAT32 ? 4 : 6) * NumCUs()) return false;
    const bool exact = dtype == HIPCX_FLOAT32 && std::min(inputs, units) < kExactTerms;
    const int64_t rounds = (StepTiles(rows, units, exact ? 1 : 4) + NumCUs() - 1) / NumCUs();
    return rounds * (inputs + units) <= (exact ? 960 : dtype == HIPCX_FLOAT32 ? 5300 : 7800);
}

template <typename T>
void RunLstmStep(LstmStepArgs& p, hipStream_t stream) {
    auto launch = [&](auto acc, auto blocks, auto row_blocks, auto chains) {
        using Acc = decltype(acc);
        constexpr int NB = decltype(blocks)::value, RB = decltype(row_blocks)::value, CH = decltype(chains)::value, kLds = 8 * 16 * (RB + NB) * kSmallDotPitch;
        static_assert(kLds >= 8 * 16 * RB * (16 * NB + 4) * static_cast<int>(sizeof(Acc)), "the sums fit the staging areas");
        p.tiles_m = (p.M + 16 * RB - 1) / (16 * RB), p.tiles_n = (p.H + 4 * NB - 1) / (4 * NB);
        struct StepTag {};
        EnsureDynamicLds<StepTag>(reinterpret_cast<const void*>(LstmStepKernel<T, Acc, NB, RB, CH>), kLds);
        hipLaunchKernelGGL((LstmStepKernel<T, Acc, NB, RB, CH>), dim3(static_cast<unsigned>(p.tiles_m * p.tiles_n)), dim3(512), kLds, stream, p);
        CheckLaunch("lstm_step");
    };
    using std::integral_constant;
    using One = integral_constant<int, 1>;
    using Two = integral_constant<int, 2>;
    using Four = integral_constant<int, 4>;
    // float32: chains of 8 terms for few rows, whose separate products are summed in short chains, and for few terms, of 16 else.  2-norm of the error of h, 64 rows,
    // the separate calls and chains of 16 and 8: 64 units of 64 inputs 9.6e-8, 9.9e-8, 9.3e-8; 97 of 97 1.02e-7, 1.03e-7, 9.6e-8; 200 of 200, in chains of 16, 1.19e-7,
    // 1.05e-7.  us, 16 and 8: 128 rows of 100 units 4.26 and 4.34, 4096 of 127 25.9 and 26.6.
    const bool short_chains = std::min(p.side[0].K, p.side[1].K) < 128;
    auto run = [&](auto acc, auto blocks, auto row_blocks) {
        if constexpr (sizeof(T) == 4 && std::is_same_v<decltype(acc), float>) {
            if (decltype(row_blocks)::value == 1 || short_chains) return launch(acc, blocks, row_blocks, Four{});
        }
        if constexpr (sizeof(T) == 2 || std::is_same_v<decltype(acc), double> || decltype(row_blocks)::value == 2) launch(acc, blocks, row_blocks, Two{});
    };
    if constexpr (sizeof(T) == 4) {
        if (std::min(p.side[0].K, p.side[1].K) < kExactTerms) return run(0.0, One{}, Two{});
    }
    int nb = 4;  // the narrowest tiles that find each of them a compute unit
    for (int b = 3; b >= 1; --b) {
        if (StepTiles(p.M, p.H, b) <= NumCUs()) nb = b;
    }
    if (p.M <= 16 && nb == 1) return run(0.f, One{}, One{});
    if (p.M <= 16 && nb == 2) return run(0.f, Two{}, One{});
    switch (nb) {
        case 1: return run(0.f, One{}, Two{});
        case 2: return run(0.f, Two{}, Two{});
        case 3: return run(0.f, integral_constant<int, 3>{}, Two{});
        default: return run(0.f, integral_constant<int, 4>{}, Two{});
    }
}

// A matrix whose rows LstmStepKernel reads: dense, of 16 bytes or more, the span below 2^31 bytes.
bool StepRows(const hipcx_array* a, int64_t rows, int64_t cols, int dtype, int64_t least) {
    const int64_t it = ItemSize(dtype);
    return a->ndim == 2 && a->dtype == dtype && a->shape[0] == rows && a->shape[1] == cols && cols >= least && a->strides[1] == it && a->strides[0] >= 0 &&
           a->strides[0] % it == 0 && reinterpret_cast<uintptr_t>(a->data) % it == 0 && rows * a->strides[0] + cols * it < (1LL << 31);
}

}  // namespace
}  // namespace hipcx

using namespace hipcx;

extern "C" {

int hipcx_lstm_step_supported(const hipcx_array* c, const hipcx_array* x, const hipcx_array* wx, const hipcx_array* bx, const hipcx_array* h, const hipcx_array* wh) {
    if (c == nullptr || x == nullptr || wx == nullptr || h == nullptr || wh == nullptr) return 0;
    if ((c->dtype != HIPCX_FLOAT32 && c->dtype != HIPCX_FLOAT16) || c->ndim != 2 || x->ndim != 2) return 0;
    const int64_t M = c->shape[0], H = c->shape[1], piece = 16 / ItemSize(c->dtype);
    if (M < 1 || H < 1 || H >= (1 << 28) || !StepTakes(M, H, x->shape[1], c->dtype)) return 0;
    return StepRows(c, M, H, c->dtype, 1) && StepRows(x, M, x->shape[1], c->dtype, piece) && StepRows(h, M, H, c->dtype, piece) &&
           StepRows(wx, 4 * H, x->shape[1], c->dtype, piece) && StepRows(wh, 4 * H, H, c->dtype, piece) &&
           (bx == nullptr || (bx->ndim == 1 && bx->dtype == c->dtype && bx->shape[0] == 4 * H && bx->strides[0] % ItemSize(c->dtype) == 0));
}

int hipcx_lstm_step(const hipcx_array* c, const hipcx_array* x, const hipcx_array* wx, const hipcx_array* bx, const hipcx_array* h, const hipcx_array* wh,
                    const hipcx_array* h_out, const hipcx_array* c_out, void* stream) {
    return Guard([&] {
        for (const hipcx_array* a : {c, x, wx, h, wh, h_out, c_out}) ValidateArray(a, "lstm_step");
        if (bx != nullptr) ValidateArray(bx, "lstm_step");
        HIPCX_REQUIRE(hipcx_lstm_step_supported(c, x, wx, bx, h, wh) != 0, HIPCX_NOT_IMPLEMENTED_ERROR, "lstm_step: hipcx_lstm_step_supported says no");
        const int64_t M = c->shape[0], H = c->shape[1], it = ItemSize(c->dtype);
        HIPCX_REQUIRE(StepRows(h_out, M, H, c->dtype, 1) && StepRows(c_out, M, H, c->dtype, 1), HIPCX_DIMENSION_ERROR, "lstm_step: outputs must be like c");
        LstmStepArgs p{};
        p.side[0] = {x->data, wx->data, static_cast<int>(x->shape[1]), static_cast<unsigned>(x->strides[0]), static_cast<unsigned>(wx->strides[0])};
        p.side[1] = {h->data, wh->data, static_cast<int>(H), static_cast<unsigned>(h->strides[0]), static_cast<unsigned>(wh->strides[0])};
        const int64_t chunk = 128 / it, of_x = (p.side[0].K + chunk - 1) / chunk, of_h = (H + chunk - 1) / chunk;
        int64_t least = INT64_MAX;  // chunks of the wave that has most
        for (int n = 1; n < 8; ++n) {
            const int64_t most = std::max((of_x + n - 1) / n, (of_h + 7 - n) / (8 - n));
            if (most < least) least = most, p.x_waves = n;
        }
        p.M = static_cast<int>(M), p.H = static_cast<int>(H);
        if (bx != nullptr) p.bias = bx->data, p.bias_stride = bx->strides[0] / it;
        p.c = c->data, p.h_out = h_out->data, p.c_out = c_out->data;
        p.c_row = c->strides[0] / it, p.h_out_row = h_out->strides[0] / it, p.c_out_row = c_out->strides[0] / it;
        if (c->dtype == HIPCX_FLOAT32) RunLstmStep<float>(p, AsStream(stream));
        else RunLstmStep<half_t>(p, AsStream(stream));
    });
}

}  // extern "C"
