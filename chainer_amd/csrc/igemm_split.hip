// The implicit GEMM of igemm.h for float32 operands on the bfloat16 matrix pipes.
//
// v_mfma_f32_32x32x16_bf16 does sixteen times the multiply-adds of v_mfma_f32_32x32x2_f32 in a clock.  A float is the sum of three
// bfloat16 numbers, exactly: x1 = bf16(x), x2 = bf16(x - x1), x3 = x - x1 - x2 (24 significant bits = 3 x 8; rounding to nearest leaves
// remainders of at most half a unit, which have 16 and 8 bits; such splits are published, e.g. Henry, Tang and Heinecke, ARITH 2019).  Of the
// nine products of two such sums all but x3 w3, at most 2^-34 of x w, are computed.  A bfloat16 product is exact in float32; the matrix pipe's
// additions are not rounded to nearest (one product added to the sum of its small parts may be off by a whole unit).  Hence two accumulators:
// x1 w1, whose 16 bits leave room for a few terms without any rounding and which is rounded once for 16 terms, and the seven others, 2^-8 of it,
// whose roundings do not show; they are added at the end.  Largest relative error of one term 5.98e-8 (5.96e-8 on the float pipe, rounded to
// nearest; 1.5e-7 with one accumulator and six products), 2-norm for two to eight terms among zeros 2.6 to 2.8e-8 (3.1 to 5.4e-8; 4.1 to
// 8.2e-8), for more see LaunchShape.
//
// Where the split is not exact the tile is computed again on the float pipe, by the same workgroup: a sum that is not finite (an operand that
// is infinite, NaN or beyond bfloat16's range, or a sum that overflowed), a nonzero sum so small that its parts' roundings to multiples of 2^-149 add
// up, or a nonzero operand below 2^-110, whose last bits bfloat16 has no numbers for (its least is 2^-133), in a row whose sum is small enough
// for those to count.
//
// Layout: a workgroup's rows of x and w are split while they are staged, each element once, into three planes of LDS, 16 k at a time; a plane's
// rows have 32 bytes, whose two pieces change places every eight rows, so that the staging writes and the fragment reads (16 bytes of 16 rows) both
// use all banks.  12 fragment reads feed 32 MFMAs of a wave's 64 x 64 block.  The next step's rows are split into the other stage between the MFMAs of
// the current one, with one barrier a step; 48 KiB for a 128 x 128 tile, two workgroups to a compute unit, as the registers allow.
// Bound by the MFMAs (at [4096,4096]^2 0.44 of 0.81 ms) and by the splitting.
#include "igemm_split.h"

#include <type_traits>

namespace hipcx {
namespace {

using bf16x2_t = __attribute__((ext_vector_type(2))) __bf16;
using bf16x8_t = __attribute__((ext_vector_type(8))) __bf16;
using float2_t = __attribute__((ext_vector_type(2))) float;

// Two floats as three pairs of bfloat16.
__device__ __forceinline__ void SplitPair(unsigned a_bits, unsigned b_bits, unsigned (&part)[3]) {
    float a = __uint_as_float(a_bits), b = __uint_as_float(b_bits);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const unsigned u = __builtin_bit_cast(unsigned, __builtin_convertvector(float2_t{a, b}, bf16x2_t));
        part[i] = u;
        a -= __builtin_bit_cast(float, u << 16);
        b -= __builtin_bit_cast(float, u & 0xffff0000u);
    }
}

__device__ __forceinline__ void MfmaBf16(const Bytes16& a, const Bytes16& b, float16_t& acc) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), acc, 0, 0, 0);
}

constexpr int kSplitStep = 16;  // k of a step
constexpr int kSplitRow = 2 * kSplitStep;  // bytes of a row in a plane
constexpr int kSplitFloatRow = 4 * kSplitStep + 16;
// Twice the bits of a number, less one, as unsigned: zero is the largest.  The least value that splits exactly is 2^-110.
constexpr unsigned kSplitLeast = (17u << 24) - 1u;

__device__ __forceinline__ unsigned SplitKey(unsigned bits) { return (bits << 1) - 1u; }

// Sums from here on are not rounded to multiples of 2^-149 by their parts' additions.
constexpr float kSplitLeastSum = 0x1p-120f;

// Whether all sums are finite (x * 0 is 0 for those only) and none is a tiny one.
__device__ __forceinline__ bool AllOrdinary(const float16_t (&acc)[2][2]) {
    bool all = true;
    unsigned least = ~0u;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            float zero = 0.f;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                zero += acc[i][j][v] * 0.f;
                least = min(least, SplitKey(__float_as_uint(acc[i][j][v])));
            }
            all &= zero == 0.f;
        }
    return all & (least >= SplitKey(__float_as_uint(kSplitLeastSum)));
}

template <int WM, int WN, int LB, bool PM>
__global__ __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(2))) void IGemmSplitKernel(IGemmArgs<float> p) {
    constexpr int NT = 64 * WM * WN;
    constexpr int BM = 64 * WM;
    constexpr int BN = 64 * WN;
    constexpr int CPR = 4 * kSplitStep / LB;  // chunks per row
    constexpr int EPC = LB / 4;
    constexpr int XCH = BM * CPR / NT;
    constexpr int WCH = BN * CPR / NT;
    constexpr int RPP = NT / CPR;  // rows per pass
    constexpr int PLANE = (BM + BN) * kSplitRow;
    constexpr int STAGE = 3 * PLANE;
    constexpr int kOut = 0x7fffffff;  // an offset beyond any buffer: zeros
    using Chunk = typename BytesOf<LB>::type;

    static_assert((BM + BN) * kSplitFloatRow <= 2 * STAGE, "rows of floats fit the two stages");
    __shared__ __align__(16) char lds[2 * STAGE];

    int tile_m, tile_n;
    unsigned slice = 0;
    if (p.ksplit > 1) {  // as in IGemmFastKernel
        slice = blockIdx.x;
        tile_n = static_cast<int>(blockIdx.y) % p.tiles_n;
        tile_m = static_cast<int>(blockIdx.y) / p.tiles_n;
    } else if (!TileOfBanded(p.tiles_m, p.tiles_n, p.band, tile_m, tile_n)) {
        return;
    }
    const int m0 = tile_m * BM;
    const int n0 = tile_n * BN;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wm = wave % WM;
    const int wn = wave / WM;
    const int kc = tid % CPR;
    const int row0 = tid / CPR;

    // Rows of x: byte offsets from the first image of the tile; the host has checked that they fit.
    const int ohw = p.OH * p.OW;
    const int img0 = m0 / ohw;
    const __amdgpu_buffer_rsrc_t xr = MakeRsrc(p.x + img0 * p.xsN, 0x7ffffffcu);
    const __amdgpu_buffer_rsrc_t wr = MakeRsrc(p.w + n0 * p.wsK, 0x7ffffffcu);
    int xoff[XCH], ih0[XCH], iw0[XCH];
#pragma unroll
    for (int i = 0; i < XCH; ++i) {
        const int m = m0 + row0 + i * RPP;
        const int img = m / ohw, pix = m - img * ohw;
        const int oh = pix / p.OW, ow = pix - oh * p.OW;
        ih0[i] = m < p.M ? oh * p.stride_h - p.pad_h : -0x40000000;  // fails every bounds check
        iw0[i] = ow * p.stride_w - p.pad_w;
        xoff[i] = m < p.M ? static_cast<int>(((img - img0) * p.xsN + ih0[i] * p.xsH + iw0[i] * p.xsW + kc * EPC) * 4) : 0;
    }
    int woff[WCH];
#pragma unroll
    for (int i = 0; i < WCH; ++i) {
        const int n = row0 + i * RPP;
        woff[i] = n0 + n < p.K ? static_cast<int>((n * p.wsK + kc * EPC) * 4) : -1;
    }

    const int nk = (p.Kg + kSplitStep - 1) / kSplitStep;
    const int xh = static_cast<int>(p.xsH * 4), xw = static_cast<int>(p.xsW * 4);

    Chunk xreg[XCH], wreg[WCH];
    auto load = [&](const __amdgpu_buffer_rsrc_t& rsrc, int off) {
        if constexpr (LB == 16) return __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, 0, 0);
        else return __builtin_amdgcn_raw_buffer_load_b64(rsrc, off, 0, 0);
    };
    // The step to be loaded next: first k, its filter position and the channel there.  A step lies inside one filter position (the host has checked
    // that, or there is only one), so that all of this is scalar and without a branch.
    int k_next = 0, r_next = 0, s_next = 0, c_next = 0;
    auto seek = [&](int kt) {
        k_next = kt * kSplitStep;
        const int rs = k_next / p.C;
        c_next = k_next - rs * p.C;
        r_next = rs / p.S;
        s_next = rs - r_next * p.S;
    };
    auto load_tile = [&] {
        const int step = r_next * xh + s_next * xw + c_next * 4;
        const bool kvalid = k_next + kc * EPC < p.Kg;
        const int r = r_next, s = s_next, kbase = k_next;
        k_next += kSplitStep;
        c_next += kSplitStep;
        const bool next_s = c_next >= p.C;
        c_next = next_s ? 0 : c_next;
        s_next += next_s;
        const bool next_r = s_next == p.S;
        s_next = next_r ? 0 : s_next;
        r_next += next_r;
#pragma unroll
        for (int i = 0; i < XCH; ++i) {
            const bool ok = kvalid & (static_cast<unsigned>(ih0[i] + r) < static_cast<unsigned>(p.H)) & (static_cast<unsigned>(iw0[i] + s) < static_cast<unsigned>(p.W));
            xreg[i] = load(xr, ok ? xoff[i] + step : kOut);
        }
#pragma unroll
        for (int i = 0; i < WCH; ++i) wreg[i] = load(wr, (kvalid & (woff[i] >= 0)) ? woff[i] + kbase * 4 : kOut);
    };

    unsigned least = ~0u;  // of the keys of what this thread staged
    auto split_chunk = [&](const Chunk& v, int row, char* stage) {
        unsigned a[3], b[3];
        least = min(least, min(SplitKey(v[0]), SplitKey(v[1])));
        SplitPair(v[0], v[1], a);
        char* at = stage + row * kSplitRow;
        if constexpr (LB == 16) {
            least = min(least, min(SplitKey(v[2]), SplitKey(v[3])));
            SplitPair(v[2], v[3], b);
            at += ((kc >> 1) ^ ((row >> 3) & 1)) * 16 + (kc & 1) * 8;
#pragma unroll
            for (int i = 0; i < 3; ++i) *reinterpret_cast<Bytes8*>(at + i * PLANE) = Bytes8{a[i], b[i]};
        } else {
            at += ((kc >> 2) ^ ((row >> 3) & 1)) * 16 + (kc & 3) * 4;
#pragma unroll
            for (int i = 0; i < 3; ++i) *reinterpret_cast<unsigned*>(at + i * PLANE) = a[i];
        }
    };
    auto split_tile = [&](char* stage) {
#pragma unroll
        for (int i = 0; i < XCH; ++i) split_chunk(xreg[i], row0 + i * RPP, stage);
#pragma unroll
        for (int i = 0; i < WCH; ++i) split_chunk(wreg[i], BM + row0 + i * RPP, stage);
    };
    const int lr = lane & 31, g = lane >> 5;
    const int xfrag = (wm * 64 + lr) * kSplitRow + (g ^ ((lr >> 3) & 1)) * 16;
    const int wfrag = (BM + wn * 64 + lr) * kSplitRow + (g ^ ((lr >> 3) & 1)) * 16;
    float16_t acc[2][2], low[2][2];
    auto clear = [&] {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f, low[i][j][v] = 0.f;
    };
    // One step: the fragments of stage kt & 1 are multiplied while the next step's rows, which have arrived in registers, are split into the other
    // stage and the loads of the step behind it go out.
    auto step = [&](int kt, auto split_tag, auto load_tag) {
        char* const cur = lds + (kt & 1) * STAGE;
        Bytes16 xf[3][2], wf[3][2];
#pragma unroll
        for (int i = 2; i >= 0; --i)
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                xf[i][t] = *reinterpret_cast<const Bytes16*>(cur + xfrag + i * PLANE + t * 32 * kSplitRow);
                wf[2 - i][t] = *reinterpret_cast<const Bytes16*>(cur + wfrag + (2 - i) * PLANE + t * 32 * kSplitRow);
            }
        if constexpr (decltype(split_tag)::value) split_tile(lds + (~kt & 1) * STAGE);
        if constexpr (decltype(load_tag)::value) load_tile();
        constexpr int kX[8] = {2, 1, 2, 0, 1, 1, 0, 0}, kW[8] = {1, 2, 0, 2, 1, 0, 1, 0};
#pragma unroll
        for (int c = 0; c < 8; ++c)
#pragma unroll
            for (int ti = 0; ti < 2; ++ti)
#pragma unroll
                for (int tj = 0; tj < 2; ++tj) {
                    float16_t& sum = c == 7 ? acc[ti][tj] : low[ti][tj];
                    if (PM) MfmaBf16(xf[kX[c]][ti], wf[kW[c]][tj], sum);
                    else MfmaBf16(wf[kW[c]][ti], xf[kX[c]][tj], sum);
                }
        if constexpr (decltype(split_tag)::value) {
            __builtin_amdgcn_sched_group_barrier(0x100, 12, 0);
#pragma unroll
            for (int i = 0; i < 32; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
                if (i % 2 == 1) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
            }
        }
        __syncthreads();
    };

    int kt_begin = 0, kt_end = nk;
    if (p.ksplit > 1) {
        kt_begin = static_cast<int>(static_cast<int64_t>(nk) * slice / p.ksplit);
        kt_end = static_cast<int>(static_cast<int64_t>(nk) * (slice + 1) / p.ksplit);
    }
    clear();
    if (kt_begin < kt_end) {
        using std::false_type;
        using std::true_type;
        seek(kt_begin);
        load_tile();
        split_tile(lds + (kt_begin & 1) * STAGE);
        if (kt_begin + 1 < kt_end) load_tile();
        __syncthreads();
        int kt = kt_begin;
        for (; kt + 2 < kt_end; ++kt) step(kt, true_type{}, true_type{});
        if (kt + 1 < kt_end) step(kt++, true_type{}, false_type{});
        step(kt, false_type{}, false_type{});
    }

#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] += low[i][j];
    bool again = !AllOrdinary(acc);
    if (__syncthreads_or(least < kSplitLeast)) {
        // Operands lost at most 2^-134 each, which changes a sum by less than 2^-133 terms times the largest operand: by less than 2^-29 of it, an eighth of
        // a rounding, from 2^-104 terms times that operand on.  The rows are read once more, to see which of them this is about.
        constexpr int kDeep = 16 / (XCH + WCH);  // steps in flight
        unsigned* const keys = reinterpret_cast<unsigned*>(lds);  // the least key of each row, then the waves' largest operands
        unsigned row_least[XCH + WCH], most = 0;
#pragma unroll
        for (int i = 0; i < XCH + WCH; ++i) row_least[i] = ~0u;
        seek(kt_begin);
        for (int kt = kt_begin; kt < kt_end; kt += kDeep) {  // (what lies beyond kt_end may count too; beyond the last k are zeros)
            Chunk rows[kDeep][XCH + WCH];
#pragma unroll
            for (int u = 0; u < kDeep; ++u) {
                load_tile();
#pragma unroll
                for (int i = 0; i < XCH; ++i) rows[u][i] = xreg[i];
#pragma unroll
                for (int i = 0; i < WCH; ++i) rows[u][XCH + i] = wreg[i];
            }
#pragma unroll
            for (int u = 0; u < kDeep; ++u)
#pragma unroll
                for (int i = 0; i < XCH + WCH; ++i)
#pragma unroll
                    for (int e = 0; e < EPC; ++e) {
                        row_least[i] = min(row_least[i], SplitKey(rows[u][i][e]));
                        most = max(most, rows[u][i][e] & 0x7fffffffu);
                    }
        }
#pragma unroll
        for (int i = 0; i < XCH + WCH; ++i) {
#pragma unroll
            for (int o = 1; o < CPR; o <<= 1) row_least[i] = min(row_least[i], static_cast<unsigned>(__shfl_xor(static_cast<int>(row_least[i]), o)));
            if (kc == 0) keys[i < XCH ? row0 + i * RPP : BM + row0 + (i - XCH) * RPP] = row_least[i];
        }
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) most = max(most, static_cast<unsigned>(__shfl_xor(static_cast<int>(most), o)));
        if (lane == 0) keys[BM + BN + wave] = most;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < WM * WN; ++i) most = max(most, keys[BM + BN + i]);
        const float enough = 0x1p-104f * static_cast<float>((kt_end - kt_begin) * kSplitStep) * __uint_as_float(most);
#pragma unroll
        for (int ti = 0; ti < 2; ++ti)
#pragma unroll
            for (int tj = 0; tj < 2; ++tj) {
                const int row_at = PM ? wm * 64 + ti * 32 : BM + wn * 64 + ti * 32, col_at = PM ? BM + wn * 64 + tj * 32 : wm * 64 + tj * 32;
                const unsigned col = keys[col_at + lr];
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const unsigned row = keys[row_at + 8 * (v / 4) + 4 * g + v % 4];
                    // (a sum over a row of zeros is zero)
                    again |= (min(row, col) < kSplitLeast) & (max(row, col) != ~0u) & (fabsf(acc[ti][tj][v]) < enough);
                }
            }
    }
    if (__syncthreads_or(again)) {
        clear();
        seek(kt_begin);
        for (int kt = kt_begin; kt < kt_end; ++kt) {
            load_tile();
#pragma unroll
            for (int i = 0; i < XCH; ++i) *reinterpret_cast<Chunk*>(lds + (row0 + i * RPP) * kSplitFloatRow + kc * LB) = xreg[i];
#pragma unroll
            for (int i = 0; i < WCH; ++i) *reinterpret_cast<Chunk*>(lds + (BM + row0 + i * RPP) * kSplitFloatRow + kc * LB) = wreg[i];
            __syncthreads();
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                Bytes16 xf[2], wf[2];
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    xf[t] = *reinterpret_cast<const Bytes16*>(lds + (wm * 64 + t * 32 + lr) * kSplitFloatRow + (2 * q + g) * 16);
                    wf[t] = *reinterpret_cast<const Bytes16*>(lds + (BM + wn * 64 + t * 32 + lr) * kSplitFloatRow + (2 * q + g) * 16);
                }
#pragma unroll
                for (int ti = 0; ti < 2; ++ti)
#pragma unroll
                    for (int tj = 0; tj < 2; ++tj) {
                        if (PM) MfmaTile<float>(xf[ti], wf[tj], acc[ti][tj]);
                        else MfmaTile<float>(wf[ti], xf[tj], acc[ti][tj]);
                    }
            }
            __syncthreads();
        }
    }
    if (p.ksplit > 1) {
        if constexpr (!PM) StorePartial<float>(p, m0, n0, wm, wn, lane, acc, slice);
        return;
    }
    if (PM) {
        StoreTilePM<float>(p, m0, n0, wm, wn, lane, acc);
    } else {
        StoreTile<float>(p, m0, n0, wm, wn, lane, acc);
    }
}

}  // namespace

template <int WM, int WN>
bool IGemmSplit(const IGemmArgs<float>& p, int chunk_bytes, bool pm, dim3 grid, hipStream_t stream) {
    constexpr int BM = 64 * WM, BN = 64 * WN;
    // A single tile of a few terms stays on the float pipe: bound by the launch and the first loads, it has a microsecond to gain ([6,40] . [40,64] 8.3 and
    // 7.4 us) and keeps the sums, rounded to nearest term by term, that recurrent networks amplify.
    if (p.tiles_m * p.tiles_n == 1 && p.Kg < 64) return false;
    if (p.batch > 0 || p.w_taps_s > 0 || p.xsN < 0 || p.xsH < 0 || p.xsW < 0 || p.wsK < 0) return false;
    if ((p.R > 1 || p.S > 1) && p.C % kSplitStep != 0) return false;  // a step would reach over several filter positions
    // the kernel's offsets from a tile's first image and first filter have 32 bits
    const double limit = 2147483000.0 / sizeof(float), images = BM / (static_cast<double>(p.OH) * p.OW) + 2;
    const double image = static_cast<double>(p.H + p.pad_h) * p.xsH + static_cast<double>(p.W + p.pad_w) * p.xsW + p.Kg;
    if (images * p.xsN + image >= limit || static_cast<double>(BN) * p.wsK + p.Kg >= limit) return false;
    auto launch = [&](auto chunk, auto orientation) {
        hipLaunchKernelGGL((IGemmSplitKernel<WM, WN, decltype(chunk)::value, decltype(orientation)::value>), grid, dim3(64 * WM * WN), 0, stream, p);
    };
    using std::false_type;
    using std::true_type;
    if (chunk_bytes == 16) pm ? launch(std::integral_constant<int, 16>{}, true_type{}) : launch(std::integral_constant<int, 16>{}, false_type{});
    else pm ? launch(std::integral_constant<int, 8>{}, true_type{}) : launch(std::integral_constant<int, 8>{}, false_type{});
    return true;
}
template bool IGemmSplit<1, 1>(const IGemmArgs<float>&, int, bool, dim3, hipStream_t);
template bool IGemmSplit<2, 2>(const IGemmArgs<float>&, int, bool, dim3, hipStream_t);
template bool IGemmSplit<4, 1>(const IGemmArgs<float>&, int, bool, dim3, hipStream_t);

}  // namespace hipcx
