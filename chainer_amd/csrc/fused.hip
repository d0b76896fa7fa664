// Routine chains that the reference runs as many small kernels, as one or two; the routines take them wherever their arrays allow:
//   * LogSoftmax (CX/routines/reduction.cc:78-92): AMax, Subtract, Exp, Sum, Log, Add, Subtract -- 5 reads and 3 writes of
//     the array -- as one read + one write when a row fits in a workgroup's registers, two reads + one write otherwise;
//   * softmax cross entropy (chainer/functions/loss/softmax_cross_entropy.py:123-130): LogSoftmax and a masked mean, about 15 kernels,
//     as one read;
//   * the Lstm cell (CX/routines/connection.cc:396-446): ~25 strided elementwise kernels as one.
// They evaluate the same float operations in the same order as the chain (Exp/Tanh/Log are the same device functions the
// separate kernels call; no contraction), so for float32/float64 the Lstm cell is bit-identical to the chain and LogSoftmax
// differs only through the order of the row sum.  float16 computes in float and rounds once.
#include <algorithm>

#include "common.h"
#include "lstm_cell.h"

namespace hipcx {
namespace {

template <typename C>
__device__ __forceinline__ C ExpOf(C v) {
    if constexpr (std::is_same_v<C, float>) return expf(v);
    else return exp(v);
}
template <typename C>
__device__ __forceinline__ C LogOf(C v) {
    if constexpr (std::is_same_v<C, float>) return logf(v);
    else return log(v);
}
// AMax's update (native/native_device/statistics.cc:27-48): NaN wins, otherwise strictly greater.
template <typename C>
__device__ __forceinline__ C MaxNan(C acc, C v) {
    return (v != v || acc < v) ? v : acc;
}

template <typename C>
__device__ __forceinline__ C ShflDown(C v, int d) {
    if constexpr (sizeof(C) == 4) {
        return __shfl_down(v, d, 64);
    } else {
        long long b = __builtin_bit_cast(long long, v);
        int lo = __shfl_down(static_cast<int>(b & 0xffffffffLL), d, 64);
        int hi = __shfl_down(static_cast<int>(b >> 32), d, 64);
        return __builtin_bit_cast(C, (static_cast<long long>(hi) << 32) | (static_cast<long long>(lo) & 0xffffffffLL));
    }
}

// Block-wide reductions for NT threads (result valid in every thread).
template <typename C, int NT, bool IS_MAX>
__device__ __forceinline__ C BlockReduce(C v, C* scratch) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        C o = ShflDown(v, d);
        v = IS_MAX ? MaxNan(v, o) : v + o;
    }
    const int wave = threadIdx.x >> 6;
    __syncthreads();  // scratch may still be read from a previous reduction
    if ((threadIdx.x & 63) == 0) scratch[wave] = v;
    __syncthreads();
    C r = scratch[0];
#pragma unroll
    for (int w = 1; w < NT / 64; ++w) r = IS_MAX ? MaxNan(r, scratch[w]) : r + scratch[w];
    return r;
}

template <typename T, int V>
struct alignas(sizeof(T) * V) Pack {
    T e[V];
};

// 16 bytes at any address: rows of odd length start anywhere, and the hardware takes vector accesses there too.
template <typename T, int V>
__device__ __forceinline__ Pack<T, V> LoadPack(const T* p) {
    Pack<T, V> v;
    __builtin_memcpy(&v, p, sizeof(v));
    return v;
}
template <typename T, int V>
__device__ __forceinline__ void StorePack(T* p, const Pack<T, V>& v) {
    __builtin_memcpy(p, &v, sizeof(v));
}

// ---- LogSoftmax, rows that fit in registers: a workgroup of 256 to a row, or a wave to each of four, VPT packs of 16 bytes per thread.  The row's last
// pack moves back over its neighbour's elements, which are counted once and written twice with the same values: no access is conditional.
// Bound by its bytes where rows are many: float32/float16 in us, rows taken element by element before, 64000 x 300 74/53 -> 31/31.5, 50000 x 1001 122/129 -> 73/43
// (a read and a write: 69/35), 5398 x 1158 23.8 -> 14.7; by its start where they are few: 333 x 1001 3.1. ----
template <typename T, int NT, int VPT>
__global__ __launch_bounds__(256) void LogSoftmaxRowKernel(const T* x, T* out, int64_t rows, int n, int64_t x_row, int64_t o_row) {
    using C = compute_t<T>;
    constexpr int V = 16 / sizeof(T);
    __shared__ C scratch[4];
    const int t = threadIdx.x % NT;
    const int64_t row = static_cast<int64_t>(blockIdx.x) * (256 / NT) + threadIdx.x / NT;
    if (NT == 64 && row >= rows) return;  // a whole wave
    auto reduce = [&](C v, auto is_max) {
        constexpr bool MAX = decltype(is_max)::value;
        if constexpr (NT == 256) {
            return BlockReduce<C, 256, MAX>(v, scratch);
        } else {
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) {
                const C o = static_cast<C>(__shfl_xor(v, d, 64));
                v = MAX ? MaxNan(v, o) : v + o;
            }
            return v;
        }
    };
    const T* xr = x + row * x_row;
    T* orow = out + row * o_row;
    Pack<T, V> v[VPT];
    int at[VPT], skip[VPT];  // of a pack, elements of the one in front
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int e0 = (i * NT + t) * V;
        at[i] = min(e0, n - V);
        skip[i] = e0 - at[i];
        v[i] = LoadPack<T, V>(xr + at[i]);
    }
    C m = -INFINITY;
#pragma unroll
    for (int i = 0; i < VPT; ++i)
#pragma unroll
        for (int j = 0; j < V; ++j) {
            if (j >= skip[i]) m = MaxNan(m, static_cast<C>(v[i].e[j]));
        }
    m = reduce(m, std::true_type{});
    C s = 0;
#pragma unroll
    for (int i = 0; i < VPT; ++i)
#pragma unroll
        for (int j = 0; j < V; ++j) {
            const C e = ExpOf<C>(static_cast<C>(v[i].e[j]) - m);
            s += j >= skip[i] ? e : C(0);
        }
    s = reduce(s, std::false_type{});
    const C lse = m + LogOf<C>(s);
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        if (skip[i] >= V) continue;
        Pack<T, V> p;
#pragma unroll
        for (int j = 0; j < V; ++j) p.e[j] = static_cast<T>(static_cast<C>(v[i].e[j]) - lse);
        StorePack<T, V>(orow + at[i], p);
    }
}

// ---- LogSoftmax, short rows: LPR lanes of a wave hold a row of at most 16 * LPR elements (MAXE per lane), 64 / LPR rows to a wave.
// A wave per row leaves most lanes without an element when rows are classes (10, 16, ...) and is bounded by the launch of its
// workgroups: [65536, 16] float32 ran 65536 of them. ----
template <typename T, int LPR>
__global__ __launch_bounds__(256) void LogSoftmaxShortRowKernel(const T* x, T* out, int64_t rows, int n, int64_t x_row, int64_t o_row) {
    using C = compute_t<T>;
    constexpr int MAXE = 4;
    const int64_t row = static_cast<int64_t>(blockIdx.x) * (256 / LPR) + threadIdx.x / LPR;
    const int lane = threadIdx.x % LPR;
    if (row >= rows) return;  // whole groups of LPR lanes leave: the shuffles below stay inside a group
    const T* xr = x + row * x_row;
    C v[MAXE];
    C m = -INFINITY;
#pragma unroll
    for (int i = 0; i < MAXE; ++i) {
        const int e = i * LPR + lane;
        v[i] = e < n ? static_cast<C>(xr[e]) : static_cast<C>(-INFINITY);
        if (e < n) m = MaxNan(m, v[i]);
    }
#pragma unroll
    for (int d = LPR / 2; d >= 1; d >>= 1) m = MaxNan(m, static_cast<C>(__shfl_xor(m, d, LPR)));
    C s = 0;
#pragma unroll
    for (int i = 0; i < MAXE; ++i) {
        if (i * LPR + lane < n) s += ExpOf<C>(v[i] - m);
    }
#pragma unroll
    for (int d = LPR / 2; d >= 1; d >>= 1) s += static_cast<C>(__shfl_xor(s, d, LPR));
    const C lse = m + LogOf<C>(s);
    T* orow = out + row * o_row;
#pragma unroll
    for (int i = 0; i < MAXE; ++i) {
        if (i * LPR + lane < n) orow[i * LPR + lane] = static_cast<T>(v[i] - lse);
    }
}

// ---- LogSoftmax, long rows: pass 1 leaves (max, sum of exp(x - max)) per (row, segment); pass 2 merges a row's
// segments, then rewrites its own segment ----
constexpr int kSegThreads = 256;

// A segment in packs of 16 bytes, wherever it starts, its last elements one by one.
template <typename T, typename F>
__device__ __forceinline__ void ForSegment(const T* xr, int64_t lo, int64_t hi, F&& f) {
    constexpr int V = 16 / sizeof(T);
    const int64_t full = lo + (hi - lo) / V * V;
#pragma unroll 4
    for (int64_t e = lo + static_cast<int64_t>(threadIdx.x) * V; e < full; e += kSegThreads * V) {
        const Pack<T, V> p = LoadPack<T, V>(xr + e);
#pragma unroll
        for (int j = 0; j < V; ++j) f(p.e[j]);
    }
    for (int64_t e = full + threadIdx.x; e < hi; e += kSegThreads) f(xr[e]);
}

template <typename T>
__global__ __launch_bounds__(kSegThreads) void LogSoftmaxPartialKernel(const T* x, compute_t<T>* part, int64_t n, int64_t x_row, int64_t seg_len,
                                                                       int nseg) {
    using C = compute_t<T>;
    __shared__ C scratch[kSegThreads / 64];
    const int row = blockIdx.x / nseg, seg = blockIdx.x - row * nseg;
    const T* xr = x + static_cast<int64_t>(row) * x_row;
    const int64_t lo = seg * seg_len, hi = min(n, lo + seg_len);
    C m = -INFINITY;
    ForSegment<T>(xr, lo, hi, [&](T v) { m = MaxNan(m, static_cast<C>(v)); });
    m = BlockReduce<C, kSegThreads, true>(m, scratch);
    C s = 0;
    ForSegment<T>(xr, lo, hi, [&](T v) { s += ExpOf<C>(static_cast<C>(v) - m); });  // second walk hits L2
    s = BlockReduce<C, kSegThreads, false>(s, scratch);
    // a segment of -inf only: its terms are exp(-inf - rowmax) = 0 unless the whole row is -inf (then 0 * exp(NaN) = NaN below,
    // which is what the chain gives for such a row)
    if (m == static_cast<C>(-INFINITY)) s = 0;
    if (threadIdx.x == 0) {
        part[2 * static_cast<int64_t>(blockIdx.x)] = m;
        part[2 * static_cast<int64_t>(blockIdx.x) + 1] = s;
    }
}

template <typename T>
__global__ __launch_bounds__(kSegThreads) void LogSoftmaxApplyKernel(const T* x, T* out, const compute_t<T>* part, int64_t n, int64_t x_row,
                                                                     int64_t o_row, int64_t seg_len, int nseg) {
    using C = compute_t<T>;
    constexpr int V = 16 / sizeof(T);
    __shared__ C scratch[kSegThreads / 64];
    const int row = blockIdx.x / nseg, seg = blockIdx.x - row * nseg;
    const C* pr = part + 2 * static_cast<int64_t>(row) * nseg;
    C m = -INFINITY;
    for (int i = threadIdx.x; i < nseg; i += kSegThreads) m = MaxNan(m, pr[2 * i]);
    m = BlockReduce<C, kSegThreads, true>(m, scratch);
    C s = 0;
    for (int i = threadIdx.x; i < nseg; i += kSegThreads) {
        C mi = pr[2 * i], si = pr[2 * i + 1];
        s += si * ExpOf<C>(mi - m);
    }
    s = BlockReduce<C, kSegThreads, false>(s, scratch);
    const C lse = m + LogOf<C>(s);
    const T* xr = x + static_cast<int64_t>(row) * x_row;
    T* orow = out + static_cast<int64_t>(row) * o_row;
    const int64_t lo = seg * seg_len, hi = min(n, lo + seg_len);
    const int64_t full = lo + (hi - lo) / V * V;
#pragma unroll 4
    for (int64_t e = lo + static_cast<int64_t>(threadIdx.x) * V; e < full; e += kSegThreads * V) {
        Pack<T, V> p = LoadPack<T, V>(xr + e);
#pragma unroll
        for (int j = 0; j < V; ++j) p.e[j] = static_cast<T>(static_cast<C>(p.e[j]) - lse);
        StorePack<T, V>(orow + e, p);
    }
    for (int64_t e = full + threadIdx.x; e < hi; e += kSegThreads) orow[e] = static_cast<T>(static_cast<C>(xr[e]) - lse);
}

constexpr int64_t kRowInRegisters = 16384 * 4;  // bytes of a row the register kernel holds (256 threads x 16 packs x 16 bytes)
constexpr int64_t kSegmentBytes = 64 * 1024;

struct LsmShape {
    int64_t rows, n;
    int64_t x_row, o_row;  // element strides
};

LsmShape CheckLogSoftmax(const hipcx_array* x, const hipcx_array* out) {
    ValidateArray(x, "x");
    ValidateArray(out, "out");
    HIPCX_REQUIRE(IsFloatDtype(x->dtype), HIPCX_DTYPE_ERROR, std::string("log_softmax: floating point dtype required, got ") + DtypeName(x->dtype));
    HIPCX_REQUIRE(x->dtype == out->dtype, HIPCX_DTYPE_ERROR, "log_softmax: out must have x's dtype");
    HIPCX_REQUIRE(x->ndim == 2 && SameShape(x, out), HIPCX_DIMENSION_ERROR, "log_softmax: x and out must be 2-D of one shape (softmax axis 1)");
    const int64_t it = ItemSize(x->dtype);
    HIPCX_REQUIRE((x->shape[1] <= 1 || (x->strides[1] == it && out->strides[1] == it)) && x->strides[0] % it == 0 && out->strides[0] % it == 0 &&
                          x->strides[0] >= 0 && out->strides[0] >= 0,
                  HIPCX_NOT_IMPLEMENTED_ERROR, "log_softmax: rows must be dense along axis 1");
    return LsmShape{x->shape[0], x->shape[1], x->strides[0] / it, out->strides[0] / it};
}

// Rows of one launch: a grid holds less than 2^32 threads, at most 256 of them (and two or more segments) to a row.  More rows than
// these take several launches, each of them far longer than its start.
constexpr int64_t kRowsPerLaunch = int64_t{1} << 21;

// Elements of a segment of rows of n: rows that are few are cut into more of them, two workgroups to a compute unit, of at least 16 KiB: a row of
// 64 KiB segments kept one compute unit busy for each (7 x 70001 float32: 33 us, 9.5 now; 3 x 1000000: 19.5, 13.3; 100000: 16.3, 9.3).
int64_t LogSoftmaxSegment(int64_t rows, int64_t n, int64_t it) {
    const int64_t want = std::max<int64_t>(1, 2 * NumCUs() / rows), most = kSegmentBytes / it, least = kSegmentBytes / 4 / it;
    return std::min(most, std::max(least, ((n + want - 1) / want + 15) / 16 * 16));
}
// Whether rows go through segments: those beyond a workgroup's registers, and 16-bit ones as long as these in elements that are too few to occupy the chip
// (20 x 30000 float16: 8.9 us, 12.8 in registers; 37 x 20011: 9.8 and 10.3; 64 x 16000: 11.1 and 9.1).
bool LogSoftmaxInSegments(int64_t rows, int64_t n, int64_t it) {
    return n * it > kRowInRegisters || (rows <= 64 && n > kRowInRegisters / 4);
}

template <typename T>
void RunLogSoftmax(const T* xp, T* op, const LsmShape& sh, void* workspace, size_t workspace_bytes, hipStream_t stream) {
    constexpr int V = 16 / sizeof(T);
    constexpr int64_t it = sizeof(T);
    const int64_t packs = (sh.n + V - 1) / V;
    auto short_rows = [&](auto lpr) {
        constexpr int LPR = decltype(lpr)::value;
        const int64_t blocks = (sh.rows + 256 / LPR - 1) / (256 / LPR);
        hipLaunchKernelGGL((LogSoftmaxShortRowKernel<T, LPR>), dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, xp, op, sh.rows,
                           static_cast<int>(sh.n), sh.x_row, sh.o_row);
    };
    auto rows = [&](auto threads, auto per_thread) {
        constexpr int NT = decltype(threads)::value, VPT = decltype(per_thread)::value;
        const int64_t blocks = (sh.rows + 256 / NT - 1) / (256 / NT);
        hipLaunchKernelGGL((LogSoftmaxRowKernel<T, NT, VPT>), dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, xp, op, sh.rows, static_cast<int>(sh.n),
                           sh.x_row, sh.o_row);
    };
    auto segments = [&](int64_t seg_len) { return (sh.n + seg_len - 1) / seg_len; };
    auto bytes = [&](int64_t nseg) { return static_cast<size_t>(sh.rows * nseg) * 2 * sizeof(compute_t<T>); };
    int64_t seg_len = LogSoftmaxSegment(sh.rows, sh.n, it);
    bool cut = LogSoftmaxInSegments(sh.rows, sh.n, it);
    if (cut && (workspace == nullptr || workspace_bytes < bytes(segments(seg_len)))) {  // the fewest that do, then
        seg_len = kSegmentBytes / it;
        cut = sh.n * it > kRowInRegisters;
    }
    using std::integral_constant;
    const bool many = sh.rows >= 2048;  // workgroups of four waves to a row otherwise (3000 x 1000: 6.2 us, 7.0 with them; 1500 x 2000: 7.1, 6.4)
    // up to four elements to a lane: beyond 128 of them a row fills a wave with 16-byte loads
    if (sh.n <= 16) {
        short_rows(integral_constant<int, 4>{});
    } else if (sh.n <= 64) {
        short_rows(integral_constant<int, 16>{});
    } else if (sh.n <= 128) {
        short_rows(integral_constant<int, 32>{});
    } else if (cut) {
        const int64_t nseg = segments(seg_len);
        HIPCX_REQUIRE(sh.rows * nseg < (1LL << 31), HIPCX_NOT_IMPLEMENTED_ERROR, "log_softmax: problem too large for one launch");
        const size_t need = bytes(nseg);
        HIPCX_REQUIRE(workspace != nullptr && workspace_bytes >= need, HIPCX_CHAINERX_ERROR,
                      "log_softmax: workspace of " + std::to_string(need) + " bytes required");
        auto* part = static_cast<compute_t<T>*>(workspace);
        const unsigned blocks = static_cast<unsigned>(sh.rows * nseg);
        hipLaunchKernelGGL(LogSoftmaxPartialKernel<T>, dim3(blocks), dim3(kSegThreads), 0, stream, xp, part, sh.n, sh.x_row, seg_len, static_cast<int>(nseg));
        CheckLaunch("log_softmax_partial");
        hipLaunchKernelGGL(LogSoftmaxApplyKernel<T>, dim3(blocks), dim3(kSegThreads), 0, stream, xp, op, part, sh.n, sh.x_row, sh.o_row, seg_len,
                           static_cast<int>(nseg));
    } else if (packs <= 64) {
        rows(integral_constant<int, 64>{}, integral_constant<int, 1>{});
    } else if (many && packs <= 128) {
        rows(integral_constant<int, 64>{}, integral_constant<int, 2>{});
    } else if (many && packs <= 256) {
        rows(integral_constant<int, 64>{}, integral_constant<int, 4>{});
    } else if (many && packs <= 512) {
        rows(integral_constant<int, 64>{}, integral_constant<int, 8>{});
    } else if (packs <= 256) {
        rows(integral_constant<int, 256>{}, integral_constant<int, 1>{});
    } else if (packs <= 256 * 2) {
        rows(integral_constant<int, 256>{}, integral_constant<int, 2>{});
    } else if (packs <= 256 * 4) {
        rows(integral_constant<int, 256>{}, integral_constant<int, 4>{});
    } else if (packs <= 256 * 10) {
        rows(integral_constant<int, 256>{}, integral_constant<int, 10>{});
    } else {
        rows(integral_constant<int, 256>{}, integral_constant<int, 16>{});
    }
    CheckLaunch("log_softmax");
}

// ---- softmax cross entropy ----
// What a row contributes is the score of its label, x[label] - (max + log(sum of exponentials)).  The chain multiplies every score
// with a 0 / 1 mask, so a score of -inf elsewhere in the row turns the sum into NaN (0 * inf): the smallest other score is kept to see
// that.  Every element is read once, 16 bytes per access at any address, and held in registers between the maximum and the sum.
// Three shapes (PlanXent); us, against a wave to a row with one element per lane and step, twice over (and the chain of 15 kernels):
//   XentKernel       short rows in the registers of 16 lanes or a wave.  One workgroup does a small batch alone; others leave partial
//                    sums for XentFinishKernel.  Bound by the latency of a few loads and the exponentials behind them.  float32
//                    [100,10] 4.5 -> 4.4 (53), [1000,10] 18 -> 6.0 (60), [900,18] 70 -> 6.1 (60), [128,1000] 10.4 -> 6.6 (60),
//                    [20000,1500] 58 -> 38 (332).
//   XentBlockKernel  longer rows, a workgroup to a row: bound by memory and, at few packs to a thread, by its three reductions.
//                    [4480,10000] 121 -> 72 (482).  Rows too few to fill the chip are cut into segments, each a workgroup's, which
//                    XentMergeKernel puts together in double: [128,10000] 51 -> 12 (65), [1,1000000] 3878 -> 11 (65).
struct XentArgs {
    const void* x;
    const void* t;
    void* out;
    double* partial;  // XentBlockKernel with segments: {maximum, sum, least other} of each; else {sum of scores, labels} per workgroup, or
                      // null: one workgroup writes the result itself
    int64_t rows, n, x_row, t_stride;
    int t_dtype;
    int nseg;         // segments of a row
    int64_t seg_len;  // elements, a multiple of 16 bytes
};

__device__ __forceinline__ int64_t LoadInteger(const void* t, int64_t i, int dtype) {
    switch (dtype) {
        case HIPCX_INT8: return static_cast<const int8_t*>(t)[i];
        case HIPCX_INT16: return static_cast<const int16_t*>(t)[i];
        case HIPCX_INT32: return static_cast<const int32_t*>(t)[i];
        case HIPCX_UINT8: return static_cast<const uint8_t*>(t)[i];
        default: return static_cast<const int64_t*>(t)[i];
    }
}

// The label of a row, -1 where it names no class.
__device__ __forceinline__ int64_t LoadLabel(const XentArgs& p, int64_t row) {
    const int64_t label = LoadInteger(p.t, row * p.t_stride, p.t_dtype);
    return label >= 0 && label < p.n ? label : -1;
}

// -sum / count with the roundings of Sum, Sum, Divide(-1, .) and Multiply.
template <typename T>
__device__ __forceinline__ T XentResult(double sum, double count) {
    using C = compute_t<T>;
    const C s = static_cast<C>(static_cast<T>(sum)), n = static_cast<C>(static_cast<T>(count));
    const C factor = static_cast<C>(static_cast<T>(C(-1) / n));
    return static_cast<T>(s * factor);
}

// Adds up (a, b) of all threads of a workgroup; valid in thread 0.
template <int NT>
__device__ __forceinline__ void BlockSum2(double& a, double& b, double (*scratch)[2]) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        a += ShflDown(a, d);
        b += ShflDown(b, d);
    }
    if ((threadIdx.x & 63) == 0) {
        scratch[threadIdx.x >> 6][0] = a;
        scratch[threadIdx.x >> 6][1] = b;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < NT / 64; ++w) {
            a += scratch[w][0];
            b += scratch[w][1];
        }
    }
}

template <typename T, int V>
struct __attribute__((packed, aligned(sizeof(T)))) AnyPack {
    T e[V];
};

// Elements [lo, end) of a row (end >= V), U packs of V to a lane, LANES lanes side by side.  The last pack moves back to end at `end`:
// its first skip[u] elements are not this lane's (all V beyond the end).
template <typename T, int V, int U, int LANES>
struct XentShare {
    using C = compute_t<T>;
    C v[U][V];
    int skip[U];

    __device__ __forceinline__ void Load(const T* xr, int64_t lo, int64_t end, int lane) {
        AnyPack<T, V> p[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t first = lo + static_cast<int64_t>(u * LANES + lane) * V;
            const int64_t from = first < end - V ? first : end - V;
            skip[u] = static_cast<int>(first - from < V ? first - from : V);
            p[u] = *reinterpret_cast<const AnyPack<T, V>*>(xr + from);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int j = 0; j < V; ++j) v[u][j] = static_cast<C>(p[u].e[j]);
    }

    // The maximum, and the least of the elements other than `label`.
    __device__ __forceinline__ void Extremes(int64_t lo, int64_t end, int lane, int64_t label, C& m, C& least) const {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (u > 0 && lo + u * LANES * V >= end) break;  // (the same for all lanes)
            const int64_t first = lo + static_cast<int64_t>(u * LANES + lane) * V;
            const int64_t at = label - (first < end - V ? first : end - V);
#pragma unroll
            for (int j = 0; j < V; ++j) {
                if (j < skip[u]) continue;
                m = MaxNan(m, v[u][j]);
                if (j != at && v[u][j] < least) least = v[u][j];
            }
        }
    }

    __device__ __forceinline__ C SumExp(int64_t lo, int64_t end, C m) const {
        C s = 0;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (u > 0 && lo + u * LANES * V >= end) break;
#pragma unroll
            for (int j = 0; j < V; ++j) s += j >= skip[u] ? ExpOf<C>(v[u][j] - m) : C(0);
        }
        return s;
    }
};

// Adds a row's contribution, with the roundings of LogSoftmax, Multiply and Sum.
template <typename T>
__device__ __forceinline__ void XentAddRow(const T* xr, int64_t n, int64_t label, compute_t<T> m, compute_t<T> s, compute_t<T> least, double& sum,
                                           double& count) {
    using C = compute_t<T>;
    const C lse = m + LogOf<C>(s);
    const bool counts = label >= 0;
    C score = counts ? static_cast<C>(static_cast<T>(static_cast<C>(xr[label]) - lse)) : C(0);
    if (n > (counts ? 1 : 0)) score += static_cast<C>(static_cast<T>(least - lse)) * C(0);
    sum += static_cast<double>(score);
    count += counts ? 1.0 : 0.0;
}

// The workgroup's {sum of scores, labels}, or the result itself.
template <typename T, int NT>
__device__ __forceinline__ void XentStore(const XentArgs& p, double sum, double count) {
    __shared__ double scratch[NT / 64][2];
    BlockSum2<NT>(sum, count, scratch);
    if (threadIdx.x != 0) return;
    if (p.partial != nullptr) {
        p.partial[2 * blockIdx.x] = sum;
        p.partial[2 * blockIdx.x + 1] = count;
    } else {
        *static_cast<T*>(p.out) = XentResult<T>(sum, count);
    }
}

// E elements of a row to each of LPR lanes.
template <typename T, int LPR, int E, int NT>
__global__ __launch_bounds__(NT) void XentKernel(XentArgs p) {
    using C = compute_t<T>;
    constexpr int V = E * sizeof(T) < 16 ? E : 16 / sizeof(T), U = E / V;
    const int lane = threadIdx.x % LPR;
    double sum = 0, count = 0;
    for (int64_t row = static_cast<int64_t>(blockIdx.x) * (NT / LPR) + threadIdx.x / LPR; row < p.rows; row += static_cast<int64_t>(gridDim.x) * (NT / LPR)) {
        const T* xr = static_cast<const T*>(p.x) + row * p.x_row;
        const int64_t label = LoadLabel(p, row);
        XentShare<T, V, U, LPR> share;
        share.Load(xr, 0, p.n, lane);
        C m = -INFINITY, least = INFINITY;
        share.Extremes(0, p.n, lane, label, m, least);
#pragma unroll
        for (int d = LPR / 2; d >= 1; d >>= 1) {
            m = MaxNan(m, static_cast<C>(__shfl_xor(m, d, LPR)));
            const C o = static_cast<C>(__shfl_xor(least, d, LPR));
            least = o < least ? o : least;
        }
        C s = share.SumExp(0, p.n, m);
#pragma unroll
        for (int d = LPR / 2; d >= 1; d >>= 1) s += static_cast<C>(__shfl_xor(s, d, LPR));
        if (lane == 0) XentAddRow<T>(xr, p.n, label, m, s, least, sum, count);
    }
    XentStore<T, NT>(p, sum, count);
}

// s * exp(m - to) of a part of a row; a part of -inf alone has no terms (or the whole row has none, and the score becomes NaN).
__device__ __forceinline__ double Rescaled(double s, double m, double to) { return m == -INFINITY ? 0.0 : s * exp(m - to); }

constexpr int kXentThreads = 256;

// U packs of a row to a thread at a time.
template <typename T, int U>
__global__ __launch_bounds__(kXentThreads) void XentBlockKernel(XentArgs p) {
    using C = compute_t<T>;
    constexpr int V = 16 / sizeof(T);
    constexpr int64_t CHUNK = kXentThreads * U * V;
    __shared__ C scratch[kXentThreads / 64];
    double sum = 0, count = 0;
    for (int64_t part = blockIdx.x; part < p.rows * p.nseg; part += gridDim.x) {
        const int64_t row = part / p.nseg, lo = (part - row * p.nseg) * p.seg_len, hi = min(p.n, lo + p.seg_len);
        const T* xr = static_cast<const T*>(p.x) + row * p.x_row;
        const int64_t label = LoadLabel(p, row);
        C m = -INFINITY, least = INFINITY;
        double s = 0;  // of exp(x - m), so far
        for (int64_t from = lo; from < hi; from += CHUNK) {
            const int64_t end = min(hi, from + CHUNK);
            XentShare<T, V, U, kXentThreads> share;
            share.Load(xr, from, end, threadIdx.x);
            C mc = -INFINITY;
            share.Extremes(from, end, threadIdx.x, label, mc, least);
            mc = BlockReduce<C, kXentThreads, true>(mc, scratch);
            const C sc = BlockReduce<C, kXentThreads, false>(share.SumExp(from, end, mc), scratch);
            const C both = MaxNan(m, mc);
            s = hi - lo <= CHUNK && mc != static_cast<C>(-INFINITY) ? static_cast<double>(sc) : Rescaled(s, m, both) + Rescaled(sc, mc, both);
            m = both;
        }
        least = -BlockReduce<C, kXentThreads, true>(-least, scratch);
        if (threadIdx.x == 0) {
            if (p.nseg > 1) {
                p.partial[3 * part] = m;
                p.partial[3 * part + 1] = s;
                p.partial[3 * part + 2] = least;
            } else {
                XentAddRow<T>(xr, p.n, label, m, static_cast<C>(s), least, sum, count);
            }
        }
    }
    if (p.nseg == 1) XentStore<T, kXentThreads>(p, sum, count);
}

// The result of rows in segments: LPR lanes put a row together.
template <typename T, int LPR>
__global__ __launch_bounds__(1024) void XentMergeKernel(XentArgs p) {
    using C = compute_t<T>;
    const int lane = threadIdx.x % LPR;
    double sum = 0, count = 0;
    for (int64_t row = threadIdx.x / LPR; row < p.rows; row += 1024 / LPR) {
        const double* part = p.partial + 3 * row * p.nseg;
        double m = -INFINITY, least = INFINITY, s = 0;
#pragma unroll 4
        for (int i = lane; i < p.nseg; i += LPR) {
            m = MaxNan(m, part[3 * i]);
            least = part[3 * i + 2] < least ? part[3 * i + 2] : least;
        }
#pragma unroll
        for (int d = LPR / 2; d >= 1; d >>= 1) {
            m = MaxNan(m, __shfl_xor(m, d, LPR));
            const double o = __shfl_xor(least, d, LPR);
            least = o < least ? o : least;
        }
#pragma unroll 4
        for (int i = lane; i < p.nseg; i += LPR) s += Rescaled(part[3 * i + 1], part[3 * i], m);
#pragma unroll
        for (int d = LPR / 2; d >= 1; d >>= 1) s += __shfl_xor(s, d, LPR);
        if (lane == 0) {
            XentAddRow<T>(static_cast<const T*>(p.x) + row * p.x_row, p.n, LoadLabel(p, row), static_cast<C>(m),
                          static_cast<C>(s), static_cast<C>(least), sum, count);
        }
    }
    p.partial = nullptr;
    XentStore<T, 1024>(p, sum, count);
}

template <typename T>
__global__ __launch_bounds__(256) void XentFinishKernel(XentArgs p, int n_partial) {
    double sum = 0, count = 0;
    for (int i = threadIdx.x; i < n_partial; i += 256) {
        sum += p.partial[2 * i];
        count += p.partial[2 * i + 1];
    }
    p.partial = nullptr;
    XentStore<T, 256>(p, sum, count);
}

struct XentPlan {
    int blocks = 1;
    int nseg = 0;  // 0: XentKernel
    int64_t seg_len = 0;
    size_t Bytes() const { return nseg > 1 ? static_cast<size_t>(blocks) * 3 * sizeof(double) : blocks > 1 ? static_cast<size_t>(blocks) * 2 * sizeof(double) : 0; }
};

// Rows of at most 64 elements or 4 KB, 8 KB where there are four for every compute unit: XentKernel.  One workgroup does the batch alone
// while that costs no more than a second launch and the memory for partial sums between the two, 2 us on the device and 5 on the host:
// [512,10] float32 9.7 us alone, 6.0 in two; [256,40] 7.3, [64,256] 8.1, [32,1000] 9.4 against 6.0-6.5.  Else a workgroup of four waves
// to every four (16 short) rows, up to eight to a compute unit.
// Longer rows: a workgroup each once there is one for every compute unit ([20000,1500] float32 would take 71 us so, 38 as waves), else
// segments of 8 KB and more, up to four to a compute unit ([1,1000000] with 4 KB: 21 us, 11 with 8: the merge is one workgroup's).
XentPlan PlanXent(int64_t rows, int64_t n, int64_t item) {
    XentPlan pl;
    if (n <= 64 || n * item <= (rows >= 4 * NumCUs() ? 8192 : 4096)) {
        const int64_t lpr = n <= 64 ? 16 : 64;
        const int64_t alone = n <= 16 ? 512 : n <= 64 ? 256 : n <= 256 ? 64 : 32;  // rows
        if (rows > alone) pl.blocks = static_cast<int>(std::min<int64_t>((rows * lpr + 255) / 256, int64_t{8} * NumCUs()));
        return pl;
    }
    if (rows >= NumCUs()) {
        pl.nseg = 1;
        pl.seg_len = n;
        pl.blocks = static_cast<int>(std::min<int64_t>(rows, int64_t{8} * NumCUs()));
        return pl;
    }
    const int64_t vec = 16 / item, most = (n * item + 8191) / 8192;
    const int64_t segments = std::min<int64_t>((int64_t{4} * NumCUs() + rows - 1) / rows, most);
    pl.seg_len = ((n + segments - 1) / segments + vec - 1) / vec * vec;
    pl.nseg = static_cast<int>((n + pl.seg_len - 1) / pl.seg_len);
    pl.blocks = static_cast<int>(rows) * pl.nseg;
    return pl;
}

// f(E) for the least power of two E of at least n / lanes elements to a lane.
template <int E, int MOST, typename F>
void ForElementsPerLane(int64_t n, int lanes, F&& f) {
    if constexpr (E < MOST) {
        if (n > static_cast<int64_t>(E) * lanes) return ForElementsPerLane<2 * E, MOST>(n, lanes, f);
    }
    f(std::integral_constant<int, E>{});
}

template <typename T>
void LaunchXent(const XentArgs& p, const XentPlan& plan, hipStream_t stream) {
    constexpr int V = 16 / sizeof(T);
    const dim3 grid(plan.blocks);
    if (plan.nseg > 0) {
        const int64_t packs = (p.seg_len + V - 1) / V;
        if (packs <= 2 * kXentThreads) hipLaunchKernelGGL((XentBlockKernel<T, 2>), grid, dim3(kXentThreads), 0, stream, p);
        else if (packs <= 4 * kXentThreads) hipLaunchKernelGGL((XentBlockKernel<T, 4>), grid, dim3(kXentThreads), 0, stream, p);
        else hipLaunchKernelGGL((XentBlockKernel<T, 8>), grid, dim3(kXentThreads), 0, stream, p);
    } else if (p.n <= 64) {
        ForElementsPerLane<1, 4>(p.n, 16, [&](auto e) {
            constexpr int E = decltype(e)::value;
            if (plan.blocks == 1) hipLaunchKernelGGL((XentKernel<T, 16, E, 1024>), grid, dim3(1024), 0, stream, p);
            else hipLaunchKernelGGL((XentKernel<T, 16, E, 256>), grid, dim3(256), 0, stream, p);
        });
    } else {
        ForElementsPerLane<2, 8 * V>(p.n, 64, [&](auto e) {
            constexpr int E = decltype(e)::value;
            if (plan.blocks == 1) hipLaunchKernelGGL((XentKernel<T, 64, E, 1024>), grid, dim3(1024), 0, stream, p);
            else hipLaunchKernelGGL((XentKernel<T, 64, E, 256>), grid, dim3(256), 0, stream, p);
        });
    }
    CheckLaunch("softmax_cross_entropy");
    if (plan.nseg > 1) {
        if (plan.nseg <= 16) hipLaunchKernelGGL((XentMergeKernel<T, 16>), dim3(1), dim3(1024), 0, stream, p);
        else hipLaunchKernelGGL((XentMergeKernel<T, 64>), dim3(1), dim3(1024), 0, stream, p);
        CheckLaunch("softmax_cross_entropy_merge");
    } else if (plan.blocks > 1) {
        hipLaunchKernelGGL((XentFinishKernel<T>), dim3(1), dim3(256), 0, stream, p, plan.blocks);
        CheckLaunch("softmax_cross_entropy_finish");
    }
}

// ---- Lstm cell ----
template <typename T>
__global__ __launch_bounds__(256) void LstmCellKernel(const T* c, const T* x, T* h_out, T* c_out, int64_t total, int H, int64_t c_row, int64_t x_row,
                                                      int64_t h_row, int64_t co_row, int vec_ok) {
    using C = compute_t<T>;
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (idx >= total) return;
    const int64_t b = idx / H;
    const int j = static_cast<int>(idx - b * H);
    const T* xg = x + b * x_row + 4 * static_cast<int64_t>(j);
    C g[4];
    if (vec_ok) {
        Pack<T, 4> p = *reinterpret_cast<const Pack<T, 4>*>(xg);
#pragma unroll
        for (int k = 0; k < 4; ++k) g[k] = static_cast<C>(p.e[k]);
    } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) g[k] = static_cast<C>(xg[k]);
    }
    C cn;
    const C h = LstmCell<C>(g, static_cast<C>(c[b * c_row + j]), cn);
    c_out[b * co_row + j] = static_cast<T>(cn);
    h_out[b * h_row + j] = static_cast<T>(h);
}

}  // namespace
}  // namespace hipcx

using namespace hipcx;

extern "C" {

size_t hipcx_log_softmax_workspace_size(const hipcx_array* x) {
    if (x == nullptr || x->ndim != 2 || !IsFloatDtype(x->dtype)) return 0;
    const int64_t it = ItemSize(x->dtype);
    if (x->shape[0] == 0 || !LogSoftmaxInSegments(x->shape[0], x->shape[1], it)) return 0;
    const int64_t seg_len = LogSoftmaxSegment(x->shape[0], x->shape[1], it);
    const int64_t nseg = (x->shape[1] + seg_len - 1) / seg_len;
    return static_cast<size_t>(x->shape[0] * nseg) * 2 * (x->dtype == HIPCX_FLOAT64 ? 8 : 4);
}

int hipcx_log_softmax(const hipcx_array* x, const hipcx_array* out, void* workspace, size_t workspace_bytes, void* stream) {
    return Guard([&] {
        LsmShape sh = CheckLogSoftmax(x, out);
        if (sh.rows == 0 || sh.n == 0) return;
        VisitFloatDtype(x->dtype, [&](auto tag) {
            using T = typename decltype(tag)::type;
            for (int64_t row = 0; row < sh.rows; row += kRowsPerLaunch) {
                LsmShape part = sh;
                part.rows = std::min(kRowsPerLaunch, sh.rows - row);
                RunLogSoftmax<T>(static_cast<const T*>(x->data) + row * sh.x_row, static_cast<T*>(out->data) + row * sh.o_row, part, workspace,
                                 workspace_bytes, AsStream(stream));
            }
        });
    });
}

size_t hipcx_softmax_cross_entropy_workspace_size(const hipcx_array* x) {
    if (x == nullptr || x->ndim != 2 || x->shape[0] == 0 || x->shape[1] == 0) return 0;
    return PlanXent(x->shape[0], x->shape[1], ItemSize(x->dtype)).Bytes();
}

int hipcx_softmax_cross_entropy(const hipcx_array* x, const hipcx_array* t, const hipcx_array* out, void* workspace, size_t workspace_bytes,
                                void* stream) {
    return Guard([&] {
        ValidateArray(x, "x");
        ValidateArray(t, "t");
        ValidateArray(out, "out");
        HIPCX_REQUIRE(IsFloatDtype(x->dtype) && out->dtype == x->dtype, HIPCX_DTYPE_ERROR, "softmax_cross_entropy: x and out need one float dtype");
        HIPCX_REQUIRE(!IsFloatDtype(t->dtype) && t->dtype != HIPCX_BOOL, HIPCX_DTYPE_ERROR, "softmax_cross_entropy: labels need an integer dtype");
        HIPCX_REQUIRE(x->ndim == 2 && t->ndim == 1 && t->shape[0] == x->shape[0] && TotalSize(out) == 1, HIPCX_DIMENSION_ERROR,
                      "softmax_cross_entropy: x [B, n], t [B] and an out of one element are needed");
        const int64_t it = ItemSize(x->dtype);
        HIPCX_REQUIRE((x->shape[1] <= 1 || x->strides[1] == it) && x->strides[0] % it == 0 && t->strides[0] % ItemSize(t->dtype) == 0,
                      HIPCX_NOT_IMPLEMENTED_ERROR, "softmax_cross_entropy: rows must be dense along axis 1");
        XentArgs p{};
        p.x = x->data;
        p.t = t->data;
        p.out = out->data;
        p.rows = x->shape[0];
        p.n = x->shape[1];
        p.x_row = x->strides[0] / it;
        p.t_stride = t->strides[0] / ItemSize(t->dtype);
        p.t_dtype = t->dtype;
        if (p.n == 0) p.rows = 0;  // nothing to read, no label counts
        const XentPlan plan = p.rows > 0 ? PlanXent(p.rows, p.n, it) : XentPlan();
        p.nseg = plan.nseg;
        p.seg_len = plan.seg_len;
        if (plan.Bytes() > 0) {
            HIPCX_REQUIRE(workspace != nullptr && workspace_bytes >= plan.Bytes(), HIPCX_CHAINERX_ERROR,
                          "softmax_cross_entropy: workspace of " + std::to_string(plan.Bytes()) + " bytes required");
            p.partial = static_cast<double*>(workspace);
        }
        VisitFloatDtype(x->dtype, [&](auto tag) { LaunchXent<typename decltype(tag)::type>(p, plan, AsStream(stream)); });
    });
}

int hipcx_lstm_cell(const hipcx_array* c, const hipcx_array* x, const hipcx_array* h_out, const hipcx_array* c_out, void* stream) {
    return Guard([&] {
        ValidateArray(c, "c");
        ValidateArray(x, "x");
        ValidateArray(h_out, "h_out");
        ValidateArray(c_out, "c_out");
        HIPCX_REQUIRE(IsFloatDtype(c->dtype), HIPCX_DTYPE_ERROR, "Expected data type float");
        HIPCX_REQUIRE(c->dtype == x->dtype, HIPCX_DTYPE_ERROR, "Datatypes of c and x should be equal");
        HIPCX_REQUIRE(h_out->dtype == c->dtype && c_out->dtype == c->dtype, HIPCX_DTYPE_ERROR, "lstm_cell: outputs must have c's dtype");
        HIPCX_REQUIRE(c->ndim == 2 && x->ndim == 2, HIPCX_NOT_IMPLEMENTED_ERROR, "lstm_cell: 2-D c and x only");
        HIPCX_REQUIRE(x->shape[0] <= c->shape[0], HIPCX_DIMENSION_ERROR, "The batch size of x must be equal to or less than the size of c");
        HIPCX_REQUIRE(x->shape[1] == 4 * c->shape[1], HIPCX_DIMENSION_ERROR,
                      "Expected dimension at axis 1 of x to be equal 4 times dimension at axis 1 of c.");
        HIPCX_REQUIRE(x->shape[0] == c->shape[0], HIPCX_NOT_IMPLEMENTED_ERROR, "lstm_cell: ragged batches are not on the supported path");
        HIPCX_REQUIRE(SameShape(h_out, c) && SameShape(c_out, c), HIPCX_DIMENSION_ERROR, "lstm_cell: outputs must have c's shape");
        const int64_t it = ItemSize(c->dtype);
        auto dense_rows = [&](const hipcx_array* a) {
            return (a->shape[1] <= 1 || a->strides[1] == it) && a->strides[0] % it == 0 && a->strides[0] >= 0;
        };
        HIPCX_REQUIRE(dense_rows(c) && dense_rows(x) && dense_rows(h_out) && dense_rows(c_out), HIPCX_NOT_IMPLEMENTED_ERROR,
                      "lstm_cell: rows must be dense along axis 1");
        const int64_t B = c->shape[0], H = c->shape[1];
        const int64_t total = B * H;
        if (total == 0) return;
        HIPCX_REQUIRE(H < (1LL << 31), HIPCX_NOT_IMPLEMENTED_ERROR, "lstm_cell: problem too large for one launch");
        const int vec_ok = reinterpret_cast<uintptr_t>(x->data) % (4 * it) == 0 && x->strides[0] % (4 * it) == 0;
        const int64_t rows = std::max<int64_t>(1, (int64_t{1} << 31) / H);  // of one launch: a grid holds less than 2^32 threads
        VisitFloatDtype(c->dtype, [&](auto tag) {
            using T = typename decltype(tag)::type;
            const int64_t c_row = c->strides[0] / it, x_row = x->strides[0] / it, h_row = h_out->strides[0] / it, co_row = c_out->strides[0] / it;
            for (int64_t b = 0; b < B; b += rows) {
                const int64_t part = std::min(rows, B - b) * H;
                hipLaunchKernelGGL(LstmCellKernel<T>, dim3(static_cast<unsigned>((part + 255) / 256)), dim3(256), 0, AsStream(stream),
                                   static_cast<const T*>(c->data) + b * c_row, static_cast<const T*>(x->data) + b * x_row,
                                   static_cast<T*>(h_out->data) + b * h_row, static_cast<T*>(c_out->data) + b * co_row, part, static_cast<int>(H),
                                   c_row, x_row, h_row, co_row, vec_ok);
            }
        });
        CheckLaunch("lstm_cell");
    });
}

}  // extern "C"
