// Elementwise engine: one launcher for every map-style kernel (arithmetic, math, select, compare,
// cast-copy, fill).
//
// Host side: the operands' (shape, byte-strides) are normalised -- unit axes dropped, axes ordered
// by decreasing output stride (any common permutation is legal for a map), mergeable neighbours
// fused -- so that an NCHW view of channels-last memory, a broadcast row vector, or a transposed
// matrix all collapse to a "rows x cols" problem whenever their memory allows it.
//
// Device side: a thread handles up to kEwUnroll vectors of VEC elements (16 bytes of the widest operand), fewer when the array is
// small: bound by memory when large, by the latency of one load-compute-store round when small, and then the work wants to be
// spread over as many compute units as there are.  A row is cut into whole vectors from its start; where VEC does not divide it,
// the last unit loads the row's last VEC elements and stores only those its neighbour does not.  Addresses need no alignment (the
// hardware takes 16-byte accesses anywhere), so odd widths and offsets run at the speed of even ones: [333, 1001] float16
// relu 3.9 -> 2.6 us, the 49 of a ResNet-50 pass over one image 4.4 -> 2.7 us on average.  Operands whose inner stride is 0 are read once per vector as a scalar.  With VEC == 1 any inner
// stride is accepted.  More than two remaining axes are decomposed with div/mod per vector (not per element).
#pragma once

#include <algorithm>
#include <cstdlib>
#include <initializer_list>

#include "common.h"

namespace hipcx {

constexpr int kEwMaxOperands = 6;  // out + up to 5 inputs
constexpr int kEwThreads = 256;
constexpr int kEwUnroll = 4;

struct EwPlan {
    int nops = 0;  // operand 0 is the output
    int ndim = 0;  // after normalisation; 0 means a single element
    int64_t total = 0;
    int64_t shape[HIPCX_MAX_NDIM];
    int64_t strides[kEwMaxOperands][HIPCX_MAX_NDIM];  // bytes
    char* ptr[kEwMaxOperands];
    int64_t itemsize[kEwMaxOperands];
};

// Builds the normalised iteration plan.  All operands must have the same shape.
inline EwPlan MakeEwPlan(std::initializer_list<const hipcx_array*> ops) {
    EwPlan p;
    p.nops = static_cast<int>(ops.size());
    HIPCX_REQUIRE(p.nops >= 1 && p.nops <= kEwMaxOperands, HIPCX_CHAINERX_ERROR, "bad operand count");
    const hipcx_array* arr[kEwMaxOperands];
    int k = 0;
    for (const hipcx_array* a : ops) {
        ValidateArray(a, "operand");
        arr[k++] = a;
    }
    const hipcx_array* out = arr[0];
    for (int i = 1; i < p.nops; ++i) {
        HIPCX_REQUIRE(SameShape(out, arr[i]), HIPCX_DIMENSION_ERROR,
                      "operand shapes differ: " + ShapeStr(out) + " vs " + ShapeStr(arr[i]));
    }
    p.total = TotalSize(out);
    for (int i = 0; i < p.nops; ++i) {
        p.ptr[i] = static_cast<char*>(arr[i]->data);
        p.itemsize[i] = ItemSize(arr[i]->dtype);
    }
    // 1. drop unit axes
    int dims[HIPCX_MAX_NDIM];
    int nd = 0;
    for (int d = 0; d < out->ndim; ++d) {
        if (out->shape[d] != 1) dims[nd++] = d;
    }
    // 2. order by decreasing |out stride| (stable, so equal strides keep their logical order)
    std::stable_sort(dims, dims + nd, [&](int a, int b) { return std::llabs(out->strides[a]) > std::llabs(out->strides[b]); });
    // 3. merge neighbours that every operand walks as one run
    int m = 0;
    for (int j = 0; j < nd; ++j) {
        int d = dims[j];
        bool merged = false;
        if (m > 0) {
            merged = true;
            for (int i = 0; i < p.nops; ++i) {
                if (p.strides[i][m - 1] != out->shape[d] * arr[i]->strides[d]) {
                    merged = false;
                    break;
                }
            }
        }
        if (merged) {
            p.shape[m - 1] *= out->shape[d];
            for (int i = 0; i < p.nops; ++i) p.strides[i][m - 1] = arr[i]->strides[d];
        } else {
            p.shape[m] = out->shape[d];
            for (int i = 0; i < p.nops; ++i) p.strides[i][m] = arr[i]->strides[d];
            ++m;
        }
    }
    p.ndim = m;
    return p;
}

// Device-side view of the plan: `cols` is the innermost axis, the others are "outer" axes.
template <int NOPS>
struct EwArgs {
    char* ptr[NOPS];
    int64_t col_stride[NOPS];  // bytes between consecutive elements of the inner axis (0 = broadcast)
    int64_t outer_stride[NOPS][HIPCX_MAX_NDIM - 1];
    int64_t outer_shape[HIPCX_MAX_NDIM - 1];
    int n_outer;
    int64_t cols;   // elements
    int64_t cvecs;  // vectors per row, the last one overlapping its neighbour when VEC does not divide cols
    int64_t nvec;   // rows * cvecs
    int64_t index_base;  // C-order position of the first element (problems cut into several launches)
    int per_thread; // vectors per thread, 1 or kEwUnroll
    int stream_in;  // bit i + 1: input i is too large to stay in the last-level cache and is loaded without allocating there
};

template <typename T, int N>
struct alignas(sizeof(T) * N) Vec {
    T v[N];
};

// The bytes of a vector as machine words.  Loads keep them packed until every load of a thread has been issued: taken apart into
// elements where they are loaded, each would be waited for before the next is issued.
template <int BYTES>
struct RawOf;
template <>
struct RawOf<16> {
    using type = unsigned __attribute__((ext_vector_type(4)));
    typedef unsigned any_address __attribute__((ext_vector_type(4), aligned(1)));
};
template <>
struct RawOf<8> {
    using type = unsigned __attribute__((ext_vector_type(2)));
    typedef unsigned any_address __attribute__((ext_vector_type(2), aligned(1)));
};
template <>
struct RawOf<4> {
    using type = unsigned;
    typedef unsigned any_address __attribute__((aligned(1)));
};
template <>
struct RawOf<2> {
    using type = uint16_t;
    typedef uint16_t any_address __attribute__((aligned(1)));
};
template <>
struct RawOf<1> {
    using type = uint8_t;
    typedef uint8_t any_address;
};
template <typename V>
using raw_t = typename RawOf<sizeof(V)>::type;

// Vector access at any address.
template <typename V>
__device__ __forceinline__ raw_t<V> LoadRaw(const char* p) {
    return *reinterpret_cast<const typename RawOf<sizeof(V)>::any_address*>(p);
}

// A 16-byte vector load that does not allocate in the caches (other sizes: a plain load); the address is 16-byte aligned, because
// the compiler drops the non-temporal hint from a load of unknown alignment.  A tensor larger than the memory-side
// cache that is read front to back with allocating loads evicts its own tail -- the part the producer left there -- before reaching it.
template <typename V>
__device__ __forceinline__ raw_t<V> LoadStreaming(const char* p) {
    if constexpr (sizeof(V) == 16) {
        return __builtin_nontemporal_load(reinterpret_cast<const typename RawOf<16>::type*>(p));
    } else {
        return LoadRaw<V>(p);
    }
}

// One element in the first place of a vector; the others are filled in when it is used.
template <typename V>
__device__ __forceinline__ raw_t<V> LoadFirst(const char* p) {
    V v{};
    v.v[0] = *reinterpret_cast<const std::remove_reference_t<decltype(v.v[0])>*>(p);
    return __builtin_bit_cast(raw_t<V>, v);
}

template <typename T>
__device__ __forceinline__ compute_t<T> LoadAs(const char* p) {
    return static_cast<compute_t<T>>(*reinterpret_cast<const T*>(p));
}

// Type of the first input: Op::In0 when the op declares one (a bool condition in front of numeric operands), else Op::In.
template <typename Op, typename = void>
struct FirstInOf {
    using type = typename Op::In;
};
template <typename Op>
struct FirstInOf<Op, std::void_t<typename Op::In0>> {
    using type = typename Op::In0;
};

// Ops that set `static constexpr bool kNarrowVectors = true` are also instantiated for 8- and 4-byte vectors.
template <typename Op, typename = void>
struct HasNarrowVectors : std::false_type {};
template <typename Op>
struct HasNarrowVectors<Op, std::enable_if_t<Op::kNarrowVectors>> : std::true_type {};

// Op interface:
//   using In = ...; using Out = ...; static constexpr int kNumIn = n;  (optionally using In0 = ... for the first input)
//   __device__ compute_t<Out> operator()(compute_t<In> a, compute_t<In> b, compute_t<In> c, compute_t<In> d, int64_t index) const
// `index` is the C-order position in the *normalised* iteration space; only ops that ask for it
// (kNeedsIndex) get a meaningful value, and those are launched on contiguous outputs.
//
// One round of U vectors per thread.  Every load is issued before the first is used and none is conditional: units past the end
// read the last unit again and store nothing.  STREAM: inputs marked in stream_in are loaded without allocating in the caches.
// BCAST: some operand stands still along the inner axis and is read as one element per vector.
template <typename Op, int VEC, bool BCAST, int U, bool STREAM>
__device__ __forceinline__ void EwBody(const EwArgs<Op::kNumIn + 1>& args, const Op& op) {
    using In = typename Op::In;
    using In0 = typename FirstInOf<Op>::type;
    using Out = typename Op::Out;
    using CIn = compute_t<In>;
    constexpr int NIN = Op::kNumIn;
    constexpr int NOPS = NIN + 1;
    using InVec = Vec<In, VEC>;
    using In0Vec = Vec<In0, VEC>;
    using OutVec = Vec<Out, VEC>;

    const unsigned nvec = static_cast<unsigned>(args.nvec);
    const unsigned cvecs = static_cast<unsigned>(args.cvecs);
    const unsigned base = blockIdx.x * (kEwThreads * U) + threadIdx.x;
    const bool one_row = nvec == cvecs;  // no divisions

    int64_t off[U][NOPS];
    int skip[U];  // elements at the front of the vector that belong to its neighbour
    int64_t index0[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const unsigned v = min(base + u * kEwThreads, nvec - 1);
        const unsigned row = one_row ? 0 : v / cvecs;
        int64_t col = static_cast<int64_t>(v - row * cvecs) * VEC;
        skip[u] = VEC > 1 && col + VEC > args.cols ? static_cast<int>(col + VEC - args.cols) : 0;
        col -= skip[u];
        index0[u] = Op::kNeedsIndex ? args.index_base + static_cast<int64_t>(row) * args.cols + col : 0;
#pragma unroll
        for (int i = 0; i < NOPS; ++i) off[u][i] = col * args.col_stride[i];
        if (args.n_outer > 1) {
            unsigned r = row;
            for (int d = args.n_outer - 1; d >= 0; --d) {
                const unsigned q = r / static_cast<unsigned>(args.outer_shape[d]);
                const unsigned rem = r - q * static_cast<unsigned>(args.outer_shape[d]);
                r = q;
#pragma unroll
                for (int i = 0; i < NOPS; ++i) off[u][i] += static_cast<int64_t>(rem) * args.outer_stride[i][d];
            }
        } else if (!one_row) {
#pragma unroll
            for (int i = 0; i < NOPS; ++i) off[u][i] += static_cast<int64_t>(row) * args.outer_stride[i][0];
        }
    }

    raw_t<InVec> in_raw[U][NIN > 1 ? NIN : 1];
    raw_t<In0Vec> in0_raw[U];
    auto load = [&](auto tag, int i, const char* p) {
        using V = typename decltype(tag)::type;
        if (BCAST && args.col_stride[i + 1] == 0) return LoadFirst<V>(p);
        if constexpr (STREAM) {
            if ((args.stream_in >> (i + 1)) & 1) return LoadStreaming<V>(p);  // (uniform; a small operand stays cached)
            asm volatile("" ::: "memory");  // the compiler would merge the two loads into one without the hint
            const raw_t<V> r = LoadRaw<V>(p);
            asm volatile("" ::: "memory");
            return r;
        }
        return LoadRaw<V>(p);
    };
#pragma unroll
    for (int u = 0; u < U; ++u) {
        if constexpr (NIN > 0) in0_raw[u] = load(Tag<In0Vec>{}, 0, args.ptr[1] + off[u][1]);
#pragma unroll
        for (int i = 1; i < NIN; ++i) in_raw[u][i] = load(Tag<InVec>{}, i, args.ptr[i + 1] + off[u][i + 1]);
    }
    asm volatile("" ::: "memory");  // no load moves down to its use
#pragma unroll
    for (int u = 0; u < U; ++u) {
        In0Vec in0;
        InVec in[NIN > 1 ? NIN : 1];
        if constexpr (NIN > 0) in0 = __builtin_bit_cast(In0Vec, in0_raw[u]);
#pragma unroll
        for (int i = 1; i < NIN; ++i) in[i] = __builtin_bit_cast(InVec, in_raw[u][i]);
        if constexpr (BCAST) {
            if (args.col_stride[NIN > 0 ? 1 : 0] == 0) {
#pragma unroll
                for (int e = 1; e < VEC; ++e) in0.v[e] = in0.v[0];
            }
#pragma unroll
            for (int i = 1; i < NIN; ++i) {
                if (args.col_stride[i + 1] == 0) {
#pragma unroll
                    for (int e = 1; e < VEC; ++e) in[i].v[e] = in[i].v[0];
                }
            }
        }
        OutVec o;
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            CIn a = NIN > 0 ? static_cast<CIn>(in0.v[e]) : CIn{};
            CIn b = NIN > 1 ? static_cast<CIn>(in[NIN > 1 ? 1 : 0].v[e]) : CIn{};
            CIn c = NIN > 2 ? static_cast<CIn>(in[NIN > 2 ? 2 : 0].v[e]) : CIn{};
            CIn d = NIN > 3 ? static_cast<CIn>(in[NIN > 3 ? 3 : 0].v[e]) : CIn{};
            if constexpr (NIN > 4) {
                CIn f = static_cast<CIn>(in[4].v[e]);
                o.v[e] = static_cast<Out>(op.Apply5(a, b, c, d, f));
            } else {
                o.v[e] = static_cast<Out>(op(a, b, c, d, index0[u] + e));
            }
        }
        char* q = args.ptr[0] + off[u][0];
        if (base + u * kEwThreads < nvec) {
            if (VEC == 1 || skip[u] == 0) {
                *reinterpret_cast<typename RawOf<sizeof(OutVec)>::any_address*>(q) = __builtin_bit_cast(raw_t<OutVec>, o);
            } else {
#pragma unroll
                for (int e = 1; e < VEC; ++e) {
                    if (e >= skip[u]) reinterpret_cast<Out*>(q)[e] = o.v[e];
                }
            }
        }
    }
}

template <typename Op, int VEC, bool BCAST>
__global__ __launch_bounds__(kEwThreads) void EwKernel(EwArgs<Op::kNumIn + 1> args, Op op) {
    if (args.per_thread == 1) {
        EwBody<Op, VEC, BCAST, 1, false>(args, op);
    } else if (VEC > 1 && Op::kNumIn > 0 && args.stream_in) {
        EwBody<Op, VEC, BCAST, kEwUnroll, (VEC > 1 && Op::kNumIn > 0)>(args, op);
    } else {
        EwBody<Op, VEC, BCAST, kEwUnroll, false>(args, op);
    }
}

template <typename Op, int VEC>
inline void LaunchEwVec(const EwPlan& p, const Op& op, hipStream_t stream, int64_t index_base = 0) {
    constexpr int NOPS = Op::kNumIn + 1;
    int nd = p.ndim;
    int64_t cols = nd > 0 ? p.shape[nd - 1] : 1;
    int64_t rows = nd > 0 ? p.total / cols : 1;
    const int64_t cvecs = (cols + VEC - 1) / VEC;
    // a launch counts its vectors in 31 bits: larger problems are cut in two along their outermost axis (of more than one entry, which
    // it may have been cut down to); along the inner axis, so that the second part starts as well aligned as the first
    if (rows * cvecs >= (int64_t{1} << 31) - kEwThreads * kEwUnroll) {
        int d = 0;
        while (p.shape[d] == 1) ++d;  // (the product of the extents is far from 1)
        const int64_t first = d == nd - 1 ? p.shape[d] / 2 / VEC * VEC : p.shape[d] / 2;
        const int64_t per_entry = p.total / p.shape[d];
        for (int half = 0; half < 2; ++half) {
            EwPlan q = p;
            q.shape[d] = half == 0 ? first : p.shape[d] - first;
            q.total = per_entry * q.shape[d];
            if (half == 1) {
                for (int i = 0; i < p.nops; ++i) q.ptr[i] += first * p.strides[i][d];
            }
            LaunchEwVec<Op, VEC>(q, op, stream, index_base + (half == 1 ? per_entry * first : 0));
        }
        return;
    }
    EwArgs<NOPS> a;
    std::memset(&a, 0, sizeof(a));
    bool bcast = false;
    for (int i = 0; i < NOPS; ++i) {
        a.ptr[i] = p.ptr[i];
        a.col_stride[i] = nd > 0 ? p.strides[i][nd - 1] : 0;
        bcast = bcast || (i > 0 && a.col_stride[i] == 0);
    }
    a.n_outer = nd > 1 ? nd - 1 : 1;
    if (nd > 1) {
        for (int d = 0; d < nd - 1; ++d) {
            a.outer_shape[d] = p.shape[d];
            for (int i = 0; i < NOPS; ++i) a.outer_stride[i][d] = p.strides[i][d];
        }
    } else {
        a.outer_shape[0] = 1;
    }
    a.cols = cols;
    a.cvecs = cvecs;
    a.nvec = rows * cvecs;
    a.index_base = index_base;
    // an input streams when its own footprint (the axes it is not broadcast along) exceeds the threshold: a bias row added to a
    // large matrix is read once per matrix row and has to stay in the cache
    a.stream_in = 0;
    for (int i = 1; i < NOPS; ++i) {
        int64_t footprint = static_cast<int64_t>(sizeof(typename Op::In));
        for (int d = 0; d < nd; ++d) {
            if (p.strides[i][d] != 0) footprint *= p.shape[d];
        }
        bool aligned = cols % VEC == 0 && reinterpret_cast<uintptr_t>(p.ptr[i]) % 16 == 0;
        for (int d = 0; d + 1 < nd; ++d) aligned = aligned && p.strides[i][d] % 16 == 0;
        if (footprint > StreamingThresholdBytes() && aligned) a.stream_in |= 1 << i;
    }
    // one vector per thread until every compute unit has a few workgroups, then more loads in flight per thread
    a.per_thread = a.nvec <= static_cast<int64_t>(NumCUs()) * kEwThreads * 4 ? 1 : kEwUnroll;
    const int64_t per_block = static_cast<int64_t>(kEwThreads) * a.per_thread;
    dim3 grid(static_cast<unsigned>((a.nvec + per_block - 1) / per_block)), block(kEwThreads);
    if (VEC > 1 && bcast) {
        hipLaunchKernelGGL((EwKernel<Op, VEC, (VEC > 1 && Op::kNumIn > 0)>), grid, block, 0, stream, a, op);
    } else {
        hipLaunchKernelGGL((EwKernel<Op, VEC, false>), grid, block, 0, stream, a, op);
    }
    CheckLaunch("elementwise");
}

// Picks the widest vector the operands' strides allow and launches.
template <typename Op>
inline void LaunchElementwise(const EwPlan& p, const Op& op, hipStream_t stream) {
    using In = typename Op::In;
    using Out = typename Op::Out;
    constexpr int NOPS = Op::kNumIn + 1;
    if (p.total == 0) return;
    constexpr int kWidest = sizeof(In) > sizeof(Out) ? sizeof(In) : sizeof(Out);
    constexpr int kMaxVec = 16 / kWidest >= 1 ? 16 / kWidest : 1;  // 16-byte accesses on the widest operand

    int nd = p.ndim;
    int64_t cols = nd > 0 ? p.shape[nd - 1] : 1;
    bool unit = true;  // every operand that moves along the inner axis moves by one element: only then vectors can be used
    for (int i = 0; i < NOPS; ++i) {
        int64_t cs = nd > 0 ? p.strides[i][nd - 1] : 0;
        unit = unit && (cs == p.itemsize[i] || (cs == 0 && i > 0));
    }
    // Two instantiations per op keep the code object small: 16-byte vectors, or scalars.  Ops that declare kNarrowVectors (plain
    // copies: the strided copies of Im2Col, transposes and staging) also get 8- and 4-byte vectors, for rows shorter than 16 bytes.
    if (kMaxVec > 1 && unit && cols >= kMaxVec) return LaunchEwVec<Op, kMaxVec>(p, op, stream);
    if constexpr (HasNarrowVectors<Op>::value) {
        if constexpr (kMaxVec >= 4) {
            if (unit && cols >= kMaxVec / 2) return LaunchEwVec<Op, kMaxVec / 2>(p, op, stream);
        }
        if constexpr (kMaxVec >= 8) {
            if (unit && cols >= kMaxVec / 4) return LaunchEwVec<Op, kMaxVec / 4>(p, op, stream);
        }
    }
    return LaunchEwVec<Op, 1>(p, op, stream);
}

}  // namespace hipcx
