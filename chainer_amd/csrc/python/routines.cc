// chainer_amd._host: the routines a network issues per layer.  Each restates one routine of CX/routines/*.cc over the C ABI --
// promotion, broadcasting, output allocation, one kernel call per CallKernel<...> -- like the interpreted ones of
// chainer_amd/routines.py, which imports these.
#include <algorithm>
#include <vector>

#include "host.h"

namespace host {
namespace {

int BroadcastShape(const Array* a, const Array* b, int64_t* shape) {
    const int n = std::max(a->d.ndim, b->d.ndim);
    for (int i = 0; i < n; ++i) {
        const int ia = i - (n - a->d.ndim), ib = i - (n - b->d.ndim);
        const int64_t x = ia < 0 ? 1 : a->d.shape[ia], y = ib < 0 ? 1 : b->d.shape[ib];
        if (x != y && x != 1 && y != 1) {
            PyErr_Format(g.exceptions[HIPCX_DIMENSION_ERROR], "operands could not be broadcast together with shapes %R %R", a->shape, b->shape);
            throw PyError();
        }
        shape[i] = y == 1 ? x : y;
    }
    return n;
}

bool ShapeIs(const Array* a, int n, const int64_t* shape) { return a->d.ndim == n && std::equal(shape, shape + n, a->d.shape); }

Ref Broadcast(Array* a, int n, const int64_t* shape) { return ShapeIs(a, n, shape) ? NewRef(a) : BroadcastTo(a, n, shape); }

// An operand of a kernel that wants `shape` and `code`.
Ref Operand(Array* a, int n, const int64_t* shape, int code) {
    Ref b = Broadcast(a, n, shape);
    return b.arr()->d.dtype == code ? std::move(b) : Cast(b.arr(), code);
}

PyObject* const kLayoutFlag = PyUnicode_InternFromString("LAYOUT_FOLLOWS_INPUT");

// Output allocation of the element-wise routines.  ChainerX routines call Empty(shape): C-contiguous.  With LAYOUT_FOLLOWS_INPUT
// (opt-in) a dense input's axis order is kept instead, so channels-last data stays channels-last.
Ref EmptyFor(const Array* x, int n, const int64_t* shape, int code) {
    if (Flag(kLayoutFlag) && ShapeIs(x, n, shape) && std::find(x->d.strides, x->d.strides + n, 0) == x->d.strides + n) {
        int64_t st[HIPCX_MAX_NDIM];
        DenseStridesLike(x, ItemSize(code), st);
        int64_t bytes = ItemSize(code);
        for (int i = 0; i < n; ++i) bytes *= std::max<int64_t>(1, shape[i]);
        return EmptyStrided(n, shape, st, bytes, code);
    }
    return Empty(n, shape, code);
}

using BinaryFn = int (*)(const hipcx_array*, const hipcx_array*, const hipcx_array*, void*);
using ScalarFn = int (*)(const hipcx_array*, hipcx_scalar, const hipcx_array*, void*);
using UnaryFn = int (*)(const hipcx_array*, const hipcx_array*, void*);

// BroadcastBinary (CX/routines/routines_util.h:53-72): operands arrive equal-shaped, cast to out's dtype.
Ref Binary(BinaryFn fn, Array* x1, Array* x2, int code, PyObject* out_arg) {
    int64_t shape[HIPCX_MAX_NDIM];
    const int n = BroadcastShape(x1, x2, shape);
    Ref out;
    if (Given(out_arg)) {
        out = NewRef(AsArray(out_arg, "out"));
        if (!ShapeIs(out.arr(), n, shape)) {
            PyErr_Format(g.exceptions[HIPCX_DIMENSION_ERROR], "in-place operand shape %R does not match the operands", out.arr()->shape);
            throw PyError();
        }
        code = out.arr()->d.dtype;
    } else {
        out = EmptyFor(x1, n, shape, code);
    }
    Ref a = Operand(x1, n, shape, code), b = Operand(x2, n, shape, code);
    void* stream = Stream();
    Call([&] { return fn(a.d(), b.d(), out.d(), stream); });
    return out;
}

Ref BinaryScalar(ScalarFn fn, Array* x, const hipcx_scalar& s, int code, PyObject* out_arg) {
    Ref out = Given(out_arg) ? NewRef(AsArray(out_arg, "out")) : EmptyFor(x, x->d.ndim, x->d.shape, code);
    Ref a = Cast(x, out.arr()->d.dtype);
    void* stream = Stream();
    Call([&] { return fn(a.d(), s, out.d(), stream); });
    return out;
}

hipcx_scalar IntScalar(int64_t v) {
    hipcx_scalar s;
    std::memset(&s, 0, sizeof(s));
    s.kind = HIPCX_KIND_INT;
    s.i = v;
    s.f = static_cast<double>(v);
    return s;
}

Ref Unary(UnaryFn fn, Array* x) {
    const int code = MathDtype(x->d.dtype);
    Ref a = Cast(x, code);
    Ref out = EmptyLike(x, code);
    void* stream = Stream();
    Call([&] { return fn(a.d(), out.d(), stream); });
    return out;
}

// x1 op x2 where either side may be a scalar and the operation commutes.
PyObject* Commutative(BinaryFn fn, ScalarFn scalar_fn, PyObject** arg) {
    const int code = ResultType({arg[0], arg[1]});
    if (IsArray(arg[0]) && IsArray(arg[1])) {
        return Binary(fn, reinterpret_cast<Array*>(arg[0]), reinterpret_cast<Array*>(arg[1]), code, arg[2]).release();
    }
    const bool left = IsArray(arg[0]);
    return BinaryScalar(scalar_fn, AsArray(arg[left ? 0 : 1], "operand"), ToScalar(arg[left ? 1 : 0]), code, arg[2]).release();
}

HOST_FN(Add) {
    HOST_TRY;
    HOST_ARGS("add", 2, "x1", "x2", "out");
    return Commutative(hipcx_add, hipcx_add_as, arg);
    HOST_CATCH(nullptr);
}

HOST_FN(Multiply) {
    HOST_TRY;
    HOST_ARGS("multiply", 2, "x1", "x2", "out");
    return Commutative(hipcx_multiply, hipcx_multiply_as, arg);
    HOST_CATCH(nullptr);
}

// Negative = Multiply(x, Scalar{-1}) (CX/routines/arithmetic.cc).
Ref NegativeOf(Array* x) {
    if (x->d.dtype == HIPCX_BOOL) Raise(HIPCX_DTYPE_ERROR, "Cannot negate a boolean array.");
    return BinaryScalar(hipcx_multiply_as, x, IntScalar(-1), x->d.dtype, nullptr);
}

HOST_FN(Negative) {
    HOST_TRY;
    HOST_ARGS("negative", 1, "x");
    return NegativeOf(AsArray(arg[0], "x")).release();
    HOST_CATCH(nullptr);
}

HOST_FN(Subtract) {
    HOST_TRY;
    HOST_ARGS("subtract", 2, "x1", "x2", "out");
    const int code = ResultType({arg[0], arg[1]});
    if (Kind(code) == 0) Raise(HIPCX_DTYPE_ERROR, "Boolean arguments are not supported in subtract.");
    if (IsScalar(arg[1])) return BinaryScalar(hipcx_subtract_as, AsArray(arg[0], "x1"), ToScalar(arg[1]), code, arg[2]).release();
    if (IsScalar(arg[0])) {  // Subtract(Scalar, Array) = Add(-Array, Scalar) (CX/routines/arithmetic.cc)
        Ref neg = NegativeOf(AsArray(arg[1], "x2"));
        return BinaryScalar(hipcx_add_as, neg.arr(), ToScalar(arg[0]), ResultType({neg.get(), arg[0]}), nullptr).release();
    }
    return Binary(hipcx_subtract, AsArray(arg[0], "x1"), AsArray(arg[1], "x2"), code, arg[2]).release();
    HOST_CATCH(nullptr);
}

Ref DivideScalar(const hipcx_scalar& s, Array* x, int code, PyObject* out_arg) {
    Ref out = Given(out_arg) ? NewRef(AsArray(out_arg, "out")) : EmptyLike(x, code);
    Ref a = Cast(x, out.arr()->d.dtype);
    void* stream = Stream();
    Call([&] { return hipcx_divide_sa(s, a.d(), out.d(), stream); });
    return out;
}

// TrueDivide: integer operands are computed in float32 (CX/routines/arithmetic.cc Divide).
HOST_FN(Divide) {
    HOST_TRY;
    HOST_ARGS("divide", 2, "x1", "x2", "out");
    const int code = MathDtype(ResultType({arg[0], arg[1]}));
    if (IsScalar(arg[1])) return BinaryScalar(hipcx_divide_as, AsArray(arg[0], "x1"), ToScalar(arg[1]), code, arg[2]).release();
    if (IsScalar(arg[0])) return DivideScalar(ToScalar(arg[0]), AsArray(arg[1], "x2"), code, arg[2]).release();
    return Binary(hipcx_divide, AsArray(arg[0], "x1"), AsArray(arg[1], "x2"), code, arg[2]).release();
    HOST_CATCH(nullptr);
}

// Reciprocal(x) = Scalar{1} / x (CX/routines/arithmetic.cc).
HOST_FN(Reciprocal) {
    HOST_TRY;
    HOST_ARGS("reciprocal", 1, "x");
    Array* x = AsArray(arg[0], "x");
    return DivideScalar(IntScalar(1), x, MathDtype(x->d.dtype), nullptr).release();
    HOST_CATCH(nullptr);
}

#define UNARY_ROUTINE(Name, name)                               \
    HOST_FN(Name) {                                             \
        HOST_TRY;                                               \
        HOST_ARGS(#name, 1, "x");                               \
        return Unary(hipcx_##name, AsArray(arg[0], "x")).release(); \
        HOST_CATCH(nullptr);                                    \
    }
UNARY_ROUTINE(Exp, exp)
UNARY_ROUTINE(Log, log)
UNARY_ROUTINE(Tanh, tanh)
UNARY_ROUTINE(Sqrt, sqrt)

// Sigmoid(x) = Reciprocal(1 + Exp(-x)) (CX/routines/activation.cc:74-78), its four steps in one kernel.
HOST_FN(Sigmoid) {
    HOST_TRY;
    HOST_ARGS("sigmoid", 1, "x");
    auto fn = [](const hipcx_array* x, const hipcx_array* out, void* stream) { return hipcx_unary(HIPCX_UNARY_SIGMOID, x, out, stream); };
    return Unary(fn, AsArray(arg[0], "x")).release();
    HOST_CATCH(nullptr);
}

using SelectFn = int (*)(const hipcx_array*, hipcx_scalar, hipcx_scalar, const hipcx_array*, const hipcx_array*, void*);

// x1 < / > x2 ? pos : neg with scalar x2 and pos (CX/routines/misc.cc:34-58).
Ref Select(SelectFn fn, Array* x1, const hipcx_scalar& x2, const hipcx_scalar& pos, Array* neg, int code, bool follow_layout) {
    Ref out = follow_layout ? EmptyFor(x1, x1->d.ndim, x1->d.shape, code) : EmptyLike(x1, code);
    Ref a = Cast(x1, code), b = Cast(neg, code);
    void* stream = Stream();
    Call([&] { return fn(a.d(), x2, pos, b.d(), out.d(), stream); });
    return out;
}

HOST_FN(IfLessElse) {
    HOST_TRY;
    HOST_ARGS("if_less_else", 4, "x1", "x2", "pos", "neg");
    return Select(hipcx_if_less_else_assa, AsArray(arg[0], "x1"), ToScalar(arg[1]), ToScalar(arg[2]), AsArray(arg[3], "neg"),
                  ResultType({arg[2], arg[3]}), true)
            .release();
    HOST_CATCH(nullptr);
}

// IfLessElse(x, 0, 0, Add(g1, g2)) of float arrays of one shape and dtype in one kernel, or None.
HOST_FN(AddReluGrad) {
    HOST_TRY;
    HOST_ARGS("add_relu_grad", 3, "x", "g1", "g2");
    Array *x = AsArray(arg[0], "x"), *g1 = AsArray(arg[1], "g1"), *g2 = AsArray(arg[2], "g2");
    for (const Array* g : {g1, g2}) {
        if (!IsFloat(x->d.dtype) || g->d.dtype != x->d.dtype || !ShapeIs(g, x->d.ndim, x->d.shape)) Py_RETURN_NONE;
    }
    Ref out = EmptyLike(x, x->d.dtype);
    void* stream = Stream();
    Call([&] { return hipcx_add_relu_grad(&x->d, &g1->d, &g2->d, out.d(), stream); });
    return out.release();
    HOST_CATCH(nullptr);
}

HOST_FN(IfGreaterElse) {
    HOST_TRY;
    HOST_ARGS("if_greater_else", 4, "x1", "x2", "pos", "neg");
    return Select(hipcx_if_greater_else_assa, AsArray(arg[0], "x1"), ToScalar(arg[1]), ToScalar(arg[2]), AsArray(arg[3], "neg"),
                  ResultType({arg[2], arg[3]}), false)
            .release();
    HOST_CATCH(nullptr);
}

// Maximum(array, scalar) = IfLessElse(x1, x2, x2, x1) (CX/routines/misc.cc:210-216); array, array: x1 > x2 ? x1 : x2.
HOST_FN(Maximum) {
    HOST_TRY;
    HOST_ARGS("maximum", 2, "x1", "x2");
    if (IsScalar(arg[0])) std::swap(arg[0], arg[1]);
    const int code = ResultType({arg[0], arg[1]});
    Array* x1 = AsArray(arg[0], "x1");
    if (IsScalar(arg[1])) {
        hipcx_scalar s = ToScalar(arg[1]);
        return Select(hipcx_if_less_else_assa, x1, s, s, x1, code, true).release();
    }
    Array* x2 = AsArray(arg[1], "x2");
    int64_t shape[HIPCX_MAX_NDIM];
    const int n = BroadcastShape(x1, x2, shape);
    Ref a = Operand(x1, n, shape, code), b = Operand(x2, n, shape, code);
    Ref out = Empty(n, shape, code);
    void* stream = Stream();
    Call([&] { return hipcx_if_greater_else_aaaa(a.d(), b.d(), a.d(), b.d(), out.d(), stream); });
    return out.release();
    HOST_CATCH(nullptr);
}

// Relu(x) = Maximum(0, x) in the math dtype of x (CX/routines/activation.cc:80-84).
HOST_FN(Relu) {
    HOST_TRY;
    HOST_ARGS("relu", 1, "x");
    Array* x = AsArray(arg[0], "x");
    const int code = MathDtype(x->d.dtype);
    Ref xc = Cast(x, code);
    const hipcx_scalar zero = IntScalar(0);
    return Select(hipcx_if_less_else_assa, xc.arr(), zero, zero, xc.arr(), code, true).release();
    HOST_CATCH(nullptr);
}

PyObject* Compare(BinaryFn fn, PyObject* p1, PyObject* p2) {
    Array* x1 = AsArray(p1, "x1");
    Ref scalar;
    if (IsScalar(p2)) {
        scalar = Empty(0, nullptr, x1->d.dtype);
        hipcx_scalar s = ToScalar(p2);
        void* stream = Stream();
        Call([&] { return hipcx_fill(scalar.d(), s, stream); });
        p2 = scalar.get();
    }
    Array* x2 = AsArray(p2, "x2");
    if ((x1->d.dtype == HIPCX_BOOL) != (x2->d.dtype == HIPCX_BOOL)) {
        Raise(HIPCX_DTYPE_ERROR, "Comparison of bool and non-bool dtypes is not supported.");
    }
    const int code = Promote(x1->d.dtype, x2->d.dtype);
    int64_t shape[HIPCX_MAX_NDIM];
    const int n = BroadcastShape(x1, x2, shape);
    Ref a = Operand(x1, n, shape, code), b = Operand(x2, n, shape, code);
    Ref out = Empty(n, shape, HIPCX_BOOL);
    void* stream = Stream();
    Call([&] { return fn(a.d(), b.d(), out.d(), stream); });
    return out.release();
}

#define COMPARE_ROUTINE(Name, name)                 \
    HOST_FN(Name) {                                 \
        HOST_TRY;                                   \
        HOST_ARGS(#name, 2, "x1", "x2");            \
        return Compare(hipcx_##name, arg[0], arg[1]); \
        HOST_CATCH(nullptr);                        \
    }
COMPARE_ROUTINE(Equal, equal)
COMPARE_ROUTINE(NotEqual, not_equal)
COMPARE_ROUTINE(Greater, greater)
COMPARE_ROUTINE(GreaterEqual, greater_equal)

HOST_FN(Full) {
    HOST_TRY;
    HOST_ARGS("full", 2, "shape", "value", "dtype");
    int64_t shape[HIPCX_MAX_NDIM];
    const int n = ToShape(arg[0], shape);
    const int code = Given(arg[2]) ? DtypeCode(arg[2]) : ScalarDtype(arg[1]);
    Ref out = Empty(n, shape, code);
    hipcx_scalar s = ToScalar(arg[1]);
    void* stream = Stream();
    Call([&] { return hipcx_fill(out.d(), s, stream); });
    return out.release();
    HOST_CATCH(nullptr);
}

// ---------------------------------------------------------------------------------------------
// manipulation
// ---------------------------------------------------------------------------------------------
std::vector<Ref> Sequence(PyObject* arrays) {
    Ref seq(PySequence_List(arrays));
    if (!seq) throw PyError();
    std::vector<Ref> v;
    v.reserve(PyList_GET_SIZE(seq.get()));
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(seq.get()); ++i) v.push_back(NewRef(AsArray(PyList_GET_ITEM(seq.get(), i), "array")));
    return v;
}

// Split into views (CX/routines/manipulation.cc Split).
HOST_FN(Split) {
    HOST_TRY;
    HOST_ARGS("split", 2, "a", "indices_or_sections", "axis");
    Array* a = AsArray(arg[0], "a");
    const int axis = NormalizeAxis(arg[2] != nullptr ? ToInt(arg[2]) : 0, a->d.ndim);
    const int64_t dim = a->d.shape[axis];
    std::vector<std::pair<int64_t, int64_t>> bounds;
    if (PyIndex_Check(arg[1])) {
        const int64_t n = ToInt(arg[1]);
        if (n <= 0 || dim % n != 0) Raise(HIPCX_DIMENSION_ERROR, "array split does not result in an equal division");
        for (int64_t i = 0; i < n; ++i) bounds.emplace_back(i * (dim / n), (i + 1) * (dim / n));
    } else {
        Ref seq(PySequence_Fast(arg[1], "sections must be an int or a sequence of ints"));
        if (!seq) throw PyError();
        int64_t start = 0;
        for (Py_ssize_t i = 0; i <= PySequence_Fast_GET_SIZE(seq.get()); ++i) {
            int64_t stop = dim;
            if (i < PySequence_Fast_GET_SIZE(seq.get())) {
                stop = std::min(std::max<int64_t>(ToInt(PySequence_Fast_GET_ITEM(seq.get(), i)), 0), dim);
            }
            bounds.emplace_back(start, std::max(start, stop));
            start = stop;
        }
    }
    Ref list(PyList_New(static_cast<Py_ssize_t>(bounds.size())));
    if (!list) throw PyError();
    int64_t shape[HIPCX_MAX_NDIM];
    std::copy(a->d.shape, a->d.shape + a->d.ndim, shape);
    for (size_t i = 0; i < bounds.size(); ++i) {
        shape[axis] = bounds[i].second - bounds[i].first;
        const int64_t offset = shape[axis] > 0 ? bounds[i].first * a->d.strides[axis] : 0;
        PyList_SET_ITEM(list.get(), static_cast<Py_ssize_t>(i), View(a, offset, a->d.ndim, shape, a->d.strides).release());
    }
    return list.release();
    HOST_CATCH(nullptr);
}

// Every input into its view of the result.
void CopyInto(const std::vector<Ref>& arrays, const std::vector<hipcx_array>& views) {
    void* stream = Stream();
    std::vector<const hipcx_array*> from, to;
    for (size_t i = 0; i < views.size(); ++i) {
        from.push_back(&arrays[i].arr()->d);
        to.push_back(&views[i]);
    }
    Call([&] { return hipcx_copy_many(from.data(), to.data(), static_cast<int>(from.size()), stream); });
}

// Concatenate = Empty + a copy of every input (CopyKernel, CX/routines/manipulation.cc:415-460).
HOST_FN(Concatenate) {
    HOST_TRY;
    HOST_ARGS("concatenate", 1, "arrays", "axis");
    std::vector<Ref> arrays = Sequence(arg[0]);
    if (arrays.empty()) Raise(HIPCX_DIMENSION_ERROR, "Need at least one array to concatenate");
    Array* first = arrays[0].arr();
    const int axis = NormalizeAxis(arg[1] != nullptr ? ToInt(arg[1]) : 0, first->d.ndim);
    int64_t shape[HIPCX_MAX_NDIM];
    const int n = first->d.ndim;
    std::copy(first->d.shape, first->d.shape + n, shape);
    shape[axis] = 0;
    int code = first->d.dtype;
    for (const Ref& r : arrays) {
        const Array* a = r.arr();
        if (a->d.ndim != n) Raise(HIPCX_DIMENSION_ERROR, "all the input arrays must have same number of dimensions");
        for (int i = 0; i < n; ++i) {
            if (i != axis && a->d.shape[i] != shape[i]) {
                Raise(HIPCX_DIMENSION_ERROR, "all the input array dimensions except for the concatenation axis must match exactly");
            }
        }
        shape[axis] += a->d.shape[axis];
        code = Promote(code, a->d.dtype);
    }
    Ref out = Empty(n, shape, code);
    hipcx_array view = out.arr()->d;
    std::vector<hipcx_array> views;
    for (const Ref& r : arrays) {
        view.shape[axis] = r.arr()->d.shape[axis];
        views.push_back(view);
        view.data = static_cast<char*>(view.data) + view.shape[axis] * view.strides[axis];
    }
    CopyInto(arrays, views);
    return out.release();
    HOST_CATCH(nullptr);
}

// Stack = Empty + a copy of every input into a view of the new axis (CX/routines/manipulation.cc Stack).
HOST_FN(Stack) {
    HOST_TRY;
    HOST_ARGS("stack", 1, "arrays", "axis");
    std::vector<Ref> arrays = Sequence(arg[0]);
    if (arrays.empty()) Raise(HIPCX_DIMENSION_ERROR, "Need at least one array to stack");
    Array* first = arrays[0].arr();
    const int n = first->d.ndim;
    if (n + 1 > HIPCX_MAX_NDIM) Raise(HIPCX_DIMENSION_ERROR, "ndim %d exceeds the maximum of %d", n + 1, HIPCX_MAX_NDIM);
    const int axis = NormalizeAxis(arg[1] != nullptr ? ToInt(arg[1]) : 0, n + 1);
    int code = first->d.dtype;
    for (const Ref& r : arrays) {
        if (!ShapeIs(r.arr(), n, first->d.shape)) Raise(HIPCX_DIMENSION_ERROR, "All arrays need to have the same shape");
        code = Promote(code, r.arr()->d.dtype);
    }
    int64_t shape[HIPCX_MAX_NDIM];
    for (int i = 0; i <= n; ++i) shape[i] = i == axis ? static_cast<int64_t>(arrays.size()) : first->d.shape[i < axis ? i : i - 1];
    Ref out = Empty(n + 1, shape, code);
    hipcx_array view = out.arr()->d;
    view.ndim = n;
    const int64_t step = view.strides[axis];
    for (int i = axis; i < n; ++i) view.shape[i] = view.shape[i + 1], view.strides[i] = view.strides[i + 1];
    std::vector<hipcx_array> views;
    for (size_t i = 0; i < arrays.size(); ++i) {
        views.push_back(view);
        view.data = static_cast<char*>(view.data) + step;
    }
    CopyInto(arrays, views);
    return out.release();
    HOST_CATCH(nullptr);
}

// ---------------------------------------------------------------------------------------------
// reductions
// ---------------------------------------------------------------------------------------------
int SortedAxes(PyObject* axis, int ndim, int8_t* axes) {
    if (!Given(axis)) {
        for (int i = 0; i < ndim; ++i) axes[i] = static_cast<int8_t>(i);
        return ndim;
    }
    int64_t given[HIPCX_MAX_NDIM];
    const int n = ToShape(axis, given);
    unsigned seen = 0;
    for (int i = 0; i < n; ++i) {
        const int ax = NormalizeAxis(given[i], ndim);
        if (seen >> ax & 1) Raise(HIPCX_DIMENSION_ERROR, "Duplicate axis values.");
        seen |= 1u << ax;
    }
    int m = 0;
    for (int i = 0; i < ndim; ++i) {
        if (seen >> i & 1) axes[m++] = static_cast<int8_t>(i);
    }
    return m;
}

// EmptyReduced (CX/routines/creation.cc:56-75): kept axes get stride 0.
Ref ReducedOut(const Array* a, const int8_t* axes, int n_axes, bool keepdims, int code) {
    unsigned reduced = 0;
    for (int i = 0; i < n_axes; ++i) reduced |= 1u << axes[i];
    int64_t inner[HIPCX_MAX_NDIM], inner_strides[HIPCX_MAX_NDIM];
    int n = 0;
    for (int i = 0; i < a->d.ndim; ++i) {
        if (!(reduced >> i & 1)) inner[n++] = a->d.shape[i];
    }
    if (!keepdims) return Empty(n, inner, code);
    ContiguousStrides(n, inner, ItemSize(code), inner_strides);
    int64_t shape[HIPCX_MAX_NDIM], strides[HIPCX_MAX_NDIM];
    int k = 0;
    for (int i = 0; i < a->d.ndim; ++i) {
        const bool r = reduced >> i & 1;
        shape[i] = r ? 1 : inner[k];
        strides[i] = r ? 0 : inner_strides[k];
        k += r ? 0 : 1;
    }
    return EmptyStrided(a->d.ndim, shape, strides, Product(n, inner) * ItemSize(code), code);
}

using ReduceFn = int (*)(const hipcx_array*, const int8_t*, int, const hipcx_array*, void*, size_t, void*);

void Reduce(ReduceFn fn, const Array* a, const int8_t* axes, int n, const Array* out) {
    Workspace ws(hipcx_reduce_workspace_size(&a->d, axes, n, &out->d));
    void* stream = Stream();
    Call([&] { return fn(&a->d, axes, n, &out->d, ws.ptr, ws.bytes, stream); });
}

bool Truth(PyObject* x) {
    if (x == nullptr) return false;
    int v = PyObject_IsTrue(x);
    if (v < 0) throw PyError();
    return v != 0;
}

// Sum (CX/routines/reduction.cc:28-76): bool / int inputs accumulate and return int64.
HOST_FN(Sum) {
    HOST_TRY;
    HOST_ARGS("sum", 1, "a", "axis", "keepdims");
    Array* a = AsArray(arg[0], "a");
    int8_t axes[HIPCX_MAX_NDIM];
    const int n = SortedAxes(arg[1], a->d.ndim, axes);
    Ref out = ReducedOut(a, axes, n, Truth(arg[2]), IsFloat(a->d.dtype) ? a->d.dtype : HIPCX_INT64);
    Reduce(hipcx_sum, a, axes, n, out.arr());
    return out.release();
    HOST_CATCH(nullptr);
}

PyObject* Extreme(ReduceFn fn, PyObject** arg, bool arg_result, const char* empty_message) {
    Array* a = AsArray(arg[0], "a");
    int8_t axes[HIPCX_MAX_NDIM];
    const int n = SortedAxes(arg[1], a->d.ndim, axes);
    for (int i = 0; i < n; ++i) {
        if (a->d.shape[axes[i]] == 0) Raise(HIPCX_DIMENSION_ERROR, "%s", empty_message);
    }
    Ref out = ReducedOut(a, axes, n, !arg_result && Truth(arg[2]), arg_result ? HIPCX_INT64 : a->d.dtype);
    Reduce(fn, a, axes, n, out.arr());
    return out.release();
}

HOST_FN(AMax) {  // CX/routines/statistics.cc:21-65
    HOST_TRY;
    HOST_ARGS("amax", 1, "a", "axis", "keepdims");
    return Extreme(hipcx_amax, arg, false, "cannot compute the maximum along zero-sized axis");
    HOST_CATCH(nullptr);
}
HOST_FN(AMin) {  // CX/routines/statistics.cc:66-79
    HOST_TRY;
    HOST_ARGS("amin", 1, "a", "axis", "keepdims");
    return Extreme(hipcx_amin, arg, false, "cannot compute the minimum along zero-sized axis");
    HOST_CATCH(nullptr);
}
HOST_FN(ArgMax) {  // CX/routines/sorting.cc:21-52: int64 result, no keepdims
    HOST_TRY;
    HOST_ARGS("argmax", 1, "a", "axis");
    return Extreme(hipcx_argmax, arg, true, "cannot compute ArgMax for an empty array");
    HOST_CATCH(nullptr);
}
HOST_FN(ArgMin) {  // CX/routines/sorting.cc:54-85
    HOST_TRY;
    HOST_ARGS("argmin", 1, "a", "axis");
    return Extreme(hipcx_argmin, arg, true, "cannot compute ArgMin for an empty array");
    HOST_CATCH(nullptr);
}

// ---------------------------------------------------------------------------------------------
// linear algebra / connection
// ---------------------------------------------------------------------------------------------
Ref Zeros(int n, const int64_t* shape, int code) {
    Ref out = Empty(n, shape, code);
    void* stream = Stream();
    Call([&] { return hipcx_fill(out.d(), IntScalar(0), stream); });
    return out;
}

void DotInto(const hipcx_array* a, const hipcx_array* b, const hipcx_array* out) {
    Workspace ws(hipcx_dot_workspace_size(a, b, out));
    void* stream = Stream();
    Call([&] { return hipcx_dot(a, b, out, ws.ptr, ws.bytes, stream); });
}

// Dot for 2-D operands (CX/routines/linalg.cc:27-100): k == 0 gives zeros without a kernel.
HOST_FN(Dot) {
    HOST_TRY;
    HOST_ARGS("dot", 2, "a", "b", "out_dtype");
    Array *a = AsArray(arg[0], "a"), *b = AsArray(arg[1], "b");
    if (a->d.ndim != 2 || b->d.ndim != 2) Raise(HIPCX_DIMENSION_ERROR, "ChainerX dot supports only 2-dimensional arrays.");
    if (a->d.shape[1] != b->d.shape[0]) Raise(HIPCX_DIMENSION_ERROR, "Axis dimension mismatch");
    const int code = Given(arg[2]) ? DtypeCode(arg[2]) : Promote(a->d.dtype, b->d.dtype);
    const int64_t shape[2] = {a->d.shape[0], b->d.shape[1]};
    if (a->d.shape[1] == 0) return Zeros(2, shape, code).release();
    Ref out = Empty(2, shape, code);
    Ref ac = Cast(a, code), bc = Cast(b, code);
    DotInto(ac.d(), bc.d(), out.d());
    return out.release();
    HOST_CATCH(nullptr);
}

// Linear (CX/routines/connection.cc:322-394): DotKernel(x, w.T view), AddKernel with a stride-0 bias in its epilogue.
HOST_FN(Linear) {
    HOST_TRY;
    HOST_ARGS("linear", 2, "x", "w", "b", "n_batch_axes");
    Array *x = AsArray(arg[0], "x"), *w = AsArray(arg[1], "w"), *b = Given(arg[2]) ? AsArray(arg[2], "b") : nullptr;
    if (w->d.ndim != 2) Raise(HIPCX_DIMENSION_ERROR, "w.ndim should be 2");
    if (b != nullptr && b->d.ndim != 1) Raise(HIPCX_DIMENSION_ERROR, "b.ndim should be 1");
    const int n_batch = x->d.ndim > 0 ? NormalizeAxis(arg[3] != nullptr ? ToInt(arg[3]) : 1, x->d.ndim) : 0;
    int code = Promote(x->d.dtype, w->d.dtype);
    if (b != nullptr) code = Promote(code, b->d.dtype);
    const int64_t rows = Product(n_batch, x->d.shape), m = w->d.shape[0], k = w->d.shape[1];
    int64_t out_shape[HIPCX_MAX_NDIM];
    std::copy(x->d.shape, x->d.shape + n_batch, out_shape);
    out_shape[n_batch] = m;
    if (m == 0 || k == 0) {
        if (b != nullptr) {
            Ref bc = Cast(b, code);
            return BroadcastTo(bc.arr(), n_batch + 1, out_shape).release();
        }
        return Zeros(n_batch + 1, out_shape, code).release();
    }
    const int64_t x_shape[2] = {rows, k}, matrix_shape[2] = {rows, m};
    Ref xm = Reshape(x, 2, x_shape);
    xm = Cast(xm.arr(), code);
    Ref wc = Cast(w, code);
    hipcx_array wt = wc.arr()->d;
    std::swap(wt.shape[0], wt.shape[1]);
    std::swap(wt.strides[0], wt.strides[1]);
    Ref out = Empty(2, matrix_shape, code);
    if (b == nullptr) {
        DotInto(xm.d(), &wt, out.d());
    } else {
        Ref bc = Cast(b, code);
        if (bc.arr()->d.shape[0] != m) {  // a bias of one element is broadcast; other lengths raise
            const int64_t bias_shape[1] = {m};
            bc = BroadcastTo(bc.arr(), 1, bias_shape);
        }
        Workspace ws(hipcx_dot_workspace_size(xm.d(), &wt, out.d()));
        void* stream = Stream();
        Call([&] { return hipcx_dot_bias(xm.d(), &wt, bc.d(), out.d(), ws.ptr, ws.bytes, stream); });
    }
    return Reshape(out.arr(), n_batch + 1, out_shape).release();
    HOST_CATCH(nullptr);
}

// An int, or a sequence of n ints.
void Pair(PyObject* v, int n, int64_t fallback, int64_t* out) {
    if (v == nullptr) {
        std::fill(out, out + n, fallback);
        return;
    }
    if (PyIndex_Check(v)) {
        std::fill(out, out + n, ToInt(v));
        return;
    }
    if (ToShape(v, out) != n) {
        PyErr_Format(g.exceptions[HIPCX_DIMENSION_ERROR], "expected %d values, got %R", n, v);
        throw PyError();
    }
}

int64_t OutDim(int64_t in_dim, int64_t kernel, int64_t stride, int64_t pad, bool cover_all) {
    const int64_t n = hipcx_conv_out_dim(in_dim, kernel, stride, pad, cover_all ? 1 : 0);
    if (n < 0) Raise(HIPCX_DIMENSION_ERROR, "Output size should be positive.");
    return n;
}

bool IsChannelsLast(const Array* x) {
    return x->d.ndim == 4 && x->d.strides[1] == ItemSize(x->d.dtype) && x->d.shape[1] > 1 && x->d.shape[2] * x->d.shape[3] > 1;
}

// Output of the kernels that allocate their own result (Conv, MaxPool, AveragePool).  C-contiguous NCHW, like the CUDA backend's
// (CX/cuda/cuda_conv.cc:311); channels-last (the native backend's layout of a conv result) when the opt-in LAYOUT_FOLLOWS_INPUT
// mode is on and the input already is.
Ref SpatialOut(const Array* x, int64_t channels, const int64_t* dims, int code) {
    const int nd = x->d.ndim;
    int64_t shape[HIPCX_MAX_NDIM];
    shape[0] = x->d.shape[0];
    shape[1] = channels;
    std::copy(dims, dims + nd - 2, shape + 2);
    if (nd == 4 && Flag(kLayoutFlag) && (IsChannelsLast(x) || x->d.shape[1] < 8)) {
        const int64_t it = ItemSize(code), h = shape[2], w = shape[3];
        const int64_t strides[4] = {h * w * channels * it, it, w * channels * it, channels * it};
        return EmptyStrided(4, shape, strides, Product(4, shape) * it, code);
    }
    return Empty(nd, shape, code);
}

struct ConvArgs {
    Array *x, *w, *b;
    int n;
    int64_t stride[HIPCX_MAX_NDIM], pad[HIPCX_MAX_NDIM], dims[HIPCX_MAX_NDIM];
    bool cover_all;
};

void PrepareConv(ConvArgs* c, PyObject* stride, PyObject* pad, PyObject* cover_all) {
    c->n = c->x->d.ndim - 2;
    Pair(stride, c->n, 1, c->stride);
    Pair(pad, c->n, 0, c->pad);
    c->cover_all = Truth(cover_all);
    if (c->w->d.shape[1] != c->x->d.shape[1]) {
        PyErr_Format(g.exceptions[HIPCX_DIMENSION_ERROR], "Mismatched number of input channels in input %R and weights %R.", c->x->shape, c->w->shape);
        throw PyError();
    }
    if (c->b != nullptr && (c->b->d.ndim != 1 || c->b->d.shape[0] != c->w->d.shape[0])) {
        PyErr_Format(g.exceptions[HIPCX_DIMENSION_ERROR], "Mismatched bias shape %R for weights %R.", c->b->shape, c->w->shape);
        throw PyError();
    }
    for (int i = 0; i < c->n; ++i) c->dims[i] = OutDim(c->x->d.shape[2 + i], c->w->d.shape[2 + i], c->stride[i], c->pad[i], c->cover_all);
}

// Conv (CX/routines/connection.cc:140-208): one ConvKernel call with the bias inside.  Any number of spatial axes; the dedicated
// kernels are the 2-D ones (0 and 1 axes run through them as extents of one, 3 and more through a plain kernel).
HOST_FN(Conv) {
    HOST_TRY;
    HOST_ARGS("conv", 2, "x", "w", "b", "stride", "pad", "cover_all", "out_dtype");
    ConvArgs c;
    c.x = AsArray(arg[0], "x");
    c.w = AsArray(arg[1], "w");
    c.b = Given(arg[2]) ? AsArray(arg[2], "b") : nullptr;
    if (c.x->d.ndim < 2 || c.w->d.ndim != c.x->d.ndim) {
        PyErr_Format(g.exceptions[HIPCX_DIMENSION_ERROR], "Mismatched number of dimensions in input %R and weights %R.", c.x->shape, c.w->shape);
        throw PyError();
    }
    PrepareConv(&c, arg[3], arg[4], arg[5]);
    const int code = Given(arg[6]) ? DtypeCode(arg[6]) : ResultType({arg[0], arg[1], reinterpret_cast<PyObject*>(c.b)});
    Ref out = SpatialOut(c.x, c.w->d.shape[0], c.dims, code);
    Ref x = Cast(c.x, code), w = Cast(c.w, code), b;
    if (c.b != nullptr) b = Cast(c.b, code);
    Workspace ws(hipcx_conv_workspace_size(x.d(), w.d(), out.d()));
    void* stream = Stream();
    Call([&] { return hipcx_conv(x.d(), w.d(), b.d(), c.stride, c.pad, c.cover_all ? 1 : 0, out.d(), ws.ptr, ws.bytes, stream); });
    return out.release();
    HOST_CATCH(nullptr);
}

// Opt-in fused block: relu(fixed_batch_norm(conv(x, w, b), *bn, eps, axis=(0, 2, 3)) + residual) in one kernel call.
HOST_FN(ConvBnAct) {
    HOST_TRY;
    HOST_ARGS("conv_bn_act", 2, "x", "w", "b", "stride", "pad", "cover_all", "bn", "eps", "residual", "relu");
    ConvArgs c;
    c.x = AsArray(arg[0], "x");
    c.w = AsArray(arg[1], "w");
    c.b = nullptr;
    if (c.x->d.ndim != 4 || c.w->d.ndim != 4) Raise(HIPCX_NOT_IMPLEMENTED_ERROR, "only 2-D convolution is on the supported path");
    PrepareConv(&c, arg[3], arg[4], arg[5]);
    const int code = Promote(c.x->d.dtype, c.w->d.dtype);
    Ref out = SpatialOut(c.x, c.w->d.shape[0], c.dims, code);
    Ref x = Cast(c.x, code), w = Cast(c.w, code), b, residual, bn[4];
    if (Given(arg[2])) b = Cast(AsArray(arg[2], "b"), code);
    if (Given(arg[6])) {
        std::vector<Ref> params = Sequence(arg[6]);
        if (params.size() != 4) Raise(HIPCX_DIMENSION_ERROR, "bn is (gamma, beta, mean, var)");
        for (int i = 0; i < 4; ++i) bn[i] = Cast(params[i].arr(), code);
    }
    if (Given(arg[8])) residual = Cast(AsArray(arg[8], "residual"), code);
    hipcx_scalar eps;
    std::memset(&eps, 0, sizeof(eps));
    eps.kind = HIPCX_KIND_FLOAT;
    eps.f = arg[7] != nullptr ? PyFloat_AsDouble(arg[7]) : 2e-5;
    if (PyErr_Occurred()) throw PyError();
    const bool relu = Truth(arg[9]);
    Workspace ws(hipcx_conv_workspace_size(x.d(), w.d(), out.d()));
    void* stream = Stream();
    Call([&] {
        return hipcx_conv_bn_act(x.d(), w.d(), b.d(), c.stride, c.pad, c.cover_all ? 1 : 0, bn[0].d(), bn[1].d(), bn[2].d(), bn[3].d(), eps,
                                 residual.d(), relu ? 1 : 0, out.d(), ws.ptr, ws.bytes, stream);
    });
    return out.release();
    HOST_CATCH(nullptr);
}

hipcx_scalar FloatScalar(PyObject* x, double fallback) {
    hipcx_scalar s;
    std::memset(&s, 0, sizeof(s));
    s.kind = HIPCX_KIND_FLOAT;
    s.f = x != nullptr ? PyFloat_AsDouble(x) : fallback;
    if (PyErr_Occurred()) throw PyError();
    return s;
}

// The array seen with another shape: a descriptor when the strides allow it, else a copy held by `keep`.
hipcx_array Reshaped(Array* a, int n, const int64_t* shape, Ref* keep) {
    hipcx_array d = a->d;
    d.ndim = n;
    std::copy(shape, shape + n, d.shape);
    if (!NoCopyReshape(a->d, n, shape, d.strides)) {
        *keep = CopyOf(a, a->d.dtype);
        d.data = keep->arr()->d.data;
        ContiguousStrides(n, shape, ItemSize(a->d.dtype), d.strides);
    }
    return d;
}

// FixedBatchNorm (CX/routines/normalization.cc:414-424 with PreprocessBatchNorm :61-101).
HOST_FN(FixedBatchNorm) {
    HOST_TRY;
    HOST_ARGS("fixed_batch_norm", 5, "x", "gamma", "beta", "mean", "var", "eps", "axis");
    Array* x = AsArray(arg[0], "x");
    for (int i = 0; i < 5; ++i) {
        if (!IsFloat(AsArray(arg[i], "argument")->d.dtype)) Raise(HIPCX_DTYPE_ERROR, "BatchNorm only supports floating kind inputs.");
    }
    int8_t axes[HIPCX_MAX_NDIM] = {0};
    const int n_axes = Given(arg[6]) ? SortedAxes(arg[6], x->d.ndim, axes) : 1;
    int64_t reduced[HIPCX_MAX_NDIM];
    std::copy(x->d.shape, x->d.shape + x->d.ndim, reduced);
    for (int i = 0; i < n_axes; ++i) reduced[axes[i]] = 1;
    const int64_t size = Product(x->d.ndim, reduced);
    static const char* const names[] = {"Gamma", "Beta", "Mean", "Variance"};
    hipcx_array params[4];
    Ref keep[4];
    for (int i = 0; i < 4; ++i) {
        Array* a = reinterpret_cast<Array*>(arg[1 + i]);
        if (Size(a) != size) {
            Raise(HIPCX_DIMENSION_ERROR, "%s must have the same size as the reduced input. Actual: %lld. Expected: %lld.", names[i],
                  static_cast<long long>(Size(a)), static_cast<long long>(size));
        }
        params[i] = Reshaped(a, x->d.ndim, reduced, &keep[i]);
    }
    const hipcx_scalar eps = FloatScalar(arg[5], 2e-5);
    int64_t strides[HIPCX_MAX_NDIM];
    const int it = ItemSize(x->d.dtype);
    DenseStridesLike(x, it, strides);
    Ref out = EmptyStrided(x->d.ndim, x->d.shape, strides, Size(x) * it, x->d.dtype);
    void* stream = Stream();
    Call([&] { return hipcx_fixed_batch_norm(&x->d, &params[0], &params[1], &params[2], &params[3], eps, axes, n_axes, out.d(), stream); });
    return out.release();
    HOST_CATCH(nullptr);
}

// ---------------------------------------------------------------------------------------------
// pooling
// ---------------------------------------------------------------------------------------------
struct PoolArgs {
    int n;
    int64_t ksize[HIPCX_MAX_NDIM], stride[HIPCX_MAX_NDIM], pad[HIPCX_MAX_NDIM], dims[HIPCX_MAX_NDIM];
};

void PreparePool(PoolArgs* p, const Array* x, PyObject* ksize, PyObject* stride, PyObject* pad, bool cover_all) {
    if (x->d.ndim < 3) {
        PyErr_Format(g.exceptions[HIPCX_DIMENSION_ERROR], "pooling needs at least one spatial axis, got the shape %R", x->shape);
        throw PyError();
    }
    p->n = x->d.ndim - 2;
    Pair(ksize, p->n, 1, p->ksize);
    if (Given(stride)) {
        Pair(stride, p->n, 1, p->stride);
    } else {
        std::copy(p->ksize, p->ksize + p->n, p->stride);
    }
    Pair(pad, p->n, 0, p->pad);
    for (int i = 0; i < p->n; ++i) p->dims[i] = OutDim(x->d.shape[2 + i], p->ksize[i], p->stride[i], p->pad[i], cover_all);
}

// MaxPool (CX/routines/pooling.cc:52-123); one or more spatial axes (the dedicated kernels are the 2-D ones).
HOST_FN(MaxPool) {
    HOST_TRY;
    HOST_ARGS("max_pool", 2, "x", "ksize", "stride", "pad", "cover_all");
    Array* x = AsArray(arg[0], "x");
    const bool cover_all = Truth(arg[4]);
    PoolArgs p;
    PreparePool(&p, x, arg[1], arg[2], arg[3], cover_all);
    Ref out = SpatialOut(x, x->d.shape[1], p.dims, x->d.dtype);
    void* stream = Stream();
    Call([&] { return hipcx_max_pool(&x->d, p.ksize, p.stride, p.pad, cover_all ? 1 : 0, out.d(), stream); });
    return out.release();
    HOST_CATCH(nullptr);
}

int PadMode(PyObject* mode) {
    if (mode == nullptr) return HIPCX_PAD_IGNORE;
    if (PyUnicode_Check(mode)) {
        if (PyUnicode_CompareWithASCIIString(mode, "zero") == 0) return HIPCX_PAD_ZERO;
        if (PyUnicode_CompareWithASCIIString(mode, "ignore") == 0) return HIPCX_PAD_IGNORE;
    }
    PyErr_SetObject(PyExc_KeyError, mode);
    throw PyError();
}

// AveragePool (CX/routines/pooling.cc:125-169), float dtypes only; one or more spatial axes.
HOST_FN(AveragePool) {
    HOST_TRY;
    HOST_ARGS("average_pool", 2, "x", "ksize", "stride", "pad", "pad_mode");
    Array* x = AsArray(arg[0], "x");
    if (!IsFloat(x->d.dtype)) Raise(HIPCX_DTYPE_ERROR, "cannot apply average pooling to non-float arrays");
    const int mode = PadMode(arg[4]);
    PoolArgs p;
    PreparePool(&p, x, arg[1], arg[2], arg[3], false);
    Ref out = SpatialOut(x, x->d.shape[1], p.dims, x->d.dtype);
    void* stream = Stream();
    Call([&] { return hipcx_average_pool(&x->d, p.ksize, p.stride, p.pad, mode, out.d(), stream); });
    return out.release();
    HOST_CATCH(nullptr);
}

void CheckGout(const Array* x, const Array* gout, const PoolArgs& p) {
    bool ok = gout->d.ndim == x->d.ndim && gout->d.shape[0] == x->d.shape[0] && gout->d.shape[1] == x->d.shape[1];
    for (int i = 0; ok && i < p.n; ++i) ok = gout->d.shape[2 + i] == p.dims[i];
    if (!ok) Raise(HIPCX_DIMENSION_ERROR, "gout has the wrong shape");
}

// The dedicated kernel of MaxPoolGrad over two spatial axes: every input position gathers, in kernel-offset order, gout of the
// windows whose ArgMax it is.
HOST_FN(MaxPoolGrad2d) {
    HOST_TRY;
    HOST_ARGS("max_pool_grad", 3, "x", "gout", "ksize", "stride", "pad", "cover_all");
    Array *x = AsArray(arg[0], "x"), *gout = AsArray(arg[1], "gout");
    const bool cover_all = Truth(arg[5]);
    PoolArgs p;
    PreparePool(&p, x, arg[2], arg[3], arg[4], cover_all);
    CheckGout(x, gout, p);
    Ref gx = EmptyLike(x, x->d.dtype);
    Workspace ws(hipcx_max_pool_grad_workspace_size(&gout->d));
    void* stream = Stream();
    Call([&] { return hipcx_max_pool_grad(&x->d, &gout->d, p.ksize, p.stride, p.pad, cover_all ? 1 : 0, gx.d(), ws.ptr, ws.bytes, stream); });
    return gx.release();
    HOST_CATCH(nullptr);
}

HOST_FN(AveragePoolGrad2d) {
    HOST_TRY;
    HOST_ARGS("average_pool_grad", 3, "x", "gout", "ksize", "stride", "pad", "pad_mode");
    Array *x = AsArray(arg[0], "x"), *gout = AsArray(arg[1], "gout");
    const int mode = PadMode(arg[5]);
    PoolArgs p;
    p.n = 2;
    Pair(arg[2], 2, 1, p.ksize);
    if (Given(arg[3])) {
        Pair(arg[3], 2, 1, p.stride);
    } else {
        std::copy(p.ksize, p.ksize + 2, p.stride);
    }
    Pair(arg[4], 2, 0, p.pad);
    Ref gx = EmptyLike(x, x->d.dtype);
    void* stream = Stream();
    Call([&] { return hipcx_average_pool_grad(&gout->d, p.ksize, p.stride, p.pad, mode, gx.d(), stream); });
    return gx.release();
    HOST_CATCH(nullptr);
}

// ---------------------------------------------------------------------------------------------
// training: the calls the dedicated kernels take
// ---------------------------------------------------------------------------------------------
// ConvGradWeight over two spatial axes through hipcx_conv_grad_weight; the caller has checked shapes and dtype.
HOST_FN(ConvGradWeight2d) {
    HOST_TRY;
    HOST_ARGS("conv_grad_weight", 7, "w_dtype", "w_shape", "x", "gy", "stride", "pad", "cover_all");
    const int code = DtypeCode(arg[0]);
    int64_t w_shape[HIPCX_MAX_NDIM];
    if (ToShape(arg[1], w_shape) != 4) Raise(HIPCX_DIMENSION_ERROR, "w_shape needs four axes");
    int64_t stride[HIPCX_MAX_NDIM], pad[HIPCX_MAX_NDIM];
    Pair(arg[4], 2, 1, stride);
    Pair(arg[5], 2, 0, pad);
    const int cover_all = Truth(arg[6]) ? 1 : 0;
    Ref x = Cast(AsArray(arg[2], "x"), code), gy = Cast(AsArray(arg[3], "gy"), code);
    x = Contiguous(x.arr());
    gy = Contiguous(gy.arr());
    Ref gw = Empty(4, w_shape, code);
    Workspace ws(hipcx_conv_grad_weight_workspace_size(x.d(), gy.d(), gw.d(), stride, pad, cover_all));
    void* stream = Stream();
    Call([&] { return hipcx_conv_grad_weight(x.d(), gy.d(), stride, pad, cover_all, gw.d(), ws.ptr, ws.bytes, stream); });
    return gw.release();
    HOST_CATCH(nullptr);
}

// ConvTranspose over two spatial axes through hipcx_conv_transpose; the caller has checked shapes and dtype.
HOST_FN(ConvTranspose2d) {
    HOST_TRY;
    HOST_ARGS("conv_transpose", 7, "x", "w", "b", "stride", "pad", "out_size", "dtype");
    const int code = DtypeCode(arg[6]);
    int64_t stride[HIPCX_MAX_NDIM], pad[HIPCX_MAX_NDIM], size[HIPCX_MAX_NDIM];
    Pair(arg[3], 2, 1, stride);
    Pair(arg[4], 2, 0, pad);
    Pair(arg[5], 2, 0, size);
    Array *x0 = AsArray(arg[0], "x"), *w0 = AsArray(arg[1], "w");
    Ref x = Cast(x0, code), w = Cast(w0, code), b;
    if (Given(arg[2])) b = Cast(AsArray(arg[2], "b"), code);
    const int64_t shape[4] = {x0->d.shape[0], w0->d.shape[1], size[0], size[1]};
    Ref out = Empty(4, shape, code);
    Workspace ws(hipcx_conv_transpose_workspace_size(x.d(), w.d(), stride, pad, out.d()));
    void* stream = Stream();
    Call([&] { return hipcx_conv_transpose(x.d(), w.d(), b.d(), stride, pad, out.d(), ws.ptr, ws.bytes, stream); });
    return out.release();
    HOST_CATCH(nullptr);
}

// The dedicated batch-norm kernels take a C-contiguous x of fewer than 2^31 elements reduced over every axis but 1; the per-channel
// arrays share one dtype, x's or -- for a float16 x -- float32 (parameters and statistics of a float16 network kept in float32).
bool BnKernelApplies(const Array* x, const int8_t* axes, int n_axes, std::initializer_list<const Array*> params) {
    const int nd = x->d.ndim, pd = (*params.begin())->d.dtype;
    if (nd < 2 || n_axes != nd - 1 || !IsContiguous(x->d)) return false;
    for (int i = 0; i < n_axes; ++i) {
        if (axes[i] != (i == 0 ? 0 : i + 1)) return false;
    }
    const int64_t size = Size(x);
    if (size == 0 || size >= (int64_t{1} << 31)) return false;
    if (pd != x->d.dtype && !(x->d.dtype == HIPCX_FLOAT16 && pd == HIPCX_FLOAT32)) return false;
    return std::all_of(params.begin(), params.end(), [&](const Array* a) { return a->d.dtype == pd; });
}

int BnAxes(PyObject* axis, int ndim, int8_t* axes) {
    if (Given(axis)) return SortedAxes(axis, ndim, axes);
    int n = 0;
    for (int i = 0; i < ndim; ++i) {
        if (i != 1) axes[n++] = static_cast<int8_t>(i);
    }
    return n;
}

// BatchNorm in training mode through hipcx_batch_norm -> (out, (mean, inv_std, beta dtype)), or None for calls the dedicated
// kernels do not take.  `relu`: Relu of it, or of its sum with `residual`, through hipcx_batch_norm_relu -> (out, sum or None, state).
HOST_FN(BatchNormDirect) {
    HOST_TRY;
    HOST_ARGS("batch_norm", 5, "x", "gamma", "beta", "running_mean", "running_var", "eps", "decay", "axis", "relu", "residual");
    const bool relu = Given(arg[8]) && PyObject_IsTrue(arg[8]) == 1;
    Array* a[5];
    for (int i = 0; i < 5; ++i) {
        a[i] = AsArray(arg[i], "argument");
        if (!IsFloat(a[i]->d.dtype)) Raise(HIPCX_DTYPE_ERROR, "BatchNorm requires floating point arrays");
    }
    Array* x = a[0];
    int8_t axes[HIPCX_MAX_NDIM];
    const int n_axes = BnAxes(arg[7], x->d.ndim, axes);
    if (!BnKernelApplies(x, axes, n_axes, {a[1], a[2], a[3], a[4]})) Py_RETURN_NONE;
    Array* residual = Given(arg[9]) ? AsArray(arg[9], "residual") : nullptr;
    if (residual != nullptr && (residual->d.dtype != x->d.dtype || !ShapeIs(residual, x->d.ndim, x->d.shape) || !IsContiguous(residual->d))) Py_RETURN_NONE;
    int64_t reduced[HIPCX_MAX_NDIM];
    std::copy(x->d.shape, x->d.shape + x->d.ndim, reduced);
    for (int i = 0; i < n_axes; ++i) reduced[axes[i]] = 1;
    const int64_t channels = x->d.shape[1];
    for (int i = 1; i < 5; ++i) {
        // the running statistics are written in place: all four need to be seen as they lie in memory
        int64_t st[HIPCX_MAX_NDIM];
        if (Size(a[i]) != channels) {
            Raise(HIPCX_DIMENSION_ERROR, "cannot reshape array of size %lld into %lld channels", static_cast<long long>(Size(a[i])), static_cast<long long>(channels));
        }
        if (i >= 3 && !NoCopyReshape(a[i]->d, x->d.ndim, reduced, st)) Py_RETURN_NONE;
    }
    hipcx_array p[4];
    Ref keep[4];
    for (int i = 0; i < 4; ++i) p[i] = Reshaped(a[1 + i], x->d.ndim, reduced, &keep[i]);
    const int interm = Promote(Promote(x->d.dtype, a[1]->d.dtype), a[2]->d.dtype);  // the state's dtype (CX/routines/normalization.cc:141-150)
    const hipcx_scalar eps = FloatScalar(arg[5], 2e-5), decay = FloatScalar(arg[6], 0.9);
    Ref out = EmptyLike(x, x->d.dtype), mean = Empty(x->d.ndim, reduced, interm), inv_std = Empty(x->d.ndim, reduced, interm);
    Workspace ws(hipcx_batch_norm_workspace_size(&x->d, axes, n_axes));
    void* stream = Stream();
    if (relu) {
        Ref total = residual != nullptr ? EmptyLike(x, x->d.dtype) : Ref();
        Call([&] {
            return hipcx_batch_norm_relu(&x->d, &p[0], &p[1], &p[2], &p[3], eps, decay, axes, n_axes, residual != nullptr ? &residual->d : nullptr, total.d(),
                                         out.d(), mean.d(), inv_std.d(), ws.ptr, ws.bytes, stream);
        });
        Ref state(PyTuple_Pack(3, mean.get(), inv_std.get(), a[2]->dtype));
        if (!state) throw PyError();
        return PyTuple_Pack(3, out.get(), total ? total.get() : Py_None, state.get());
    }
    Call([&] {
        return hipcx_batch_norm(&x->d, &p[0], &p[1], &p[2], &p[3], eps, decay, axes, n_axes, out.d(), mean.d(), inv_std.d(), ws.ptr, ws.bytes, stream);
    });
    Ref state(PyTuple_Pack(3, mean.get(), inv_std.get(), a[2]->dtype));
    if (!state) throw PyError();
    return PyTuple_Pack(2, out.get(), state.get());
    HOST_CATCH(nullptr);
}

// GenericBatchNormGradKernel through hipcx_batch_norm_grad -> (gx, ggamma, gbeta), or None.
HOST_FN(BatchNormGradDirect) {
    HOST_TRY;
    HOST_ARGS("batch_norm_grad", 6, "x", "gamma", "gout", "x_mean", "x_inv_std", "beta_dtype", "axis", "relu_beta");
    Array *x = AsArray(arg[0], "x"), *gamma = AsArray(arg[1], "gamma"), *gout = AsArray(arg[2], "gout");
    Array* beta = Given(arg[7]) ? AsArray(arg[7], "beta") : nullptr;  // the gradient of Relu's input, through hipcx_batch_norm_relu_grad
    Array *mean = AsArray(arg[3], "x_mean"), *inv_std = AsArray(arg[4], "x_inv_std");
    int8_t axes[HIPCX_MAX_NDIM];
    const int n_axes = BnAxes(arg[6], x->d.ndim, axes);
    if (!BnKernelApplies(x, axes, n_axes, {gamma, mean, inv_std}) || gout->d.dtype != x->d.dtype || !ShapeIs(gout, x->d.ndim, x->d.shape) ||
        !IsContiguous(gout->d) || DtypeCode(arg[5]) != gamma->d.dtype || (beta != nullptr && beta->d.dtype != gamma->d.dtype)) {
        Py_RETURN_NONE;
    }
    int64_t reduced[HIPCX_MAX_NDIM];
    std::copy(x->d.shape, x->d.shape + x->d.ndim, reduced);
    for (int i = 0; i < n_axes; ++i) reduced[axes[i]] = 1;
    Array* in[4] = {gamma, mean, inv_std, beta};
    hipcx_array p[4];
    Ref keep[4];
    for (int i = 0; i < (beta != nullptr ? 4 : 3); ++i) {
        if (Size(in[i]) != x->d.shape[1]) {
            Raise(HIPCX_DIMENSION_ERROR, "cannot reshape array of size %lld into %lld channels", static_cast<long long>(Size(in[i])), static_cast<long long>(x->d.shape[1]));
        }
        p[i] = Reshaped(in[i], x->d.ndim, reduced, &keep[i]);
    }
    Ref gx = EmptyLike(x, x->d.dtype), ggamma = EmptyLike(gamma, gamma->d.dtype), gbeta = EmptyLike(gamma, gamma->d.dtype);
    Ref unused[2];
    const hipcx_array gg = Reshaped(ggamma.arr(), x->d.ndim, reduced, &unused[0]), gb = Reshaped(gbeta.arr(), x->d.ndim, reduced, &unused[1]);
    Workspace ws(hipcx_batch_norm_workspace_size(&x->d, axes, n_axes));
    void* stream = Stream();
    Call([&] {
        if (beta != nullptr) {
            return hipcx_batch_norm_relu_grad(&x->d, &p[0], &p[3], &gout->d, &p[1], &p[2], axes, n_axes, gx.d(), &gg, &gb, ws.ptr, ws.bytes, stream);
        }
        return hipcx_batch_norm_grad(&x->d, &p[0], &gout->d, &p[1], &p[2], axes, n_axes, gx.d(), &gg, &gb, ws.ptr, ws.bytes, stream);
    });
    return PyTuple_Pack(3, gx.get(), ggamma.get(), gbeta.get());
    HOST_CATCH(nullptr);
}

// x - g * s for every array x and its g, which is taken in x's shape; None for other than float arrays of one dtype each.
HOST_FN(SgdUpdate) {
    HOST_TRY;
    HOST_ARGS("sgd_update", 3, "params", "grads", "lr");
    std::vector<Ref> xs = Sequence(arg[0]), gs = Sequence(arg[1]);
    if (xs.size() != gs.size()) Raise(HIPCX_DIMENSION_ERROR, "sgd_update: one gradient per parameter is needed");
    if (!IsScalar(arg[2])) Py_RETURN_NONE;
    for (size_t i = 0; i < xs.size(); ++i) {
        const Array *x = xs[i].arr(), *g = gs[i].arr();
        if (!IsFloat(x->d.dtype) || g->d.dtype != x->d.dtype || Size(g) != Size(x)) Py_RETURN_NONE;
    }
    const hipcx_scalar lr = ToScalar(arg[2]);
    Ref list(PyList_New(static_cast<Py_ssize_t>(xs.size())));
    if (!list) throw PyError();
    std::vector<Ref> keep(xs.size());
    std::vector<hipcx_array> g_views(xs.size());
    std::vector<const hipcx_array*> x_ptrs, g_ptrs, out_ptrs;
    for (size_t i = 0; i < xs.size(); ++i) {
        Array* x = xs[i].arr();
        g_views[i] = Reshaped(gs[i].arr(), x->d.ndim, x->d.shape, &keep[i]);
        Ref out = EmptyLike(x, x->d.dtype);
        x_ptrs.push_back(&x->d);
        g_ptrs.push_back(&g_views[i]);
        out_ptrs.push_back(out.d());
        PyList_SET_ITEM(list.get(), static_cast<Py_ssize_t>(i), out.release());
    }
    void* stream = Stream();
    Call([&] { return hipcx_update_many(x_ptrs.data(), g_ptrs.data(), lr, out_ptrs.data(), static_cast<int>(xs.size()), stream); });
    return list.release();
    HOST_CATCH(nullptr);
}

// ---------------------------------------------------------------------------------------------
// indexing
// ---------------------------------------------------------------------------------------------
// Take (CX/routines/indexing.cc:171-205) for the bounds modes that need no read-back.
HOST_FN(TakeDeferred) {
    HOST_TRY;
    HOST_ARGS("take", 4, "a", "indices", "axis", "mode");
    Array *a = AsArray(arg[0], "a"), *indices = AsArray(arg[1], "indices");
    if (Kind(indices->d.dtype) != 1 && Kind(indices->d.dtype) != 2) Raise(HIPCX_DTYPE_ERROR, "Only arrays of integer dtype can be used as indices.");
    const int axis = NormalizeAxis(ToInt(arg[2]), a->d.ndim);
    const int mode = static_cast<int>(ToInt(arg[3]));
    const int nd = a->d.ndim - 1 + indices->d.ndim;
    if (nd > HIPCX_MAX_NDIM) Raise(HIPCX_DIMENSION_ERROR, "ndim %d exceeds the maximum of %d", nd, HIPCX_MAX_NDIM);
    int64_t shape[HIPCX_MAX_NDIM];
    int64_t* s = std::copy(a->d.shape, a->d.shape + axis, shape);
    s = std::copy(indices->d.shape, indices->d.shape + indices->d.ndim, s);
    std::copy(a->d.shape + axis + 1, a->d.shape + a->d.ndim, s);
    Ref out = Empty(nd, shape, a->d.dtype);
    void* stream = Stream();
    Call([&] { return hipcx_take(&a->d, &indices->d, static_cast<int8_t>(axis), out.d(), mode, nullptr, stream); });
    return out.release();
    HOST_CATCH(nullptr);
}

// ---------------------------------------------------------------------------------------------
// routine chains as one kernel call
// ---------------------------------------------------------------------------------------------
// LogSoftmax of a 2-D array along its unit-stride axis 1 through hipcx_log_softmax, or None for other calls: an axis without elements is
// an error that the chain's AMax raises.
HOST_FN(LogSoftmaxDirect) {
    HOST_TRY;
    HOST_ARGS("log_softmax", 1, "x", "axis");
    Array* x0 = AsArray(arg[0], "x");
    int8_t axes[HIPCX_MAX_NDIM] = {1};
    int n = 1;
    if (Given(arg[1])) {
        n = SortedAxes(arg[1], x0->d.ndim, axes);
    } else {
        NormalizeAxis(1, x0->d.ndim);
    }
    Ref x = Cast(x0, MathDtype(x0->d.dtype));
    const hipcx_array* d = x.d();
    if (d->ndim != 2 || n != 1 || axes[0] != 1 || d->shape[1] == 0 || (d->shape[1] > 1 && d->strides[1] != ItemSize(d->dtype)) ||
        d->strides[0] < 0) {
        Py_RETURN_NONE;
    }
    Ref out = EmptyLike(x.arr(), d->dtype);
    Workspace ws(hipcx_log_softmax_workspace_size(d));
    void* stream = Stream();
    Call([&] { return hipcx_log_softmax(d, out.d(), ws.ptr, ws.bytes, stream); });
    return out.release();
    HOST_CATCH(nullptr);
}

// The loss of the routine below in one call, or None for operands its kernel does not take.
HOST_FN(SoftmaxCrossEntropyDirect) {
    HOST_TRY;
    HOST_ARGS("softmax_cross_entropy", 2, "x", "t");
    Array *x0 = AsArray(arg[0], "x"), *t = AsArray(arg[1], "t");
    static const int64_t kMax[10] = {-1, -1, 127, 32767, INT32_MAX, INT64_MAX, 255, -1, -1, -1};  // the last class a label dtype can name
    if (x0->d.ndim != 2 || t->d.ndim != 1 || t->d.shape[0] != x0->d.shape[0] || x0->d.shape[0] == 0 || x0->d.shape[1] == 0 ||
        x0->d.shape[1] - 1 > kMax[t->d.dtype]) {
        Py_RETURN_NONE;
    }
    Ref x = Cast(x0, MathDtype(x0->d.dtype));
    const hipcx_array* d = x.d();
    if (d->shape[1] > 1 && d->strides[1] != ItemSize(d->dtype)) Py_RETURN_NONE;
    Ref out = Empty(0, nullptr, d->dtype);
    Workspace ws(hipcx_softmax_cross_entropy_workspace_size(d));
    void* stream = Stream();
    Call([&] { return hipcx_softmax_cross_entropy(d, &t->d, out.d(), ws.ptr, ws.bytes, stream); });
    return out.release();
    HOST_CATCH(nullptr);
}

// The Lstm cell of 2-D arrays with dense rows through hipcx_lstm_cell, or None for other calls.
HOST_FN(LstmCell) {
    HOST_TRY;
    HOST_ARGS("lstm_cell", 2, "c", "x");
    Array *c = AsArray(arg[0], "c"), *x = AsArray(arg[1], "x");
    for (const Array* a : {c, x}) {
        if (a->d.ndim != 2 || (a->d.shape[1] > 1 && a->d.strides[1] != ItemSize(a->d.dtype)) || a->d.strides[0] < 0) Py_RETURN_NONE;
    }
    Ref h = EmptyLike(c, c->d.dtype), new_c = EmptyLike(c, c->d.dtype);
    void* stream = Stream();
    Call([&] { return hipcx_lstm_cell(&c->d, &x->d, h.d(), new_c.d(), stream); });
    return PyTuple_Pack(2, h.get(), new_c.get());
    HOST_CATCH(nullptr);
}

// A step of an LSTM link through hipcx_lstm_step, or None for the calls to compose.
HOST_FN(LstmStep) {
    HOST_TRY;
    HOST_ARGS("lstm_step", 6, "c", "x", "wx", "bx", "h", "wh");
    Array *c = AsArray(arg[0], "c"), *x = AsArray(arg[1], "x"), *wx = AsArray(arg[2], "wx"), *bx = Given(arg[3]) ? AsArray(arg[3], "bx") : nullptr;
    Array *h = AsArray(arg[4], "h"), *wh = AsArray(arg[5], "wh");
    const hipcx_array* const bias = bx != nullptr ? &bx->d : nullptr;
    if (hipcx_lstm_step_supported(&c->d, &x->d, &wx->d, bias, &h->d, &wh->d) == 0) Py_RETURN_NONE;
    Ref new_h = EmptyLike(c, c->d.dtype), new_c = EmptyLike(c, c->d.dtype);
    void* stream = Stream();
    Call([&] { return hipcx_lstm_step(&c->d, &x->d, &wx->d, bias, &h->d, &wh->d, new_h.d(), new_c.d(), stream); });
    return PyTuple_Pack(2, new_h.get(), new_c.get());
    HOST_CATCH(nullptr);
}

// ---------------------------------------------------------------------------------------------
// recurrent networks
// ---------------------------------------------------------------------------------------------
std::vector<const hipcx_array*> Descriptors(const std::vector<Ref>& arrays) {
    std::vector<const hipcx_array*> v;
    v.reserve(arrays.size());
    for (const Ref& r : arrays) v.push_back(r.d());
    return v;
}

std::vector<Ref> EmptyLikeAll(const std::vector<Ref>& arrays) {
    std::vector<Ref> v;
    v.reserve(arrays.size());
    for (const Ref& r : arrays) v.push_back(EmptyLike(r.arr(), r.arr()->d.dtype));
    return v;
}

PyObject* ToList(std::vector<Ref>* arrays) {
    PyObject* list = PyList_New(static_cast<Py_ssize_t>(arrays->size()));
    if (list == nullptr) throw PyError();
    for (size_t i = 0; i < arrays->size(); ++i) PyList_SET_ITEM(list, static_cast<Py_ssize_t>(i), (*arrays)[i].release());
    return list;
}

// Output rows of every time step.
std::vector<Ref> StepOutputs(const std::vector<Ref>& xs, int64_t width, int code) {
    std::vector<Ref> ys;
    ys.reserve(xs.size());
    for (const Ref& x : xs) {
        if (x.arr()->d.ndim < 1) Raise(HIPCX_DIMENSION_ERROR, "the input of a time step needs two axes");
        const int64_t shape[2] = {x.arr()->d.shape[0], width};
        ys.push_back(Empty(2, shape, code));
    }
    return ys;
}

// hipcx_n_step_rnn -> (hy, cy or None, ys, reserve or None).
HOST_FN(RnnForward) {
    HOST_TRY;
    HOST_ARGS("rnn", 10, "n_layers", "bidirectional", "mode", "activation", "training", "hx", "cx", "ws", "bs", "xs");
    const int layers = static_cast<int>(ToInt(arg[0])), bi = Truth(arg[1]) ? 1 : 0, mode = static_cast<int>(ToInt(arg[2]));
    const int act = static_cast<int>(ToInt(arg[3])), training = Truth(arg[4]) ? 1 : 0;
    Array *hx = AsArray(arg[5], "hx"), *cx = mode == 1 ? AsArray(arg[6], "cx") : nullptr;
    if (hx->d.ndim != 3) Raise(HIPCX_DIMENSION_ERROR, "hx needs three axes");
    std::vector<Ref> ws = Sequence(arg[7]), bs = Sequence(arg[8]), xs = Sequence(arg[9]);
    Ref hy = EmptyLike(hx, hx->d.dtype), cy;
    if (cx != nullptr) cy = EmptyLike(cx, cx->d.dtype);
    std::vector<Ref> ys = StepOutputs(xs, (1 + bi) * hx->d.shape[2], hx->d.dtype);
    auto pw = Descriptors(ws), pb = Descriptors(bs), px = Descriptors(xs), py = Descriptors(ys);
    const int steps = static_cast<int>(xs.size());
    Ref reserve;
    size_t reserve_bytes = 0;
    if (training) {
        reserve_bytes = hipcx_n_step_rnn_reserve_size(layers, bi, mode, &hx->d, px.data(), steps);
        reserve = NewBuffer(reserve_bytes);
    }
    void* reserve_ptr = reserve ? reinterpret_cast<Buffer*>(reserve.get())->ptr : nullptr;
    Workspace scratch(hipcx_n_step_rnn_workspace_size(layers, bi, mode, training, &hx->d, px.data(), steps));
    void* stream = Stream();
    Call([&] {
        return hipcx_n_step_rnn(layers, bi, mode, act, &hx->d, cx != nullptr ? &cx->d : nullptr, pw.data(), pb.data(), px.data(), steps, hy.d(),
                                cy.d(), py.data(), reserve_ptr, reserve_bytes, scratch.ptr, scratch.bytes, stream);
    });
    Ref list(ToList(&ys));
    return PyTuple_Pack(4, hy.get(), cy ? cy.get() : Py_None, list.get(), reserve ? reserve.get() : Py_None);
    HOST_CATCH(nullptr);
}

// hipcx_n_step_rnn_backward -> (dhx, dcx or None, dws, dbs, dxs).
HOST_FN(RnnBackward) {
    HOST_TRY;
    HOST_ARGS("rnn_backward", 12, "n_layers", "bidirectional", "mode", "activation", "hx", "ws", "bs", "xs", "reserve", "dhy", "dcy", "dys");
    const int layers = static_cast<int>(ToInt(arg[0])), bi = Truth(arg[1]) ? 1 : 0, mode = static_cast<int>(ToInt(arg[2]));
    const int act = static_cast<int>(ToInt(arg[3]));
    Array *hx = AsArray(arg[4], "hx"), *dhy = AsArray(arg[9], "dhy"), *dcy = Given(arg[10]) && mode == 1 ? AsArray(arg[10], "dcy") : nullptr;
    std::vector<Ref> ws = Sequence(arg[5]), bs = Sequence(arg[6]), xs = Sequence(arg[7]);
    if (!Py_IS_TYPE(arg[8], &BufferType)) Raise(HIPCX_CHAINERX_ERROR, "rnn_backward needs the reserve of a training call");
    Buffer* reserve = reinterpret_cast<Buffer*>(arg[8]);
    Ref dys(PySequence_List(arg[11]));
    if (!dys) throw PyError();
    std::vector<const hipcx_array*> pdy;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(dys.get()); ++i) {
        PyObject* o = PyList_GET_ITEM(dys.get(), i);
        pdy.push_back(o == Py_None ? nullptr : &AsArray(o, "dy")->d);
    }
    if (pdy.size() != xs.size()) Raise(HIPCX_DIMENSION_ERROR, "one gradient per time step is needed");
    Ref dhx = EmptyLike(hx, hx->d.dtype), dcx;
    if (mode == 1) dcx = EmptyLike(hx, hx->d.dtype);
    std::vector<Ref> dws = EmptyLikeAll(ws), dbs = EmptyLikeAll(bs), dxs = EmptyLikeAll(xs);
    auto pw = Descriptors(ws), pb = Descriptors(bs), px = Descriptors(xs), pdw = Descriptors(dws), pdb = Descriptors(dbs), pdx = Descriptors(dxs);
    const int steps = static_cast<int>(xs.size());
    Workspace scratch(hipcx_n_step_rnn_workspace_size(layers, bi, mode, 1, &hx->d, px.data(), steps));
    void* stream = Stream();
    Call([&] {
        return hipcx_n_step_rnn_backward(layers, bi, mode, act, &hx->d, pw.data(), pb.data(), px.data(), steps, &dhy->d,
                                         dcy != nullptr ? &dcy->d : nullptr, pdy.data(), reserve->ptr, reserve->nbytes, dhx.d(), dcx.d(), pdw.data(),
                                         pdb.data(), pdx.data(), scratch.ptr, scratch.bytes, stream);
    });
    Ref lw(ToList(&dws)), lb(ToList(&dbs)), lx(ToList(&dxs));
    return PyTuple_Pack(5, dhx.get(), dcx ? dcx.get() : Py_None, lw.get(), lb.get(), lx.get());
    HOST_CATCH(nullptr);
}

}  // namespace

#define ROUTINE(name, fn, doc) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(fn)), METH_FASTCALL | METH_KEYWORDS, doc}
PyMethodDef kRoutines[] = {
        ROUTINE("add", Add, "Add (CX/routines/arithmetic.cc)."),
        ROUTINE("subtract", Subtract, "Subtract; Subtract(Scalar, Array) = Add(-Array, Scalar) (CX/routines/arithmetic.cc)."),
        ROUTINE("multiply", Multiply, "Multiply (CX/routines/arithmetic.cc)."),
        ROUTINE("divide", Divide, "TrueDivide: integer operands are computed in float32 (CX/routines/arithmetic.cc Divide)."),
        ROUTINE("negative", Negative, "Negative = Multiply(x, Scalar{-1}) (CX/routines/arithmetic.cc)."),
        ROUTINE("reciprocal", Reciprocal, "Reciprocal(x) = Scalar{1} / x (CX/routines/arithmetic.cc)."),
        ROUTINE("exp", Exp, nullptr),
        ROUTINE("log", Log, nullptr),
        ROUTINE("tanh", Tanh, nullptr),
        ROUTINE("sqrt", Sqrt, nullptr),
        ROUTINE("sigmoid", Sigmoid, "Sigmoid(x) = Reciprocal(1 + Exp(-x)) (CX/routines/activation.cc:74-78)."),
        ROUTINE("relu", Relu, "Relu(x) = Maximum(0, x) in the math dtype of x (CX/routines/activation.cc:80-84)."),
        ROUTINE("if_less_else", IfLessElse, "x1 < x2 ? pos : neg with scalar x2/pos (CX/routines/misc.cc:34-58)."),
        ROUTINE("if_greater_else", IfGreaterElse, "x1 > x2 ? pos : neg with scalar x2/pos (CX/routines/misc.cc:34-58)."),
        ROUTINE("maximum", Maximum, "Maximum(array, scalar) = IfLessElse(x1, x2, x2, x1) (CX/routines/misc.cc:210-216)."),
        ROUTINE("equal", Equal, nullptr),
        ROUTINE("not_equal", NotEqual, nullptr),
        ROUTINE("greater", Greater, nullptr),
        ROUTINE("greater_equal", GreaterEqual, nullptr),
        ROUTINE("full", Full, nullptr),
        ROUTINE("split", Split, "Split into views (CX/routines/manipulation.cc Split)."),
        ROUTINE("concatenate", Concatenate, "Concatenate = Empty + one CopyKernel per input (CX/routines/manipulation.cc:415-460)."),
        ROUTINE("stack", Stack, "Stack = Empty + one CopyKernel per input into a view of the new axis (CX/routines/manipulation.cc Stack)."),
        ROUTINE("sum", Sum, "Sum (CX/routines/reduction.cc:28-76): bool/int inputs accumulate and return int64."),
        ROUTINE("amax", AMax, "AMax (CX/routines/statistics.cc:21-65)."),
        ROUTINE("amin", AMin, "AMin (CX/routines/statistics.cc:66-79)."),
        ROUTINE("argmax", ArgMax, "ArgMax (CX/routines/sorting.cc:21-52): int64 result, no keepdims."),
        ROUTINE("argmin", ArgMin, "ArgMin (CX/routines/sorting.cc:54-85): int64 result, no keepdims."),
        ROUTINE("dot", Dot, "Dot for 2-D operands (CX/routines/linalg.cc:27-100): k == 0 gives zeros without a kernel."),
        ROUTINE("linear", Linear, "Linear (CX/routines/connection.cc:322-394): DotKernel(x, w.T view), then the bias added."),
        ROUTINE("conv", Conv, "Conv (CX/routines/connection.cc:140-208): one ConvKernel call with the bias inside; any number of spatial axes."),
        ROUTINE("conv_bn_act", ConvBnAct,
                "Opt-in fused block: relu(fixed_batch_norm(conv(x, w, b), *bn, eps, axis=(0, 2, 3)) + residual) in one kernel call.\n"
                "`bn` is None or (gamma, beta, mean, var), one value per output channel.  Not part of the ChainerX routine surface:\n"
                "the reference issues these as separate kernels (which `conv`, `fixed_batch_norm`, `add`, `relu` here do as well)."),
        ROUTINE("fixed_batch_norm", FixedBatchNorm, "FixedBatchNorm (CX/routines/normalization.cc:414-424, PreprocessBatchNorm :61-101)."),
        ROUTINE("max_pool", MaxPool, "MaxPool (CX/routines/pooling.cc:52-123); one or more spatial axes."),
        ROUTINE("average_pool", AveragePool, "AveragePool (CX/routines/pooling.cc:125-169), float dtypes only; one or more spatial axes."),
        ROUTINE("max_pool_grad_2d", MaxPoolGrad2d, nullptr),
        ROUTINE("average_pool_grad_2d", AveragePoolGrad2d, nullptr),
        ROUTINE("conv_grad_weight_2d", ConvGradWeight2d, nullptr),
        ROUTINE("conv_transpose_2d", ConvTranspose2d, nullptr),
        ROUTINE("sgd_update_direct", SgdUpdate, nullptr),
        ROUTINE("add_relu_grad_direct", AddReluGrad, nullptr),
        ROUTINE("batch_norm_direct", BatchNormDirect, nullptr),
        ROUTINE("batch_norm_grad_direct", BatchNormGradDirect, nullptr),
        ROUTINE("take_deferred", TakeDeferred, nullptr),
        ROUTINE("log_softmax_direct", LogSoftmaxDirect, nullptr),
        ROUTINE("softmax_cross_entropy_direct", SoftmaxCrossEntropyDirect, nullptr),
        ROUTINE("lstm_cell", LstmCell, nullptr),
        ROUTINE("lstm_step_direct", LstmStep, nullptr),
        ROUTINE("rnn_forward", RnnForward, nullptr),
        ROUTINE("rnn_backward", RnnBackward, nullptr),
        {nullptr, nullptr, 0, nullptr}};

}  // namespace host
