// chainer_amd._host: buffers, arrays and their views.  Semantics of the views follow chainerx::Array: host-only (shape, byte
// strides, offset) arithmetic over one allocation (CX/routines/manipulation.cc, CX/routines/indexing.cc).
#include <algorithm>
#include <cstdarg>
#include <cstddef>

#include "host.h"

#include <structmember.h>

namespace host {

State g;

namespace {
constexpr int kDevice = 0;  // one process drives one device
}

// ---------------------------------------------------------------------------------------------
// errors
// ---------------------------------------------------------------------------------------------
void Raise(int status, const char* format, ...) {
    va_list ap;
    va_start(ap, format);
    PyErr_FormatV(g.exceptions[status], format, ap);
    va_end(ap);
    throw PyError();
}

void Check(int status) {
    if (status == 0) return;
    PyObject* type = status >= 1 && status <= 8 ? g.exceptions[status] : g.exceptions[1];
    PyObject* msg = PyUnicode_DecodeUTF8(hipcx_last_error(), static_cast<Py_ssize_t>(strlen(hipcx_last_error())), "replace");
    if (msg != nullptr) {
        PyErr_SetObject(type, msg);
        Py_DECREF(msg);
    }
    throw PyError();
}

// ---------------------------------------------------------------------------------------------
// dtypes and scalars (CX/dtype.cc:12-60, CX/routines/type_util.cc:11-46)
// ---------------------------------------------------------------------------------------------
int DtypeCode(PyObject* dtype) {
    for (int i = 1; i < 10; ++i) {
        if (g.dtypes[i] == dtype) return i;
    }
    Ref dt(PyObject_CallOneArg(g.np_dtype, dtype));
    if (!dt) throw PyError();
    for (int i = 1; i < 10; ++i) {
        if (g.dtypes[i] == dt.get()) return i;
    }
    for (int i = 1; i < 10; ++i) {
        int same = PyObject_RichCompareBool(g.dtypes[i], dt.get(), Py_EQ);
        if (same < 0) throw PyError();
        if (same) return i;
    }
    PyErr_Format(g.exceptions[HIPCX_DTYPE_ERROR], "unsupported dtype: %S", dtype);
    throw PyError();
}

int Promote(int a, int b) {
    int ka = Kind(a), kb = Kind(b);
    if (ka == 0) return b;
    if (kb == 0) return a;
    if (ka == kb) return ItemSize(a) >= ItemSize(b) ? a : b;
    if (ka == 3) return a;
    if (kb == 3) return b;
    if (ka == 2) std::swap(a, b);
    return ItemSize(a) > ItemSize(b) ? a : HIPCX_INT16;  // signed one level wider than uint8
}

namespace {
// 0 bool, 1 int, 3 float, -1 no scalar
int ScalarKind(PyObject* x) {
    if (PyFloat_Check(x)) return HIPCX_KIND_FLOAT;
    if (PyBool_Check(x)) return HIPCX_KIND_BOOL;
    if (PyLong_Check(x)) return HIPCX_KIND_INT;
    if (IsArray(x) || PyTuple_Check(x) || PyList_Check(x)) return -1;
    const std::pair<PyObject*, int> types[] = {{g.np_bool, HIPCX_KIND_BOOL}, {g.np_integer, HIPCX_KIND_INT}, {g.np_floating, HIPCX_KIND_FLOAT}};
    for (auto& t : types) {
        int is = PyObject_IsInstance(x, t.first);
        if (is < 0) throw PyError();
        if (is) return t.second;
    }
    return -1;
}
}  // namespace

bool IsScalar(PyObject* x) { return ScalarKind(x) >= 0; }

int ScalarDtype(PyObject* x) {
    int k = ScalarKind(x);
    return k == HIPCX_KIND_BOOL ? HIPCX_BOOL : k == HIPCX_KIND_INT ? HIPCX_INT32 : HIPCX_FLOAT32;
}

hipcx_scalar ToScalar(PyObject* x) {
    hipcx_scalar s;
    std::memset(&s, 0, sizeof(s));
    int k = ScalarKind(x);
    if (k < 0) {
        PyErr_Format(PyExc_TypeError, "unsupported scalar type: %R", Py_TYPE(x));
        throw PyError();
    }
    s.kind = k;
    if (k == HIPCX_KIND_BOOL) {
        int v = PyObject_IsTrue(x);
        if (v < 0) throw PyError();
        s.i = v;
        s.f = v;
    } else if (k == HIPCX_KIND_INT) {
        // values beyond 64 bits keep their low bits, as a ctypes int64 field does
        Ref n(PyNumber_Index(x));
        if (!n) throw PyError();
        s.i = static_cast<int64_t>(PyLong_AsUnsignedLongLongMask(n.get()));
        if (PyErr_Occurred()) throw PyError();
        s.f = PyLong_AsDouble(n.get());
        if (s.f == -1.0 && PyErr_Occurred()) throw PyError();
    } else {
        s.f = PyFloat_AsDouble(x);
        if (s.f == -1.0 && PyErr_Occurred()) throw PyError();
    }
    return s;
}

int ResultType(std::initializer_list<PyObject*> args) {
    int arr = 0, sc = 0;
    for (PyObject* a : args) {
        if (a == nullptr) continue;
        if (IsArray(a)) {
            int c = reinterpret_cast<Array*>(a)->d.dtype;
            arr = arr == 0 ? c : Promote(arr, c);
        } else {
            int c = ScalarDtype(a);
            sc = sc == 0 ? c : Promote(sc, c);
        }
    }
    if (arr != 0) {
        auto category = [](int code) { return Kind(code) == 0 ? 0 : Kind(code) == 3 ? 2 : 1; };
        return sc != 0 && category(sc) > category(arr) ? sc : arr;
    }
    return sc;
}

Array* AsArray(PyObject* x, const char* what) {
    if (!IsArray(x)) {
        PyErr_Format(PyExc_TypeError, "%s must be a chainer_amd.ndarray, got %R", what, Py_TYPE(x));
        throw PyError();
    }
    return reinterpret_cast<Array*>(x);
}

// ---------------------------------------------------------------------------------------------
// integers, shapes
// ---------------------------------------------------------------------------------------------
int64_t ToInt(PyObject* x) {
    if (PyLong_CheckExact(x)) {
        int64_t v = PyLong_AsLongLong(x);
        if (v == -1 && PyErr_Occurred()) throw PyError();
        return v;
    }
    Ref n(PyNumber_Long(x));  // int(x)
    if (!n) throw PyError();
    int64_t v = PyLong_AsLongLong(n.get());
    if (v == -1 && PyErr_Occurred()) throw PyError();
    return v;
}

int ToShape(PyObject* x, int64_t* shape) {
    if (PyLong_Check(x) || (!PyTuple_Check(x) && !PyList_Check(x) && PyIndex_Check(x))) {
        shape[0] = ToInt(x);
        return 1;
    }
    Ref seq(PySequence_Fast(x, "a shape is an int or a sequence of ints"));
    if (!seq) throw PyError();
    Py_ssize_t n = PySequence_Fast_GET_SIZE(seq.get());
    if (n > HIPCX_MAX_NDIM) Raise(HIPCX_DIMENSION_ERROR, "ndim %zd exceeds the maximum of %d", n, HIPCX_MAX_NDIM);
    for (Py_ssize_t i = 0; i < n; ++i) shape[i] = ToInt(PySequence_Fast_GET_ITEM(seq.get(), i));
    return static_cast<int>(n);
}

int NormalizeAxis(int64_t axis, int ndim) {
    if (axis < -ndim || axis >= ndim) {
        Raise(HIPCX_DIMENSION_ERROR, "axis %lld is out of bounds for array of dimension %d", static_cast<long long>(axis), ndim);
    }
    return static_cast<int>(axis < 0 ? axis + ndim : axis);
}

bool Flag(PyObject* name) {
    PyObject* v = PyDict_GetItem(g.flags, name);  // borrowed
    return v != nullptr && v != Py_False && PyObject_IsTrue(v) == 1;
}

void ContiguousStrides(int ndim, const int64_t* shape, int itemsize, int64_t* strides) {
    int64_t acc = itemsize;
    for (int i = ndim - 1; i >= 0; --i) {
        strides[i] = acc;
        acc *= std::max<int64_t>(1, shape[i]);
    }
}

void DenseStridesLike(const Array* a, int itemsize, int64_t* strides) {
    int order[HIPCX_MAX_NDIM];
    const int nd = a->d.ndim;
    for (int i = 0; i < nd; ++i) order[i] = i;
    std::stable_sort(order, order + nd, [&](int x, int y) { return std::abs(a->d.strides[x]) > std::abs(a->d.strides[y]); });
    int64_t acc = itemsize;
    for (int k = nd - 1; k >= 0; --k) {
        strides[order[k]] = acc;
        acc *= std::max<int64_t>(1, a->d.shape[order[k]]);
    }
}

bool IsContiguous(const hipcx_array& d) {
    int64_t expect = ItemSize(d.dtype);
    for (int i = d.ndim - 1; i >= 0; --i) {
        if (d.shape[i] == 0) return true;
        if (d.shape[i] != 1 && d.strides[i] != expect) return false;
        expect *= d.shape[i];
    }
    return true;
}

// Strides of `shape` over the same memory (CX/routines/manipulation.cc:153-258); false if a copy is needed.
bool NoCopyReshape(const hipcx_array& d, int ndim, const int64_t* shape, int64_t* strides) {
    const int itemsize = ItemSize(d.dtype);
    if (Product(d.ndim, d.shape) == 0) {
        ContiguousStrides(ndim, shape, itemsize, strides);
        return true;
    }
    int64_t od[HIPCX_MAX_NDIM], os[HIPCX_MAX_NDIM];
    int no = 0;
    for (int i = 0; i < d.ndim; ++i) {
        if (d.shape[i] != 1) od[no] = d.shape[i], os[no++] = d.strides[i];
    }
    int oi = 0, ni = 0;
    while (ni < ndim) {
        if (shape[ni] == 1) {
            strides[ni++] = itemsize;
            continue;
        }
        if (oi >= no) return false;
        // a group of new axes and a group of old axes of equal size
        int64_t np = shape[ni], op = od[oi];
        int nj = ni + 1, oj = oi + 1;
        while (np != op) {
            if (np < op) {
                while (nj < ndim && shape[nj] == 1) ++nj;
                if (nj >= ndim) return false;
                np *= shape[nj++];
            } else {
                if (oj >= no) return false;
                op *= od[oj++];
            }
        }
        for (int k = oi; k + 1 < oj; ++k) {
            if (os[k] != od[k + 1] * os[k + 1]) return false;
        }
        int64_t st = os[oj - 1];
        for (int k = nj - 1; k >= ni; --k) {
            strides[k] = st;
            st *= shape[k];
        }
        ni = nj;
        oi = oj;
    }
    return oi == no;
}

// ---------------------------------------------------------------------------------------------
// streams and buffers
// ---------------------------------------------------------------------------------------------
namespace {
void RequireDevice() {
    if (g.ready) return;
    Ref r(PyObject_CallNoArgs(g.require_device));
    if (!r) throw PyError();
    g.ready = true;
}
}  // namespace

void* Stream() {
    RequireDevice();
    Ref dev(PyObject_CallNoArgs(g.get_device));
    if (!dev) throw PyError();
    Ref s(PyObject_CallOneArg(g.raw_stream, dev.get()));
    if (!s) throw PyError();
    void* p = PyLong_AsVoidPtr(s.get());
    if (p == nullptr && PyErr_Occurred()) throw PyError();
    return p;
}

Ref NewBuffer(size_t nbytes) {
    void* stream = Stream();
    void* ptr = nullptr;
    Call([&] { return hipcx_malloc_on_stream(kDevice, nbytes != 0 ? nbytes : 1, stream, &ptr); });
    Buffer* b = PyObject_New(Buffer, &BufferType);
    if (b == nullptr) {
        (void)hipcx_free(kDevice, ptr);
        throw PyError();
    }
    b->ptr = ptr;
    b->nbytes = nbytes;
    b->weakrefs = nullptr;
    return Ref(b);
}

namespace {
PyObject* BufferNew(PyTypeObject*, PyObject* args, PyObject* kwargs) {
    HOST_TRY;
    Py_ssize_t n = 0;
    static const char* kw[] = {"nbytes", nullptr};
    if (!PyArg_ParseTupleAndKeywords(args, kwargs, "n", const_cast<char**>(kw), &n)) return nullptr;
    return NewBuffer(static_cast<size_t>(n)).release();
    HOST_CATCH(nullptr);
}

void BufferDealloc(PyObject* self) {
    Buffer* b = reinterpret_cast<Buffer*>(self);
    if (b->weakrefs != nullptr) PyObject_ClearWeakRefs(self);
    if (b->ptr != nullptr) (void)hipcx_free(kDevice, b->ptr);
    PyObject_Free(self);
}

PyObject* BufferAdopt(PyObject*, PyObject* args) {
    PyObject* ptr;
    Py_ssize_t nbytes;
    if (!PyArg_ParseTuple(args, "On", &ptr, &nbytes)) return nullptr;
    void* p = ptr == Py_None ? nullptr : PyLong_AsVoidPtr(ptr);
    if (p == nullptr && PyErr_Occurred()) return nullptr;
    Buffer* b = PyObject_New(Buffer, &BufferType);
    if (b == nullptr) return nullptr;
    b->ptr = p;
    b->nbytes = static_cast<size_t>(nbytes);
    b->weakrefs = nullptr;
    return reinterpret_cast<PyObject*>(b);
}

PyObject* BufferDataPtr(PyObject* self, PyObject*) { return PyLong_FromVoidPtr(reinterpret_cast<Buffer*>(self)->ptr); }
PyObject* BufferGetPtr(PyObject* self, void*) { return PyLong_FromVoidPtr(reinterpret_cast<Buffer*>(self)->ptr); }

PyObject* BufferRecordStream(PyObject* self, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
    HOST_TRY;
    HOST_ARGS("record_stream", 0, "stream");
    Buffer* b = reinterpret_cast<Buffer*>(self);
    if (b->ptr == nullptr) Py_RETURN_NONE;
    void* stream;
    if (!Given(arg[0])) {
        stream = Stream();
    } else {
        Ref handle;  // an int, or a ctypes.c_void_p
        if (PyLong_Check(arg[0])) {
            Py_INCREF(arg[0]);
            handle = Ref(arg[0]);
        } else {
            handle = Ref(PyObject_GetAttrString(arg[0], "value"));
            if (!handle) throw PyError();
        }
        stream = handle.get() == Py_None ? nullptr : PyLong_AsVoidPtr(handle.get());
        if (stream == nullptr && PyErr_Occurred()) throw PyError();
    }
    Call([&] { return hipcx_record_stream(kDevice, b->ptr, stream); });
    Py_RETURN_NONE;
    HOST_CATCH(nullptr);
}

PyMethodDef kBufferMethods[] = {
        {"data_ptr", BufferDataPtr, METH_NOARGS, "Device address of the block."},
        {"adopt", BufferAdopt, METH_VARARGS | METH_STATIC, "Takes ownership of a pointer the pool has already handed out (hipcx_from_host_memory)."},
        {"record_stream", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(BufferRecordStream)), METH_FASTCALL | METH_KEYWORDS,
         "Announces that work on this block is queued on ``stream`` (a raw stream handle; default: the current stream), which is not\n"
         "the stream it was allocated on: the pool then holds the block back after its release until that work has run\n"
         "(hipcx_record_stream)."},
        {nullptr, nullptr, 0, nullptr}};
PyGetSetDef kBufferGetSet[] = {{"ptr", BufferGetPtr, nullptr, nullptr, nullptr}, {nullptr, nullptr, nullptr, nullptr, nullptr}};
PyMemberDef kBufferMembers[] = {{"nbytes", T_PYSSIZET, offsetof(Buffer, nbytes), READONLY, nullptr}, {nullptr, 0, 0, 0, nullptr}};
}  // namespace

PyTypeObject BufferType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// ---------------------------------------------------------------------------------------------
// arrays
// ---------------------------------------------------------------------------------------------
namespace {
PyObject* IntTuple(int n, const int64_t* v) {
    PyObject* t = PyTuple_New(n);
    if (t == nullptr) throw PyError();
    for (int i = 0; i < n; ++i) {
        PyObject* o = PyLong_FromLongLong(v[i]);
        if (o == nullptr) {
            Py_DECREF(t);
            throw PyError();
        }
        PyTuple_SET_ITEM(t, i, o);
    }
    return t;
}

Ref MakeArray(PyTypeObject* type, PyObject* buf, int64_t offset, char* data, int ndim, const int64_t* shape, const int64_t* strides, int code) {
    Ref shape_tuple(IntTuple(ndim, shape));
    Array* a = reinterpret_cast<Array*>(type->tp_alloc(type, 0));
    if (a == nullptr) throw PyError();
    Py_INCREF(buf);
    a->buf = buf;
    Py_INCREF(g.dtypes[code]);
    a->dtype = g.dtypes[code];
    a->shape = shape_tuple.release();
    a->strides = nullptr;
    a->cdesc = nullptr;
    a->offset = offset;
    a->d.data = data;
    a->d.dtype = code;
    a->d.ndim = ndim;
    std::memcpy(a->d.shape, shape, ndim * sizeof(int64_t));
    std::memcpy(a->d.strides, strides, ndim * sizeof(int64_t));
    return Ref(a);
}
}  // namespace

Ref NewArray(PyObject* buf, int64_t offset, char* data, int ndim, const int64_t* shape, const int64_t* strides, int code) {
    return MakeArray(reinterpret_cast<PyTypeObject*>(g.ndarray), buf, offset, data, ndim, shape, strides, code);
}

Ref EmptyStrided(int ndim, const int64_t* shape, const int64_t* strides, int64_t bytes, int code) {
    Ref buf = NewBuffer(static_cast<size_t>(bytes));
    return NewArray(buf.get(), 0, static_cast<char*>(reinterpret_cast<Buffer*>(buf.get())->ptr), ndim, shape, strides, code);
}

Ref Empty(int ndim, const int64_t* shape, int code) {
    int64_t strides[HIPCX_MAX_NDIM];
    const int it = ItemSize(code);
    ContiguousStrides(ndim, shape, it, strides);
    return EmptyStrided(ndim, shape, strides, Product(ndim, shape) * it, code);
}

Ref NewRef(Array* a) {
    Py_INCREF(a);
    return Ref(a);
}

Ref View(Array* a, int64_t offset_delta, int ndim, const int64_t* shape, const int64_t* strides) {
    return NewArray(a->buf, a->offset + offset_delta, static_cast<char*>(a->d.data) + offset_delta, ndim, shape, strides, a->d.dtype);
}

Ref CopyOf(Array* a, int code) {
    Ref out = EmptyLike(a, code);
    void* stream = Stream();
    Call([&] { return hipcx_copy(&a->d, out.d(), stream); });
    return out;
}

Ref Cast(Array* a, int code) { return a->d.dtype == code ? NewRef(a) : CopyOf(a, code); }

Ref Contiguous(Array* a) { return IsContiguous(a->d) ? NewRef(a) : CopyOf(a, a->d.dtype); }

Ref BroadcastTo(Array* a, int ndim, const int64_t* shape) {
    const int lead = ndim - a->d.ndim;
    int64_t strides[HIPCX_MAX_NDIM] = {};
    bool ok = lead >= 0;
    for (int i = 0; ok && i < a->d.ndim; ++i) {
        const int64_t n = a->d.shape[i];
        if (n == shape[lead + i]) {
            strides[lead + i] = n != 1 ? a->d.strides[i] : 0;
        } else if (n != 1) {
            ok = false;
        }
    }
    if (!ok) {
        Ref to(IntTuple(ndim, shape));
        PyErr_Format(g.exceptions[HIPCX_DIMENSION_ERROR], "cannot broadcast %R to %R", a->shape, to.get());
        throw PyError();
    }
    return View(a, 0, ndim, shape, strides);
}

Ref Reshape(Array* a, int ndim, const int64_t* shape) {
    if (ndim == a->d.ndim && std::equal(shape, shape + ndim, a->d.shape)) return NewRef(a);
    if (Product(ndim, shape) != Size(a)) {
        Ref to(IntTuple(ndim, shape));
        PyErr_Format(g.exceptions[HIPCX_DIMENSION_ERROR], "cannot reshape array of size %lld into shape %R", static_cast<long long>(Size(a)), to.get());
        throw PyError();
    }
    int64_t strides[HIPCX_MAX_NDIM];
    if (NoCopyReshape(a->d, ndim, shape, strides)) return View(a, 0, ndim, shape, strides);
    Ref c = CopyOf(a, a->d.dtype);
    ContiguousStrides(ndim, shape, ItemSize(a->d.dtype), strides);
    return View(c.arr(), 0, ndim, shape, strides);
}

namespace {
PyObject* ArrayNew(PyTypeObject* type, PyObject* args, PyObject* kwargs) {
    HOST_TRY;
    PyObject *buf, *offset, *shape, *strides, *dtype;
    static const char* kw[] = {"buf", "offset", "shape", "strides", "dtype", nullptr};
    if (!PyArg_ParseTupleAndKeywords(args, kwargs, "OOOOO", const_cast<char**>(kw), &buf, &offset, &shape, &strides, &dtype)) return nullptr;
    int64_t sh[HIPCX_MAX_NDIM], st[HIPCX_MAX_NDIM];
    int nd = ToShape(shape, sh);
    if (ToShape(strides, st) != nd) Raise(HIPCX_DIMENSION_ERROR, "shape and strides differ in length");
    char* base;
    if (Py_IS_TYPE(buf, &BufferType)) {
        base = static_cast<char*>(reinterpret_cast<Buffer*>(buf)->ptr);
    } else {
        Ref p(PyObject_CallMethod(buf, "data_ptr", nullptr));
        if (!p) throw PyError();
        base = static_cast<char*>(PyLong_AsVoidPtr(p.get()));
        if (base == nullptr && PyErr_Occurred()) throw PyError();
    }
    const int64_t off = ToInt(offset);
    return MakeArray(type, buf, off, base + off, nd, sh, st, DtypeCode(dtype)).release();
    HOST_CATCH(nullptr);
}

int ArrayInit(PyObject*, PyObject*, PyObject*) { return 0; }  // everything is done in ArrayNew

void ArrayDealloc(PyObject* self) {
    Array* a = reinterpret_cast<Array*>(self);
    Py_XDECREF(a->buf);
    Py_XDECREF(a->dtype);
    Py_XDECREF(a->shape);
    Py_XDECREF(a->strides);
    Py_XDECREF(a->cdesc);
    Py_TYPE(self)->tp_free(self);  // (a Python subclass's own deallocator releases its type)
}

Array* Self(PyObject* o) { return reinterpret_cast<Array*>(o); }

PyObject* Incref(PyObject* o) {
    Py_INCREF(o);
    return o;
}
PyObject* GetBuf(PyObject* o, void*) { return Incref(Self(o)->buf); }
PyObject* GetDtype(PyObject* o, void*) { return Incref(Self(o)->dtype); }
PyObject* GetShape(PyObject* o, void*) { return Incref(Self(o)->shape); }
PyObject* GetStrides(PyObject* o, void*) {
    HOST_TRY;
    Array* a = Self(o);
    if (a->strides == nullptr) a->strides = IntTuple(a->d.ndim, a->d.strides);
    return Incref(a->strides);
    HOST_CATCH(nullptr);
}
PyObject* GetOffset(PyObject* o, void*) { return PyLong_FromLongLong(Self(o)->offset); }
PyObject* GetPtr(PyObject* o, void*) { return PyLong_FromVoidPtr(Self(o)->d.data); }
PyObject* GetCDesc(PyObject* o, void*) { return Incref(Self(o)->cdesc != nullptr ? Self(o)->cdesc : Py_None); }
PyObject* GetNdim(PyObject* o, void*) { return PyLong_FromLong(Self(o)->d.ndim); }
PyObject* GetSize(PyObject* o, void*) { return PyLong_FromLongLong(Size(Self(o))); }
PyObject* GetItemSize(PyObject* o, void*) { return PyLong_FromLong(ItemSize(Self(o)->d.dtype)); }
PyObject* GetNBytes(PyObject* o, void*) { return PyLong_FromLongLong(Size(Self(o)) * ItemSize(Self(o)->d.dtype)); }
PyObject* GetIsContiguous(PyObject* o, void*) { return PyBool_FromLong(IsContiguous(Self(o)->d)); }

Ref Transposed(Array* a, const int* axes) {
    int64_t sh[HIPCX_MAX_NDIM], st[HIPCX_MAX_NDIM];
    for (int i = 0; i < a->d.ndim; ++i) {
        int ax = axes != nullptr ? axes[i] : a->d.ndim - 1 - i;
        sh[i] = a->d.shape[ax];
        st[i] = a->d.strides[ax];
    }
    return View(a, 0, a->d.ndim, sh, st);
}
PyObject* GetT(PyObject* o, void*) {
    HOST_TRY;
    return Transposed(Self(o), nullptr).release();
    HOST_CATCH(nullptr);
}

PyObject* ArrayDesc(PyObject* o, PyObject*) {
    Array* a = Self(o);
    if (a->cdesc == nullptr) {
        PyObject* addr = PyLong_FromVoidPtr(&a->d);
        if (addr == nullptr) return nullptr;
        a->cdesc = PyObject_CallOneArg(g.make_cdesc, addr);
        Py_DECREF(addr);
        if (a->cdesc == nullptr) return nullptr;
    }
    return PyObject_CallOneArg(g.byref, a->cdesc);
}

PyObject* ArrayTranspose(PyObject* o, PyObject* args) {
    HOST_TRY;
    Array* a = Self(o);
    PyObject* axes = args;
    if (PyTuple_GET_SIZE(args) == 1) {
        PyObject* only = PyTuple_GET_ITEM(args, 0);
        if (only == Py_None || PyTuple_Check(only) || PyList_Check(only)) axes = only;
    }
    if (axes == Py_None) return Transposed(a, nullptr).release();
    int64_t given[HIPCX_MAX_NDIM];
    int n = ToShape(axes, given);
    if (n == 0) return Transposed(a, nullptr).release();
    int ax[HIPCX_MAX_NDIM];
    unsigned seen = 0;
    for (int i = 0; i < n; ++i) {
        ax[i] = NormalizeAxis(given[i], a->d.ndim);
        seen |= 1u << ax[i];
    }
    if (n != a->d.ndim || seen != (1u << n) - 1) {
        PyErr_Format(g.exceptions[HIPCX_DIMENSION_ERROR], "axes do not match the array: %R", axes);
        throw PyError();
    }
    return Transposed(a, ax).release();
    HOST_CATCH(nullptr);
}

PyObject* ArrayBroadcastTo(PyObject* o, PyObject* shape) {
    HOST_TRY;
    int64_t sh[HIPCX_MAX_NDIM];
    int nd = ToShape(shape, sh);
    return BroadcastTo(Self(o), nd, sh).release();
    HOST_CATCH(nullptr);
}

PyObject* ArrayReshape(PyObject* o, PyObject* args) {
    HOST_TRY;
    Array* a = Self(o);
    PyObject* shape = args;
    if (PyTuple_GET_SIZE(args) == 1) {
        PyObject* only = PyTuple_GET_ITEM(args, 0);
        if (PyTuple_Check(only) || PyList_Check(only)) shape = only;
    }
    int64_t sh[HIPCX_MAX_NDIM];
    int nd = ToShape(shape, sh);
    int unknown = -1;
    int64_t rest = 1;
    for (int i = 0; i < nd; ++i) {
        if (sh[i] == -1) {
            if (unknown >= 0) Raise(HIPCX_DIMENSION_ERROR, "can only specify one unknown dimension");
            unknown = i;
        } else {
            rest *= sh[i];
        }
    }
    if (unknown >= 0) {
        if (rest == 0 || Size(a) % rest != 0) {
            PyErr_Format(g.exceptions[HIPCX_DIMENSION_ERROR], "cannot reshape array of size %lld into shape %R", static_cast<long long>(Size(a)), shape);
            throw PyError();
        }
        sh[unknown] = Size(a) / rest;
    }
    return Reshape(a, nd, sh).release();
    HOST_CATCH(nullptr);
}

PyObject* ArraySqueeze(PyObject* o, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
    HOST_TRY;
    HOST_ARGS("squeeze", 0, "axis");
    Array* a = Self(o);
    unsigned drop = 0;
    if (!Given(arg[0])) {
        for (int i = 0; i < a->d.ndim; ++i) {
            if (a->d.shape[i] == 1) drop |= 1u << i;
        }
    } else {
        int64_t axes[HIPCX_MAX_NDIM];
        int n = ToShape(arg[0], axes);
        for (int i = 0; i < n; ++i) {
            int ax = NormalizeAxis(axes[i], a->d.ndim);
            if (a->d.shape[ax] != 1) Raise(HIPCX_DIMENSION_ERROR, "cannot squeeze an axis of extent %lld", static_cast<long long>(a->d.shape[ax]));
            drop |= 1u << ax;
        }
    }
    int64_t sh[HIPCX_MAX_NDIM], st[HIPCX_MAX_NDIM];
    int nd = 0;
    for (int i = 0; i < a->d.ndim; ++i) {
        if (drop >> i & 1) continue;
        sh[nd] = a->d.shape[i];
        st[nd++] = a->d.strides[i];
    }
    return View(a, 0, nd, sh, st).release();
    HOST_CATCH(nullptr);
}

// Basic indexing only (ints, slices, None, Ellipsis): Array::At (CX/routines/indexing.cc).
PyObject* ArrayGetItem(PyObject* o, PyObject* key) {
    HOST_TRY;
    Array* a = Self(o);
    PyObject* one[1] = {key};
    PyObject** keys = one;
    Py_ssize_t n_keys = 1;
    if (PyTuple_Check(key)) {
        n_keys = PyTuple_GET_SIZE(key);
        keys = &PyTuple_GET_ITEM(key, 0);
    }
    int real = 0, ellipses = 0;
    for (Py_ssize_t i = 0; i < n_keys; ++i) {
        if (keys[i] == Py_Ellipsis) {
            ++ellipses;
        } else if (keys[i] != Py_None) {
            ++real;
        }
    }
    if (real > a->d.ndim) Raise(HIPCX_DIMENSION_ERROR, "too many indices for array");
    if (ellipses > 1) Raise(HIPCX_DIMENSION_ERROR, "an index can only have a single ellipsis");
    if (a->d.ndim + n_keys - ellipses - real > HIPCX_MAX_NDIM) {
        Raise(HIPCX_DIMENSION_ERROR, "ndim %zd exceeds the maximum of %d", static_cast<Py_ssize_t>(a->d.ndim + n_keys - ellipses - real), HIPCX_MAX_NDIM);
    }
    int64_t sh[2 * HIPCX_MAX_NDIM], st[2 * HIPCX_MAX_NDIM];
    int nd = 0, axis = 0;
    int64_t offset = 0;
    auto whole = [&](int count) {
        for (int i = 0; i < count; ++i, ++axis) {
            sh[nd] = a->d.shape[axis];
            st[nd++] = a->d.strides[axis];
        }
    };
    for (Py_ssize_t i = 0; i < n_keys; ++i) {
        PyObject* k = keys[i];
        if (k == Py_None) {
            sh[nd] = 1;
            st[nd++] = 0;
        } else if (k == Py_Ellipsis) {
            whole(a->d.ndim - real);
        } else if (PySlice_Check(k)) {
            Py_ssize_t start, stop, step;
            if (PySlice_Unpack(k, &start, &stop, &step) < 0) throw PyError();
            Py_ssize_t n = PySlice_AdjustIndices(a->d.shape[axis], &start, &stop, step);
            if (n > 0) offset += start * a->d.strides[axis];
            sh[nd] = n;
            st[nd++] = a->d.strides[axis] * step;
            ++axis;
        } else {
            const int64_t dim = a->d.shape[axis];
            int64_t v = ToInt(k);
            if (v < -dim || v >= dim) {
                Raise(HIPCX_INDEX_ERROR, "index %lld is out of bounds for axis %d with size %lld", static_cast<long long>(v), axis, static_cast<long long>(dim));
            }
            offset += (v < 0 ? v + dim : v) * a->d.strides[axis];
            ++axis;
        }
    }
    whole(a->d.ndim - axis);
    return View(a, offset, nd, sh, st).release();
    HOST_CATCH(nullptr);
}

PyObject* ArrayItem(PyObject* o, Py_ssize_t i) {  // iteration
    PyObject* key = PyLong_FromSsize_t(i);
    PyObject* item = key != nullptr ? ArrayGetItem(o, key) : nullptr;
    Py_XDECREF(key);
    return item;
}

Py_ssize_t ArrayLen(PyObject* o) {
    if (Self(o)->d.ndim == 0) {
        PyErr_SetString(PyExc_TypeError, "len() of unsized object");
        return -1;
    }
    return static_cast<Py_ssize_t>(Self(o)->d.shape[0]);
}

PyObject* ArrayCopy(PyObject* o, PyObject*) {
    HOST_TRY;
    return CopyOf(Self(o), Self(o)->d.dtype).release();
    HOST_CATCH(nullptr);
}

PyObject* ArrayAsType(PyObject* o, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
    HOST_TRY;
    HOST_ARGS("astype", 1, "dtype", "copy");
    Array* a = Self(o);
    int code = DtypeCode(arg[0]);
    int copy = arg[1] == nullptr ? 1 : PyObject_IsTrue(arg[1]);
    if (copy < 0) throw PyError();
    return (copy ? CopyOf(a, code) : Cast(a, code)).release();
    HOST_CATCH(nullptr);
}

PyObject* ArrayAsContiguous(PyObject* o, PyObject*) {
    HOST_TRY;
    return Contiguous(Self(o)).release();
    HOST_CATCH(nullptr);
}

PyObject* ArrayFill(PyObject* o, PyObject* value) {
    HOST_TRY;
    hipcx_scalar s = ToScalar(value);
    void* stream = Stream();
    Call([&] { return hipcx_fill(&Self(o)->d, s, stream); });
    Py_RETURN_NONE;
    HOST_CATCH(nullptr);
}

PyObject* ArrayEmpty(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
    HOST_TRY;
    HOST_ARGS("empty", 2, "shape", "dtype", "strides");
    int64_t sh[HIPCX_MAX_NDIM], st[HIPCX_MAX_NDIM];
    int nd = ToShape(arg[0], sh);
    int code = DtypeCode(arg[1]);
    if (!Given(arg[2])) return Empty(nd, sh, code).release();
    if (ToShape(arg[2], st) != nd) Raise(HIPCX_DIMENSION_ERROR, "shape and strides differ in length");
    int64_t bytes = ItemSize(code);
    for (int i = 0; i < nd; ++i) bytes = sh[i] == 0 || bytes == 0 ? 0 : bytes + (sh[i] - 1) * std::abs(st[i]);
    return EmptyStrided(nd, sh, st, bytes, code).release();
    HOST_CATCH(nullptr);
}

PyCFunction Fast(PyObject* (*f)(PyObject*, PyObject* const*, Py_ssize_t, PyObject*)) {
    return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f));
}

PyMethodDef kArrayMethods[] = {
        {"desc", ArrayDesc, METH_NOARGS, "The hipcx_array descriptor of this view as a ctypes reference (built once; views are immutable)."},
        {"transpose", ArrayTranspose, METH_VARARGS, nullptr},
        {"broadcast_to", ArrayBroadcastTo, METH_O, "Stride-0 broadcast view (CX/routines/manipulation.cc:316-358)."},
        {"reshape", ArrayReshape, METH_VARARGS, "View when the strides allow it, else a contiguous copy (CX/routines/manipulation.cc:153-258)."},
        {"squeeze", Fast(ArraySqueeze), METH_FASTCALL | METH_KEYWORDS, nullptr},
        {"copy", ArrayCopy, METH_NOARGS, "C-contiguous copy (CopyKernel)."},
        {"astype", Fast(ArrayAsType), METH_FASTCALL | METH_KEYWORDS,
         "Array::AsType (CX/array.cc): a new C-contiguous array unless copy=False and the dtype matches."},
        {"as_contiguous", ArrayAsContiguous, METH_NOARGS, nullptr},
        {"fill", ArrayFill, METH_O, nullptr},
        {"empty", Fast(ArrayEmpty), METH_FASTCALL | METH_KEYWORDS | METH_STATIC, "An uninitialised array (C-contiguous unless strides are given)."},
        {nullptr, nullptr, 0, nullptr}};

PyGetSetDef kArrayGetSet[] = {
        {"_buf", GetBuf, nullptr, nullptr, nullptr},
        {"_offset", GetOffset, nullptr, nullptr, nullptr},
        {"_ptr", GetPtr, nullptr, nullptr, nullptr},
        {"_desc", GetCDesc, nullptr, nullptr, nullptr},
        {"data_ptr", GetPtr, nullptr, nullptr, nullptr},
        {"dtype", GetDtype, nullptr, nullptr, nullptr},
        {"shape", GetShape, nullptr, nullptr, nullptr},
        {"strides", GetStrides, nullptr, nullptr, nullptr},
        {"ndim", GetNdim, nullptr, nullptr, nullptr},
        {"size", GetSize, nullptr, nullptr, nullptr},
        {"itemsize", GetItemSize, nullptr, nullptr, nullptr},
        {"nbytes", GetNBytes, nullptr, nullptr, nullptr},
        {"is_contiguous", GetIsContiguous, nullptr, "C-contiguity ignoring unit axes (CX/shape.cc:15-32).", nullptr},
        {"T", GetT, nullptr, nullptr, nullptr},
        {nullptr, nullptr, nullptr, nullptr, nullptr}};

PyMappingMethods kArrayMapping = {ArrayLen, ArrayGetItem, nullptr};
PySequenceMethods kArraySequence = {};
}  // namespace

PyTypeObject ArrayType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// ---------------------------------------------------------------------------------------------
// argument parsing
// ---------------------------------------------------------------------------------------------
void Parse(const char* fn, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames, PyObject* const* names, int n_names, int n_required,
           PyObject** out) {
    if (nargs > n_names) {
        PyErr_Format(PyExc_TypeError, "%s() takes at most %d arguments (%zd given)", fn, n_names, nargs);
        throw PyError();
    }
    for (Py_ssize_t i = 0; i < nargs; ++i) out[i] = args[i];
    const Py_ssize_t n_kw = kwnames != nullptr ? PyTuple_GET_SIZE(kwnames) : 0;
    for (Py_ssize_t k = 0; k < n_kw; ++k) {
        PyObject* name = PyTuple_GET_ITEM(kwnames, k);
        int at = 0;
        while (at < n_names && names[at] != name && PyUnicode_Compare(names[at], name) != 0) ++at;
        if (at == n_names || out[at] != nullptr) {
            PyErr_Format(PyExc_TypeError, at == n_names ? "%s() got an unexpected keyword argument '%U'" : "%s() got multiple values for argument '%U'", fn, name);
            throw PyError();
        }
        out[at] = args[nargs + k];
    }
    for (int i = 0; i < n_required; ++i) {
        if (out[i] == nullptr) {
            PyErr_Format(PyExc_TypeError, "%s() missing required argument '%U'", fn, names[i]);
            throw PyError();
        }
    }
}

// ---------------------------------------------------------------------------------------------
// module
// ---------------------------------------------------------------------------------------------
namespace {
PyObject* Setup(PyObject*, PyObject* config) {
    struct {
        const char* name;
        PyObject** slot;
    } objects[] = {{"ndarray", &g.ndarray},
                   {"np_dtype", &g.np_dtype},
                   {"np_bool", &g.np_bool},
                   {"np_integer", &g.np_integer},
                   {"np_floating", &g.np_floating},
                   {"require_device", &g.require_device},
                   {"raw_stream", &g.raw_stream},
                   {"get_device", &g.get_device},
                   {"make_cdesc", &g.make_cdesc},
                   {"byref", &g.byref},
                   {"flags", &g.flags}};
    for (auto& o : objects) {
        PyObject* v = PyDict_GetItemString(config, o.name);
        if (v == nullptr) continue;
        Py_INCREF(v);
        Py_XSETREF(*o.slot, v);
    }
    if (PyObject* dtypes = PyDict_GetItemString(config, "dtypes")) {
        for (int i = 1; i < 10; ++i) {
            PyObject* v = PyList_GetItem(dtypes, i);
            if (v == nullptr) return nullptr;
            Py_INCREF(v);
            Py_XSETREF(g.dtypes[i], v);
        }
    }
    if (PyObject* exceptions = PyDict_GetItemString(config, "exceptions")) {
        for (int i = 1; i < 9; ++i) {
            PyObject* v = PyList_GetItem(exceptions, i);
            if (v == nullptr) return nullptr;
            Py_INCREF(v);
            Py_XSETREF(g.exceptions[i], v);
        }
    }
    Py_RETURN_NONE;
}

PyObject* CurrentStream(PyObject*, PyObject*) {
    HOST_TRY;
    return PyLong_FromVoidPtr(Stream());
    HOST_CATCH(nullptr);
}

PyObject* NoCopyReshapeStrides(PyObject*, PyObject* args) {
    HOST_TRY;
    PyObject *old_shape, *old_strides, *new_shape;
    int itemsize;
    if (!PyArg_ParseTuple(args, "OOOi", &old_shape, &old_strides, &new_shape, &itemsize)) return nullptr;
    hipcx_array d;
    std::memset(&d, 0, sizeof(d));
    d.ndim = ToShape(old_shape, d.shape);
    ToShape(old_strides, d.strides);
    d.dtype = itemsize == 1 ? HIPCX_UINT8 : itemsize == 2 ? HIPCX_INT16 : itemsize == 4 ? HIPCX_INT32 : HIPCX_INT64;
    int64_t sh[HIPCX_MAX_NDIM], st[HIPCX_MAX_NDIM];
    int nd = ToShape(new_shape, sh);
    if (!NoCopyReshape(d, nd, sh, st)) Py_RETURN_NONE;
    return IntTuple(nd, st);
    HOST_CATCH(nullptr);
}

PyObject* PyPromote(PyObject*, PyObject* args) {
    HOST_TRY;
    PyObject *a, *b;
    if (!PyArg_ParseTuple(args, "OO", &a, &b)) return nullptr;
    return Incref(g.dtypes[Promote(DtypeCode(a), DtypeCode(b))]);
    HOST_CATCH(nullptr);
}

PyObject* PyResultType(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HOST_TRY;
    int arr = 0, sc = 0;
    for (Py_ssize_t i = 0; i < nargs; ++i) {
        int c = IsArray(args[i]) ? Self(args[i])->d.dtype : ScalarDtype(args[i]);
        int& into = IsArray(args[i]) ? arr : sc;
        into = into == 0 ? c : Promote(into, c);
    }
    auto category = [](int code) { return Kind(code) == 0 ? 0 : Kind(code) == 3 ? 2 : 1; };
    int code = arr == 0 ? sc : sc != 0 && category(sc) > category(arr) ? sc : arr;
    return Incref(code != 0 ? g.dtypes[code] : Py_None);
    HOST_CATCH(nullptr);
}

PyMethodDef kModuleMethods[] = {
        {"setup", Setup, METH_O, nullptr},
        {"current_stream", CurrentStream, METH_NOARGS, nullptr},
        {"nocopy_reshape_strides", NoCopyReshapeStrides, METH_VARARGS, nullptr},
        {"promote_types", PyPromote, METH_VARARGS, "PromoteTypes (CX/dtype.cc:12-60)."},
        {"result_type", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(PyResultType)), METH_FASTCALL,
         "ResultType over arrays and Python scalars: scalars only matter if of a higher category (CX/routines/type_util.cc:11-46)."},
        {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "chainer_amd._host", "Native host path of chainer_amd.", -1, kModuleMethods, nullptr, nullptr, nullptr, nullptr};
}  // namespace
}  // namespace host

PyMODINIT_FUNC PyInit__host(void) {
    using namespace host;
    BufferType.tp_name = "chainer_amd._host.DeviceBuffer";
    BufferType.tp_basicsize = sizeof(Buffer);
    BufferType.tp_flags = Py_TPFLAGS_DEFAULT;
    BufferType.tp_new = BufferNew;
    BufferType.tp_dealloc = BufferDealloc;
    BufferType.tp_methods = kBufferMethods;
    BufferType.tp_getset = kBufferGetSet;
    BufferType.tp_members = kBufferMembers;
    BufferType.tp_weaklistoffset = offsetof(Buffer, weakrefs);
    BufferType.tp_doc =
            "One allocation of the backend's memory pool (Device::Allocate, CX/device.h:33); returned to the pool when the last array\n"
            "that refers to it goes away, like the deleter of the reference's ``shared_ptr<void>``.";
    ArrayType.tp_name = "chainer_amd._host.ArrayBase";
    ArrayType.tp_basicsize = sizeof(Array);
    ArrayType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE;
    ArrayType.tp_new = ArrayNew;
    ArrayType.tp_init = ArrayInit;
    ArrayType.tp_dealloc = ArrayDealloc;
    ArrayType.tp_methods = kArrayMethods;
    ArrayType.tp_getset = kArrayGetSet;
    kArraySequence.sq_length = ArrayLen;
    kArraySequence.sq_item = ArrayItem;
    ArrayType.tp_as_mapping = &kArrayMapping;
    ArrayType.tp_as_sequence = &kArraySequence;
    if (PyType_Ready(&BufferType) < 0 || PyType_Ready(&ArrayType) < 0) return nullptr;
    PyObject* m = PyModule_Create(&kModule);
    if (m == nullptr) return nullptr;
    if (PyModule_AddFunctions(m, kRoutines) < 0) return nullptr;
    Py_INCREF(&BufferType);
    Py_INCREF(&ArrayType);
    if (PyModule_AddObject(m, "DeviceBuffer", reinterpret_cast<PyObject*>(&BufferType)) < 0 ||
        PyModule_AddObject(m, "ArrayBase", reinterpret_cast<PyObject*>(&ArrayType)) < 0) {
        return nullptr;
    }
    return m;
}
