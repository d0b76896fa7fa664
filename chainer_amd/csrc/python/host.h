// Array and buffer objects of the Python package, shared by the translation units of the extension module chainer_amd._host.
//
// A call of a routine on small arrays is bounded by the host: checks, dtype promotion, the output's allocation, descriptors and
// the stream look-up took 12-25 us per call as interpreted code around ctypes, against the 2-3 us of a kernel launch.  All of
// that work is therefore done here, with the array's hipcx_array descriptor built once inside the object.
#pragma once

#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>
#include <cstring>
#include <exception>
#include <initializer_list>
#include <new>

#include "hipcx.h"

namespace host {

struct Buffer {  // one block of the device memory pool
    PyObject_HEAD
    void* ptr;
    size_t nbytes;
    PyObject* weakrefs;
};

struct Array {  // strided view of device memory; immutable
    PyObject_HEAD
    PyObject* buf;      // owner of the memory: a Buffer, or any object with data_ptr()
    PyObject* dtype;    // numpy dtype object
    PyObject* shape;    // tuple
    PyObject* strides;  // tuple, or null until somebody asks for it
    PyObject* cdesc;    // ctypes copy of `d`, or null until desc() is called
    int64_t offset;
    hipcx_array d;
};

// Objects handed over by the Python side at import.
struct State {
    PyObject* ndarray = nullptr;         // class of the arrays made here (a subclass of ArrayBase)
    PyObject* dtypes[10] = {};           // numpy dtype objects by hipcx dtype code
    PyObject* exceptions[9] = {};        // by hipcx_status
    PyObject* np_dtype = nullptr;        // numpy.dtype
    PyObject* np_bool = nullptr;         // numpy.bool_
    PyObject* np_integer = nullptr;
    PyObject* np_floating = nullptr;
    PyObject* require_device = nullptr;  // raises BackendError without a device; initialises the runtime
    PyObject* raw_stream = nullptr;      // device index -> raw handle of the current stream
    PyObject* get_device = nullptr;      // current device index
    PyObject* make_cdesc = nullptr;      // address of a hipcx_array -> ctypes copy
    PyObject* byref = nullptr;           // ctypes.byref
    PyObject* flags = nullptr;           // dict of chainer_amd.routines: the opt-in switches
    bool ready = false;                  // require_device has succeeded
};
extern State g;
extern PyTypeObject BufferType;
extern PyTypeObject ArrayType;

// Owned reference, released at the end of the scope.
class Ref {
public:
    Ref() = default;
    explicit Ref(void* p) : p_(static_cast<PyObject*>(p)) {}
    Ref(const Ref&) = delete;
    Ref& operator=(const Ref&) = delete;
    Ref(Ref&& o) noexcept : p_(o.p_) { o.p_ = nullptr; }
    Ref& operator=(Ref&& o) noexcept {
        if (this != &o) {
            Py_XDECREF(p_);
            p_ = o.p_;
            o.p_ = nullptr;
        }
        return *this;
    }
    ~Ref() { Py_XDECREF(p_); }
    explicit operator bool() const { return p_ != nullptr; }
    PyObject* get() const { return p_; }
    Array* arr() const { return reinterpret_cast<Array*>(p_); }
    const hipcx_array* d() const { return p_ != nullptr ? &reinterpret_cast<Array*>(p_)->d : nullptr; }
    PyObject* release() {
        PyObject* p = p_;
        p_ = nullptr;
        return p;
    }

private:
    PyObject* p_ = nullptr;
};

// Thrown when a Python exception is set; every function called by the interpreter ends in CATCH.  Nothing of C++ leaves one: the
// standard containers' exceptions become Python's.
struct PyError {};
#define HOST_TRY try {
#define HOST_CATCH(value)                                \
    }                                                    \
    catch (const host::PyError&) {                       \
        return value;                                    \
    }                                                    \
    catch (const std::bad_alloc&) {                      \
        PyErr_NoMemory();                                \
        return value;                                    \
    }                                                    \
    catch (const std::exception& e) {                    \
        PyErr_SetString(PyExc_RuntimeError, e.what());   \
        return value;                                    \
    }

[[noreturn]] void Raise(int status, const char* format, ...);
void Check(int status);  // raises what hipcx_last_error describes

// ---- dtypes ----
inline int ItemSize(int code) {
    static const int8_t size[10] = {0, 1, 1, 2, 4, 8, 1, 2, 4, 8};
    return size[code];
}
inline int Kind(int code) {  // 0 bool, 1 signed, 2 unsigned, 3 float
    static const int8_t kind[10] = {0, 0, 1, 1, 1, 1, 2, 3, 3, 3};
    return kind[code];
}
inline bool IsFloat(int code) { return code >= HIPCX_FLOAT16; }
inline int MathDtype(int code) { return IsFloat(code) ? code : HIPCX_FLOAT32; }
int DtypeCode(PyObject* dtype);  // anything numpy.dtype() takes
int Promote(int a, int b);
bool IsScalar(PyObject* x);
hipcx_scalar ToScalar(PyObject* x);
int ScalarDtype(PyObject* x);  // ScalarDefaultDtype: bool, int32 or float32
inline bool IsArray(PyObject* x) { return PyObject_TypeCheck(x, &ArrayType); }
Array* AsArray(PyObject* x, const char* what);  // borrowed
// ResultType over arrays and scalars: scalars only matter when of a higher category.
int ResultType(std::initializer_list<PyObject*> args);

// ---- memory, arrays ----
void* Stream();
Ref NewBuffer(size_t nbytes);
Ref NewArray(PyObject* buf, int64_t offset, char* data, int ndim, const int64_t* shape, const int64_t* strides, int code);
Ref Empty(int ndim, const int64_t* shape, int code);                                 // C-contiguous
Ref EmptyStrided(int ndim, const int64_t* shape, const int64_t* strides, int64_t bytes, int code);
inline Ref EmptyLike(const Array* a, int code) { return Empty(a->d.ndim, a->d.shape, code); }
Ref NewRef(Array* a);
Ref View(Array* a, int64_t offset_delta, int ndim, const int64_t* shape, const int64_t* strides);
Ref Cast(Array* a, int code);            // the array itself when it has the dtype, else a converted copy
Ref CopyOf(Array* a, int code);
Ref Contiguous(Array* a);
Ref BroadcastTo(Array* a, int ndim, const int64_t* shape);
Ref Reshape(Array* a, int ndim, const int64_t* shape);  // a view when the strides allow it, else of a contiguous copy
bool IsContiguous(const hipcx_array& d);
void ContiguousStrides(int ndim, const int64_t* shape, int itemsize, int64_t* strides);
// Dense strides in the axis order of the array's memory.
void DenseStridesLike(const Array* a, int itemsize, int64_t* strides);
bool NoCopyReshape(const hipcx_array& d, int ndim, const int64_t* shape, int64_t* strides);
inline int64_t Product(int n, const int64_t* v) {
    int64_t p = 1;
    for (int i = 0; i < n; ++i) p *= v[i];
    return p;
}
inline int64_t Size(const Array* a) { return Product(a->d.ndim, a->d.shape); }
int NormalizeAxis(int64_t axis, int ndim);
int64_t ToInt(PyObject* x);
int ToShape(PyObject* x, int64_t* shape);  // an int or a sequence of ints; returns the number of axes
bool Flag(PyObject* name);                 // a switch of chainer_amd.routines

// Scratch memory of one call.
struct Workspace {
    Ref buffer;
    void* ptr = nullptr;
    size_t bytes = 0;
    explicit Workspace(size_t n) : bytes(n) {
        if (n != 0) {
            buffer = NewBuffer(n);
            ptr = reinterpret_cast<Buffer*>(buffer.get())->ptr;
        }
    }
};

// Runs a library call without the interpreter lock and raises its error.
template <typename F>
inline void Call(F&& f) {
    int status;
    Py_BEGIN_ALLOW_THREADS;
    status = f();
    Py_END_ALLOW_THREADS;
    if (status != 0) Check(status);
}

// Positional and keyword arguments of a METH_FASTCALL | METH_KEYWORDS function into out[], by position in `names`.
void Parse(const char* fn, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames, PyObject* const* names, int n_names, int n_required,
           PyObject** out);
struct Names {  // interned argument names
    static constexpr int kMax = 12;
    PyObject* v[kMax];
    int n = 0;
    Names(std::initializer_list<const char*> names) {
        for (const char* s : names) v[n++] = PyUnicode_InternFromString(s);
    }
};
#define HOST_ARGS(fn, required, ...)              \
    static const host::Names names_{__VA_ARGS__}; \
    PyObject* arg[host::Names::kMax] = {};        \
    host::Parse(fn, args, nargs, kwnames, names_.v, names_.n, required, arg)
#define HOST_FN(name) PyObject* name(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames)
inline bool Given(PyObject* x) { return x != nullptr && x != Py_None; }

extern PyMethodDef kRoutines[];  // routines.cc

}  // namespace host
