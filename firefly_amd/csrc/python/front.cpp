// front.cpp - the Python front end's calls into the C ABI (include/ffkv.h) as a CPython extension.
//
// A decode step of a small model is a handful of calls of a few microseconds of GPU work each, issued from Python
// once per layer.  Through ctypes a call cost 6 to 8 us before anything was launched: about 20 argument conversions,
// and a Python call for every pointer, shape and dtype.  Here the wrappers of firefly_amd/__init__.py hand their
// tensors over as they are, and shapes, dtypes, pointers and the current stream are read natively: 1 to 2 us.  The fused
// append + decode of 4 rows of up to 255 tokens (16/8 heads), one launch: 10.1 -> 6.9 us in a row, where the GPU now sets
// the pace, and 24.2 -> 19.1 us for a call that is waited for.
// The library is the one firefly_amd loaded: bind() gets the addresses of its functions, so nothing is linked here.
// Only CPython's own API is used; tensors are read through their attributes (shape, dtype, data_ptr(), nbytes).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>
#include <vector>

#include "ffkv.h"

namespace
{

struct Functions
{
    decltype(&ffkv_append)                     append;
    decltype(&ffkv_paged_decode)               decode;
    decltype(&ffkv_append_paged_decode)        append_decode;
    decltype(&ffkv_paged_decode_shared_prefix) decode_shared;
    decltype(&ffkv_paged_decode_noalloc)       decode_noalloc;
    decltype(&ffkv_prefill_workspace_bytes)    prefill_bytes;
    decltype(&ffkv_paged_prefill_ws)           prefill;
    decltype(&ffkv_rope)                       rope;
    decltype(&ffkv_rope_append)                rope_append;
};
Functions fn{};

PyObject *s_shape, *s_dtype, *s_data_ptr, *s_nbytes, *s_cuda_stream;
struct DtypeCode
{
    PyObject* dtype;
    int       code;
};
std::vector<DtypeCode> dtypes;
PyObject *              get_device, *raw_stream, *first_stream;  // set by bind()
bool                    stream_ready = false;

// Reads a call's arguments one after the other; after the first failure (a Python exception is set) the rest read as
// zero.
struct Reader
{
    PyObject* const* a;
    bool             ok = true;

    void* ptr(PyObject* t)
    {
        if (!ok || t == Py_None) return nullptr;
        PyObject* p = PyObject_CallMethodNoArgs(t, s_data_ptr);
        void*     v = p ? PyLong_AsVoidPtr(p) : nullptr;
        Py_XDECREF(p);
        if (PyErr_Occurred()) ok = false;
        return v;
    }
    template <typename T>
    T* ptr(PyObject* t)
    {
        return static_cast<T*>(ptr(t));
    }
    // The sizes of t (a tuple), at least `least` and, when exactly is set, as many.
    PyObject* shape(PyObject* t, Py_ssize_t least, bool exactly)
    {
        if (!ok) return nullptr;
        PyObject* s = PyObject_GetAttr(t, s_shape);
        if (s != nullptr && PyTuple_Check(s))
        {
            const Py_ssize_t n = PyTuple_GET_SIZE(s);
            if (n >= least && (!exactly || n == least)) return s;
            if (exactly)
                PyErr_Format(PyExc_ValueError, "%s values to unpack (expected %zd, got %zd)",
                             n > least ? "too many" : "not enough", least, n);
            else
                PyErr_SetString(PyExc_IndexError, "tuple index out of range");
        }
        else if (s != nullptr)
            PyErr_SetString(PyExc_TypeError, "shape is not a tuple");
        Py_XDECREF(s);
        ok = false;
        return nullptr;
    }
    int item(PyObject* shape, Py_ssize_t i)
    {
        return ok ? static_cast<int>(PyLong_AsLongLong(PyTuple_GET_ITEM(shape, i))) : 0;
    }
    void dims4(PyObject* t, int& d0, int& d1, int& d2, int& d3)
    {
        PyObject* s = shape(t, 4, true);
        d0 = item(s, 0), d1 = item(s, 1), d2 = item(s, 2), d3 = item(s, 3);
        Py_XDECREF(s);
    }
    int dim(PyObject* t, Py_ssize_t i)  // negative: from the end
    {
        PyObject* s = shape(t, i < 0 ? -i : i + 1, false);
        const int v = s ? item(s, i < 0 ? PyTuple_GET_SIZE(s) + i : i) : 0;
        Py_XDECREF(s);
        return v;
    }
    int dtype(PyObject* t)
    {
        if (!ok) return 0;
        PyObject* d = PyObject_GetAttr(t, s_dtype);
        if (d != nullptr)
        {
            for (const DtypeCode& c : dtypes)
                if (c.dtype == d)
                {
                    Py_DECREF(d);
                    return c.code;
                }
            PyErr_Format(PyExc_TypeError, "unsupported dtype %S", d);
            Py_DECREF(d);
        }
        ok = false;
        return 0;
    }
    int integer(PyObject* o)  // a Python int: nothing that merely converts to one (a device tensor would synchronize)
    {
        if (!ok) return 0;
        if (!PyLong_Check(o))
        {
            PyErr_Format(PyExc_TypeError, "an int is required, not %.100s", Py_TYPE(o)->tp_name);
            ok = false;
            return 0;
        }
        const long long v = PyLong_AsLongLong(o);
        if (v == -1 && PyErr_Occurred()) ok = false;
        return static_cast<int>(v);
    }
    int blocks(PyObject* num_blocks, PyObject* cache) { return num_blocks == Py_None ? dim(cache, 0) : integer(num_blocks); }
    float real(PyObject* o)  // whatever float() takes
    {
        if (!ok) return 0.0f;
        PyObject*    f = PyNumber_Float(o);
        const double v = f ? PyFloat_AS_DOUBLE(f) : 0.0;
        Py_XDECREF(f);
        if (f == nullptr) ok = false;
        return static_cast<float>(v);
    }
    size_t nbytes(PyObject* t)
    {
        if (!ok || t == Py_None) return 0;
        PyObject*    n = PyObject_GetAttr(t, s_nbytes);
        const size_t v = n ? PyLong_AsSize_t(n) : 0;
        Py_XDECREF(n);
        if (PyErr_Occurred()) ok = false;
        return v;
    }
    // A stream argument: None is torch's current stream, else an object with cuda_stream, or a raw handle.
    void* stream(PyObject* o)
    {
        if (!ok) return nullptr;
        PyObject* h = nullptr;
        if (o == Py_None && !stream_ready)
        {
            h = PyObject_CallNoArgs(first_stream);
            stream_ready = h != nullptr;
        }
        else if (o == Py_None)
        {
            PyObject* dev = PyObject_CallNoArgs(get_device);
            h = dev ? PyObject_CallOneArg(raw_stream, dev) : nullptr;
            Py_XDECREF(dev);
        }
        else
        {
            h = PyObject_GetAttr(o, s_cuda_stream);
            if (h == nullptr && PyErr_ExceptionMatches(PyExc_AttributeError))
            {
                PyErr_Clear();
                h = PyNumber_Long(o);
            }
        }
        void* v = h ? PyLong_AsVoidPtr(h) : nullptr;
        Py_XDECREF(h);
        if (PyErr_Occurred()) ok = false;
        return v;
    }
};

bool count(Py_ssize_t got, Py_ssize_t want)
{
    if (got == want) return true;
    PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, got);
    return false;
}

// The C call, without the interpreter lock (as ctypes made it).
template <typename F>
PyObject* finish(const Reader& r, F call)
{
    if (!r.ok) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = call();
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

// k, v, k_cache, v_cache, block_table, context_lens, k_scale, v_scale, num_blocks, stream
PyObject* append(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    if (!count(n, 10)) return nullptr;
    Reader r{a};
    int    B, S, Hkv, D;
    r.dims4(a[0], B, S, Hkv, D);
    const int  mb = r.dim(a[4], -1), N = r.blocks(a[8], a[2]), st = r.dtype(a[0]), ct = r.dtype(a[2]);
    void *     k = r.ptr(a[0]), *v = r.ptr(a[1]), *kc = r.ptr(a[2]), *vc = r.ptr(a[3]);
    auto *     bt = r.ptr<int32_t>(a[4]), *cx = r.ptr<int32_t>(a[5]);
    auto *     ks = r.ptr<float>(a[6]), *vs = r.ptr<float>(a[7]);
    void*      s = r.stream(a[9]);
    return finish(r, [&] { return fn.append(k, v, st, kc, vc, ct, ks, vs, bt, cx, B, S, Hkv, D, FFKV_BLOCK_SIZE, mb, N, s); });
}

// The tensors of a decode: q, out, k_cache, v_cache, k_scale, v_scale, block_table, context_lens at a[0 .. 7],
// max_context_len, scale, num_blocks at a[8 .. 10].
struct Decode
{
    int      B, Hq, D, Hkv, mb, N, qt, ct, mcl;
    float    scale;
    void *   q, *out, *kc, *vc;
    float *  ks, *vs;
    int32_t *bt, *cx;
    Decode(Reader& r, PyObject* const* a)
    {
        B = r.dim(a[0], 0), Hq = r.dim(a[0], -2), D = r.dim(a[0], -1), Hkv = r.dim(a[2], 2);
        mb = r.dim(a[6], -1), N = r.blocks(a[10], a[2]);
        q = r.ptr(a[0]), out = r.ptr(a[1]), qt = r.dtype(a[0]), kc = r.ptr(a[2]), vc = r.ptr(a[3]), ct = r.dtype(a[2]);
        ks = r.ptr<float>(a[4]), vs = r.ptr<float>(a[5]), bt = r.ptr<int32_t>(a[6]), cx = r.ptr<int32_t>(a[7]);
        mcl = r.integer(a[8]), scale = r.real(a[9]);
    }
};

// decode's 11, workspace, stream
PyObject* decode(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    if (!count(n, 13)) return nullptr;
    Reader       r{a};
    Decode       d(r, a);
    void*        ws = r.ptr(a[11]);
    const size_t wb = r.nbytes(a[11]);
    void*        s = r.stream(a[12]);
    return finish(r, [&] {
        return fn.decode(d.q, d.out, d.qt, d.kc, d.vc, d.ct, d.ks, d.vs, d.bt, d.cx, d.B, d.Hq, d.Hkv, d.D,
                         FFKV_BLOCK_SIZE, d.mb, d.N, d.mcl, d.scale, ws, wb, s);
    });
}

// decode's 11, shared_blocks, workspace, stream
PyObject* decode_shared(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    if (!count(n, 14)) return nullptr;
    Reader       r{a};
    Decode       d(r, a);
    const int    sb = r.integer(a[11]);
    void*        ws = r.ptr(a[12]);
    const size_t wb = r.nbytes(a[12]);
    void*        s = r.stream(a[13]);
    return finish(r, [&] {
        return fn.decode_shared(d.q, d.out, d.qt, d.kc, d.vc, d.ct, d.ks, d.vs, d.bt, d.cx, d.B, d.Hq, d.Hkv, d.D,
                                FFKV_BLOCK_SIZE, d.mb, d.N, d.mcl, d.scale, sb, ws, wb, s);
    });
}

// decode's 11, k_new, v_new, workspace, stream
PyObject* append_decode(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    if (!count(n, 15)) return nullptr;
    Reader       r{a};
    Decode       d(r, a);
    void *       k = r.ptr(a[11]), *v = r.ptr(a[12]);
    const int    st = r.dtype(a[11]);
    void*        ws = r.ptr(a[13]);
    const size_t wb = r.nbytes(a[13]);
    void*        s = r.stream(a[14]);
    return finish(r, [&] {
        return fn.append_decode(k, v, st, d.q, d.out, d.qt, d.kc, d.vc, d.ct, d.ks, d.vs, d.bt, d.cx, d.B, d.Hq, d.Hkv,
                                d.D, FFKV_BLOCK_SIZE, d.mb, d.N, d.mcl, d.scale, ws, wb, s);
    });
}

// decode's 11, stream
PyObject* decode_noalloc(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    if (!count(n, 12)) return nullptr;
    Reader r{a};
    Decode d(r, a);
    void*  s = r.stream(a[11]);
    return finish(r, [&] {
        return fn.decode_noalloc(d.q, d.out, d.qt, d.kc, d.vc, d.ct, d.ks, d.vs, d.bt, d.cx, d.B, d.Hq, d.Hkv, d.D,
                                 FFKV_BLOCK_SIZE, d.mb, d.N, d.mcl, d.scale, s);
    });
}

// q, out, k_cache, v_cache, k_scale, v_scale, block_table, context_lens, max_context_len, scale, num_blocks, stream,
// scratch (bytes, q, stream) -> a tensor or None
PyObject* prefill(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    if (!count(n, 13)) return nullptr;
    Reader r{a};
    int    B, S, Hq, D;
    r.dims4(a[0], B, S, Hq, D);
    const int   Hkv = r.dim(a[2], 2);
    const bool  paged = a[6] != Py_None;
    const int   mb = paged ? r.dim(a[6], -1) : 0, N = paged ? r.blocks(a[10], a[2]) : 0;
    void *      q = r.ptr(a[0]), *out = r.ptr(a[1]), *kc = r.ptr(a[2]), *vc = r.ptr(a[3]);
    const int   qt = r.dtype(a[0]), ct = r.dtype(a[2]);
    auto *      ks = r.ptr<float>(a[4]), *vs = r.ptr<float>(a[5]);
    auto *      bt = r.ptr<int32_t>(a[6]), *cx = r.ptr<int32_t>(a[7]);
    const int   mcl = r.integer(a[8]);
    const float scale = r.real(a[9]);
    void*       s = r.stream(a[11]);
    if (!r.ok) return nullptr;
    PyObject*    ws = nullptr;
    const size_t need = fn.prefill_bytes(qt, ct, B, S, Hq, Hkv, D, paged, mb, mcl);
    if (need > 0)
    {
        PyObject* nb = PyLong_FromSize_t(need);
        ws = nb ? PyObject_CallFunctionObjArgs(a[12], nb, a[0], a[11], nullptr) : nullptr;
        Py_XDECREF(nb);
        if (ws == nullptr) return nullptr;
    }
    void*        w = ws ? r.ptr(ws) : nullptr;
    const size_t wb = ws ? r.nbytes(ws) : 0;
    PyObject*    rc = finish(r, [&] {
        return fn.prefill(q, out, qt, kc, vc, ct, ks, vs, bt, cx, B, S, Hq, Hkv, D, FFKV_BLOCK_SIZE, mb, N, mcl, scale,
                             w, wb, s);
    });
    Py_XDECREF(ws);  // its memory goes back to the allocator of the call's stream, whose later work may reuse it
    return rc;
}

// q or None, k, context_lens, theta, stream
PyObject* rope(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    if (!count(n, 5)) return nullptr;
    Reader r{a};
    int    B, S, Hkv, D;
    r.dims4(a[1], B, S, Hkv, D);
    const int   Hq = a[0] == Py_None ? 0 : r.dim(a[0], 2), st = r.dtype(a[1]);
    void *      q = r.ptr(a[0]), *k = r.ptr(a[1]);
    auto*       cx = r.ptr<int32_t>(a[2]);
    const float theta = r.real(a[3]);
    void*       s = r.stream(a[4]);
    return finish(r, [&] { return fn.rope(q, k, st, cx, B, S, Hq, Hkv, D, theta, s); });
}

// q or None, k, v, k_cache, v_cache, block_table, context_lens, theta, k_scale, v_scale, num_blocks, stream
PyObject* rope_append(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    if (!count(n, 12)) return nullptr;
    Reader r{a};
    int    B, S, Hkv, D;
    r.dims4(a[1], B, S, Hkv, D);
    const int   Hq = a[0] == Py_None ? 0 : r.dim(a[0], 2), mb = r.dim(a[5], -1), N = r.blocks(a[10], a[3]);
    const int   st = r.dtype(a[1]), ct = r.dtype(a[3]);
    void *      q = r.ptr(a[0]), *k = r.ptr(a[1]), *v = r.ptr(a[2]), *kc = r.ptr(a[3]), *vc = r.ptr(a[4]);
    auto *      bt = r.ptr<int32_t>(a[5]), *cx = r.ptr<int32_t>(a[6]);
    const float theta = r.real(a[7]);
    auto *      ks = r.ptr<float>(a[8]), *vs = r.ptr<float>(a[9]);
    void*       s = r.stream(a[11]);
    return finish(r, [&] {
        return fn.rope_append(q, k, v, st, kc, vc, ct, ks, vs, bt, cx, B, S, Hq, Hkv, D, FFKV_BLOCK_SIZE, mb, N, theta, s);
    });
}

// bind(addresses, [(dtype, code), ..], get_device, raw_stream, first_stream): the library's functions in Functions'
// order, torch's dtypes, and how the current stream's handle is found (first_stream() until it has succeeded once,
// which initialises torch's GPU state; then raw_stream(get_device())).
PyObject* bind(PyObject*, PyObject* args)
{
    PyObject *addrs, *types, *dev, *raw, *first;
    if (!PyArg_ParseTuple(args, "O!O!OOO", &PyTuple_Type, &addrs, &PyList_Type, &types, &dev, &raw, &first)) return nullptr;
    constexpr Py_ssize_t kFns = sizeof(Functions) / sizeof(void*);
    if (!count(PyTuple_GET_SIZE(addrs), kFns)) return nullptr;
    void* p[kFns];
    for (Py_ssize_t i = 0; i < kFns; ++i) p[i] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(addrs, i));
    std::vector<DtypeCode> d;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(types); ++i)
    {
        DtypeCode c{};
        if (!PyArg_ParseTuple(PyList_GET_ITEM(types, i), "Oi", &c.dtype, &c.code)) return nullptr;
        d.push_back(c);
    }
    if (PyErr_Occurred()) return nullptr;
    for (const DtypeCode& c : d) Py_INCREF(c.dtype);
    dtypes = d;  // an earlier binding's references are kept: dtypes live as long as torch
    Py_INCREF(dev), Py_INCREF(raw), Py_INCREF(first);
    get_device = dev, raw_stream = raw, first_stream = first, stream_ready = false;
    __builtin_memcpy(&fn, p, sizeof(fn));
    Py_RETURN_NONE;
}

// The next call looks the stream up through first_stream() again (a forked child has no GPU state of its own).
PyObject* forget_stream(PyObject*, PyObject*)
{
    stream_ready = false;
    Py_RETURN_NONE;
}

#define FAST(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FAST(append),         FAST(decode),  FAST(decode_shared), FAST(append_decode),
                         FAST(decode_noalloc), FAST(prefill), FAST(rope),          FAST(rope_append),
                         {"bind", bind, METH_VARARGS, nullptr},
                         {"forget_stream", forget_stream, METH_NOARGS, nullptr},
                         {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_front", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__front(void)
{
    s_shape = PyUnicode_InternFromString("shape");
    s_dtype = PyUnicode_InternFromString("dtype");
    s_data_ptr = PyUnicode_InternFromString("data_ptr");
    s_nbytes = PyUnicode_InternFromString("nbytes");
    s_cuda_stream = PyUnicode_InternFromString("cuda_stream");
    if (PyErr_Occurred()) return nullptr;
    return PyModule_Create(&module);
}
