// The operator calls of capi.Context as native functions.
//
// A caller that enqueues a network layer by layer is bound by the host: a layer of 3 us on the GPU cost 5.6 us in Python,
// 1.5 of them turning six tensors and two descriptors into ctypes objects and 0.5 in ctypes' own call.  Here an operator
// converts its arguments straight into the C call (a tensor's address by its data_ptr(), a descriptor by its buffer) and
// releases the interpreter lock around it, as ctypes does.  What a call accepts, returns and raises is what the ctypes
// binding of the remaining entry points does.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <tuple>
#include <utility>

#include "tosa_mi355.h"

namespace
{

PyObject *g_error = nullptr, *g_argument_error = nullptr, *g_tensor = nullptr;    // TmiError, ctypes.ArgumentError, DeviceTensor
PyObject *s_handle = nullptr, *s_value = nullptr, *s_ptr = nullptr, *s_data_ptr = nullptr;

template <typename D>
PyObject* g_desc = nullptr;    // the ctypes structure that mirrors D

// ---- one argument ---------------------------------------------------------------------------------------------------------
struct Buffers    // of the call's descriptors; held until it returns
{
    Py_buffer view[2];
    int n = 0;
    ~Buffers()
    {
        while (n)
            PyBuffer_Release(&view[--n]);
    }
};

bool convert(PyObject* x, int64_t& v, Buffers&)
{
    if (PyFloat_Check(x) || (!PyLong_Check(x) && !PyIndex_Check(x)))
    {
        PyErr_Format(g_argument_error, "int expected instead of %s instance", Py_TYPE(x)->tp_name);
        return false;
    }
    v = (int64_t)PyLong_AsUnsignedLongLongMask(x);
    return v != -1 || !PyErr_Occurred();
}

bool convert(PyObject* x, int32_t& v, Buffers& b)
{
    int64_t w;
    if (!convert(x, w, b))
        return false;
    v = (int32_t)w;
    return true;
}

bool address(PyObject* number, const void*& v)
{
    if (!number)
        return false;
    if (number == Py_None)
        v = nullptr;
    else
        v = (const void*)(uintptr_t)PyLong_AsUnsignedLongLongMask(number);
    Py_DECREF(number);
    return v != (const void*)(uintptr_t)-1 || !PyErr_Occurred();
}

// device pointer of a DeviceTensor, a torch tensor, an int, or None
bool convert(PyObject* x, const void*& v, Buffers&)
{
    if (x == Py_None)
    {
        v = nullptr;
        return true;
    }
    if (PyObject_TypeCheck(x, (PyTypeObject*)g_tensor))
        return address(PyObject_GetAttr(x, s_ptr), v);
    if (PyLong_Check(x))
    {
        Py_INCREF(x);
        return address(x, v);
    }
    PyObject* a = PyObject_CallMethodNoArgs(x, s_data_ptr);
    if (!a && PyErr_ExceptionMatches(PyExc_AttributeError) && !PyObject_HasAttr(x, s_data_ptr))
    {
        PyErr_Clear();
        PyErr_Format(PyExc_TypeError, "not a device tensor: %R", (PyObject*)Py_TYPE(x));
    }
    return address(a, v);
}

bool convert(PyObject* x, void*& v, Buffers& b)
{
    const void* p;
    if (!convert(x, p, b))
        return false;
    v = const_cast<void*>(p);
    return true;
}

template <typename D>
bool convert(PyObject* x, const D*& v, Buffers& b)
{
    if (!PyObject_TypeCheck(x, (PyTypeObject*)g_desc<D>))
    {
        PyErr_Format(g_argument_error, "expected %s instance instead of %s", ((PyTypeObject*)g_desc<D>)->tp_name, Py_TYPE(x)->tp_name);
        return false;
    }
    if (PyObject_GetBuffer(x, &b.view[b.n], PyBUF_SIMPLE) != 0)
        return false;
    v = (const D*)b.view[b.n++].buf;
    return true;
}

// the context of the call: Context.handle, a ctypes.c_void_p, or None once it is closed
bool convert(PyObject* self, tmi_ctx_t*& v, Buffers&)
{
    PyObject* h = PyObject_GetAttr(self, s_handle);
    if (!h)
        return false;
    const void* p = nullptr;
    if (h == Py_None)
    {
        Py_DECREF(h);
        v = nullptr;
        return true;
    }
    const bool ok = address(PyObject_GetAttr(h, s_value), p);
    Py_DECREF(h);
    v = (tmi_ctx_t*)const_cast<void*>(p);
    return ok;
}

// ---- the call -------------------------------------------------------------------------------------------------------------
PyObject* result(tmi_ctx_t* ctx, int rc)
{
    if (rc == TMI_ERROR)
    {
        PyObject* e = PyObject_CallFunction(g_error, "is", rc, tmi_last_error(ctx));
        if (e)
        {
            PyErr_SetObject(g_error, e);
            Py_DECREF(e);
        }
        return nullptr;
    }
    return PyLong_FromLong(rc);
}

// Python arguments by position or name -> at[0 .. n); the last `optional` of them may be left out (nullptr)
bool collect(const char* fn, const char* const* names, int n, int optional, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames,
             PyObject** at)
{
    if (nargs > n)
    {
        PyErr_Format(PyExc_TypeError, "%s() takes %d positional arguments but %zd were given", fn, n, nargs);
        return false;
    }
    for (int i = 0; i < n; i++)
        at[i] = i < nargs ? args[i] : nullptr;
    const Py_ssize_t nkw = kwnames ? PyTuple_GET_SIZE(kwnames) : 0;
    for (Py_ssize_t k = 0; k < nkw; k++)
    {
        PyObject* name = PyTuple_GET_ITEM(kwnames, k);
        int i          = 0;
        while (i < n && PyUnicode_CompareWithASCIIString(name, names[i]) != 0)
            i++;
        if (i == n || at[i])
        {
            PyErr_Format(PyExc_TypeError, i == n ? "%s() got an unexpected keyword argument '%U'" : "%s() got multiple values for argument '%U'",
                         fn, name);
            return false;
        }
        at[i] = args[nargs + k];
    }
    for (int i = 0; i < n - optional; i++)
        if (!at[i])
        {
            PyErr_Format(PyExc_TypeError, "%s() missing required argument: '%s'", fn, names[i]);
            return false;
        }
    return true;
}

template <auto Fn, typename... A, size_t... I>
PyObject* call(int (*)(A...), PyObject* const* at, std::index_sequence<I...>)
{
    Buffers buffers;
    std::tuple<A...> a;
    if (!(convert(at[I], std::get<I>(a), buffers) && ...))
        return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = Fn(std::get<I>(a)...);
    Py_END_ALLOW_THREADS
    return result(std::get<0>(a), rc);
}

template <typename... A>
constexpr int arity(int (*)(A...))
{
    return sizeof...(A);
}

template <auto Fn>
struct Operator
{
    static constexpr int n = arity(Fn);
    static const char* name;
    static const char* const* names;
    static PyObject* run(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames)
    {
        PyObject* at[n];
        if (!collect(name, names, n, 0, args, nargs, kwnames, at))
            return nullptr;
        return call<Fn>(Fn, at, std::make_index_sequence<n>{});
    }
};
template <auto Fn>
const char* Operator<Fn>::name = nullptr;
template <auto Fn>
const char* const* Operator<Fn>::names = nullptr;

// CONV2D / DEPTHWISE_CONV2D + RESCALE (+ CLAMP): `clamp` is None or a pair (lowest, highest)
template <auto Fn>
PyObject* run_fused(const char* name, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames)
{
    static const char* const names[] = { "self", "d", "inp", "w", "bias", "in_zp", "w_zp", "r", "mult", "shift", "out", "clamp" };
    PyObject* at[12];
    if (!collect(name, names, 12, 1, args, nargs, kwnames, at))
        return nullptr;
    PyObject *limits = nullptr, *lo = nullptr, *hi = nullptr;
    const bool clamped = at[11] && at[11] != Py_None;
    if (clamped)
    {
        limits = PySequence_Fast(at[11], "clamp must be a pair (lowest, highest)");
        if (!limits)
            return nullptr;
        if (PySequence_Fast_GET_SIZE(limits) != 2)
        {
            PyErr_SetString(PyExc_ValueError, "clamp must be a pair (lowest, highest)");
            Py_DECREF(limits);
            return nullptr;
        }
        lo = PySequence_Fast_GET_ITEM(limits, 0), hi = PySequence_Fast_GET_ITEM(limits, 1);
    }
    Buffers b;
    tmi_ctx_t* ctx;
    const tmi_conv_desc_t* d;
    const tmi_rescale_desc_t* r;
    const void *in, *w, *bias, *mult, *shift;
    void* out;
    int32_t in_zp, w_zp, v_lo = 0, v_hi = 0;
    const bool ok = convert(at[0], ctx, b) && convert(at[1], d, b) && convert(at[2], in, b) && convert(at[3], w, b) && convert(at[4], bias, b) &&
                    convert(at[5], in_zp, b) && convert(at[6], w_zp, b) && convert(at[7], r, b) && convert(at[8], mult, b) &&
                    convert(at[9], shift, b) && convert(at[10], out, b) && (!clamped || (convert(lo, v_lo, b) && convert(hi, v_hi, b)));
    Py_XDECREF(limits);
    if (!ok)
        return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = Fn(ctx, d, in, w, bias, in_zp, w_zp, r, mult, shift, clamped, v_lo, v_hi, out);
    Py_END_ALLOW_THREADS
    return result(ctx, rc);
}

PyObject* run_conv_fused(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames)
{
    return run_fused<tmi_conv2d_rescale_clamp>("conv2d_rescale_clamp", args, nargs, kwnames);
}

PyObject* run_depthwise_fused(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames)
{
    return run_fused<tmi_depthwise_conv2d_rescale_clamp>("depthwise_conv2d_rescale_clamp", args, nargs, kwnames);
}

template <auto Fn, size_t N>
PyMethodDef op(const char* name, const char* const (&names)[N], const char* doc)
{
    static_assert(N == Operator<Fn>::n, "one name for each argument of the entry point");
    Operator<Fn>::name  = name;
    Operator<Fn>::names = names;
    return PyMethodDef{ name, (PyCFunction)(void (*)())Operator<Fn>::run, METH_FASTCALL | METH_KEYWORDS, doc };
}

const char* const kConv[]    = { "self", "d", "inp", "w", "bias", "in_zp", "w_zp", "out" };
const char* const kMatmul[]  = { "self", "in_dtype", "n", "h", "c", "w", "a", "b", "a_zp", "b_zp", "out" };
const char* const kRescale[] = { "self", "r", "rank", "rows", "c", "inp", "mult", "shift", "out" };
const char* const kClamp[]   = { "self", "dtype", "n", "inp", "lo", "hi", "out" };
const char* const kAvg[]     = { "self", "d", "inp", "in_zp", "out_zp", "out" };
const char* const kMax[]     = { "self", "d", "inp", "out" };

PyMethodDef g_methods[] = {
    op<tmi_conv2d>("conv2d", kConv, "conv2d($self, d, inp, w, bias, in_zp, w_zp, out)\n--\n\nCONV2D; d: ConvDesc"),
    op<tmi_depthwise_conv2d>("depthwise_conv2d", kConv, "depthwise_conv2d($self, d, inp, w, bias, in_zp, w_zp, out)\n--\n\nDEPTHWISE_CONV2D; d: ConvDesc"),
    op<tmi_transpose_conv2d>("transpose_conv2d", kConv, "transpose_conv2d($self, d, inp, w, bias, in_zp, w_zp, out)\n--\n\nTRANSPOSE_CONV2D; d: TconvDesc"),
    op<tmi_conv3d>("conv3d", kConv, "conv3d($self, d, inp, w, bias, in_zp, w_zp, out)\n--\n\nCONV3D; d: Conv3dDesc"),
    op<tmi_matmul>("matmul", kMatmul, "matmul($self, in_dtype, n, h, c, w, a, b, a_zp, b_zp, out)\n--\n\nMATMUL"),
    op<tmi_rescale>("rescale", kRescale, "rescale($self, r, rank, rows, c, inp, mult, shift, out)\n--\n\nRESCALE; r: RescaleDesc"),
    op<tmi_clamp>("clamp", kClamp, "clamp($self, dtype, n, inp, lo, hi, out)\n--\n\nCLAMP of integers"),
    op<tmi_avg_pool2d>("avg_pool2d", kAvg, "avg_pool2d($self, d, inp, in_zp, out_zp, out)\n--\n\nAVG_POOL2D; d: PoolDesc"),
    op<tmi_max_pool2d>("max_pool2d", kMax, "max_pool2d($self, d, inp, out)\n--\n\nMAX_POOL2D; d: PoolDesc"),
    { "conv2d_rescale_clamp", (PyCFunction)(void (*)())run_conv_fused, METH_FASTCALL | METH_KEYWORDS,
      "conv2d_rescale_clamp($self, d, inp, w, bias, in_zp, w_zp, r, mult, shift, out, clamp=None)\n--\n\nCONV2D + RESCALE (+ CLAMP)" },
    { "depthwise_conv2d_rescale_clamp", (PyCFunction)(void (*)())run_depthwise_fused, METH_FASTCALL | METH_KEYWORDS,
      "depthwise_conv2d_rescale_clamp($self, d, inp, w, bias, in_zp, w_zp, r, mult, shift, out, clamp=None)\n--\n\n"
      "DEPTHWISE_CONV2D + RESCALE (+ CLAMP)" },
};

// install(Context, DeviceTensor, TmiError, ctypes.ArgumentError, ConvDesc, TconvDesc, Conv3dDesc, PoolDesc, RescaleDesc):
// the operators become methods of Context
PyObject* install(PyObject*, PyObject* args)
{
    PyObject *context, **kept[] = { &g_tensor, &g_error, &g_argument_error, &g_desc<tmi_conv_desc_t>, &g_desc<tmi_tconv_desc_t>,
                                    &g_desc<tmi_conv3d_desc_t>, &g_desc<tmi_pool_desc_t>, &g_desc<tmi_rescale_desc_t> };
    PyObject* got[8];
    if (!PyArg_ParseTuple(args, "OOOOOOOOO", &context, &got[0], &got[1], &got[2], &got[3], &got[4], &got[5], &got[6], &got[7]))
        return nullptr;
    const Py_ssize_t sizes[] = { sizeof(tmi_conv_desc_t), sizeof(tmi_tconv_desc_t), sizeof(tmi_conv3d_desc_t), sizeof(tmi_pool_desc_t),
                                 sizeof(tmi_rescale_desc_t) };
    for (int i = 0; i < 8; i++)
    {
        if (!PyType_Check(got[i]))
            return PyErr_Format(PyExc_TypeError, "install: argument %d is no type", i + 2), nullptr;
        if (i >= 3)    // the structure is as large as the one it mirrors
        {
            PyObject* one = PyObject_CallNoArgs(got[i]);
            Py_buffer view;
            if (!one || PyObject_GetBuffer(one, &view, PyBUF_SIMPLE) != 0)
                return Py_XDECREF(one), nullptr;
            const bool ok = view.len == sizes[i - 3];
            PyBuffer_Release(&view);
            Py_DECREF(one);
            if (!ok)
                return PyErr_Format(PyExc_TypeError, "install: %R has the wrong size", got[i]), nullptr;
        }
        Py_INCREF(got[i]);
        Py_XSETREF(*kept[i], got[i]);
    }
    for (PyMethodDef& m : g_methods)
    {
        PyObject* f      = PyCFunction_New(&m, nullptr);
        PyObject* method = f ? PyInstanceMethod_New(f) : nullptr;
        Py_XDECREF(f);
        if (!method || PyObject_SetAttrString(context, m.ml_name, method) != 0)
            return Py_XDECREF(method), nullptr;
        Py_DECREF(method);
    }
    Py_RETURN_NONE;
}

PyMethodDef g_functions[] = { { "install", install, METH_VARARGS, nullptr }, { nullptr, nullptr, 0, nullptr } };
PyModuleDef g_module      = { PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, g_functions, nullptr, nullptr, nullptr, nullptr };

}    // namespace

PyMODINIT_FUNC PyInit__calls()
{
    s_handle = PyUnicode_InternFromString("handle"), s_value = PyUnicode_InternFromString("value");
    s_ptr = PyUnicode_InternFromString("ptr"), s_data_ptr = PyUnicode_InternFromString("data_ptr");
    return PyModule_Create(&g_module);
}
