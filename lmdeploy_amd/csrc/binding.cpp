// The calls of lmdeploy_amd/turbomind.py that a decode step or a layer's conversion makes, from Python to the C ABI without ctypes
// in between: each tensor's checks and address, the current stream, and the call itself.  The kernel of a 4096 x 4096 matrix takes 3.3 us for one
// token; through ctypes and Python's accessors the host needed 4.9 us for such a call, and 3.9 this way, of which the runtime's launch
// takes 2.3.  A descriptor of a sequence takes 0.04 us instead of 0.8: the 128 of a decode step of 32 layers 5 us instead of 98.
// A small layer's conversion, which the host sets the time of, takes 30 us instead of 54 (in one launch instead of four).
//
// Each function takes plain arguments only: None or a contiguous GPU tensor whose type is torch.Tensor or torch.nn.Parameter
// itself, and whole numbers that fit their C types.  For anything else it returns None without having done anything, and the caller
// goes through ctypes and the tensors' attributes, which take every other form and raise every error.
//
// The library is not linked: its entry points' addresses come from the ctypes binding that has loaded it (`bind`).
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <torch/csrc/autograd/python_variable.h>

#include <limits.h>

#include "../../include/w4a16.h"

namespace {

decltype(&w4a16_gemm)            fn_gemm;
decltype(&w4a16_gemm_static)     fn_gemm_static;
decltype(&w4a16_ffn)             fn_ffn;
decltype(&w4a16_convert_s4_k_m8) fn_convert;
decltype(&w4a16_deploy_layer)    fn_deploy_layer;
PyObject *                       get_device, *get_stream, *parameter_type;  // torch's accessors, and torch.nn.Parameter

// The address of a plain contiguous tensor on the GPU, nullptr for None
bool address(PyObject* t, void** out)
{
    *out = nullptr;
    if (t == Py_None) return true;
    if ((PyObject*)Py_TYPE(t) != THPVariableClass && (PyObject*)Py_TYPE(t) != parameter_type) return false;
    try {
        const at::Tensor& v = THPVariable_Unpack(t);
        if (!v.is_cuda() || !v.is_contiguous()) return false;
        *out = v.data_ptr();
        return true;
    }
    catch (...) {  // a tensor without a storage of its own, as inside a transform
        return false;
    }
}

// `count` addresses; a mode that intercepts what is asked of a tensor has to see it
bool addresses(PyObject* const* t, int count, void** out)
{
    if (at::impl::torch_function_mode_enabled()) return false;
    for (int i = 0; i < count; ++i)
        if (!address(t[i], out + i)) return false;
    return true;
}

bool numbers(PyObject* const* o, int count, int* out)
{
    for (int i = 0; i < count; ++i) {
        int        over = 0;
        const long v    = PyLong_Check(o[i]) ? PyLong_AsLongAndOverflow(o[i], &over) : LONG_MAX;
        if (over || v < INT_MIN || v > INT_MAX) return false;
        out[i] = (int)v;
    }
    return true;
}

// a whole number as a pointer
bool pointer(PyObject* o, void** out)
{
    if (!PyLong_Check(o)) return false;
    *out = PyLong_AsVoidPtr(o);
    if (*out == nullptr && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    return true;
}

// a stream's handle; of None, torch's current stream's.  What torch's accessors raise, the general path raises again
bool stream_of(PyObject* o, void** out)
{
    if (o != Py_None) return pointer(o, out);
    PyObject* const dev = PyObject_CallNoArgs(get_device);
    PyObject* const s   = dev ? PyObject_CallOneArg(get_stream, dev) : nullptr;
    const bool      ok  = s && pointer(s, out);
    if (!s) PyErr_Clear();
    Py_XDECREF(dev);
    Py_XDECREF(s);
    return ok;
}

// (handle, C, A, B, Q, residual, m, n, k, group_size, type, algo_id, stream)
PyObject* gemm(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    void *h, *p[5], *st;
    int   v[6], rc;
    if (n != 13 || !pointer(a[0], &h) || !addresses(a + 1, 5, p) || !numbers(a + 6, 6, v) || !stream_of(a[12], &st)) Py_RETURN_NONE;
    Py_BEGIN_ALLOW_THREADS;
    rc = fn_gemm(static_cast<w4a16_handle*>(h), p[0], p[1], p[2], p[3], p[4], v[0], v[1], v[2], v[3], v[4], v[5], st);
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(rc);
}

// (C, A, B, Q, residual, m, n, k, group_size, type, algo_id, stream)
PyObject* gemm_static(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    void *p[5], *st;
    int   v[6], rc;
    if (n != 12 || !addresses(a, 5, p) || !numbers(a + 5, 6, v) || !stream_of(a[11], &st)) Py_RETURN_NONE;
    Py_BEGIN_ALLOW_THREADS;
    rc = fn_gemm_static(p[0], p[1], p[2], p[3], p[4], v[0], v[1], v[2], v[3], v[4], v[5], st);
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(rc);
}

// (handle, output, gating buffer, input, A13, Q13, A2, Q2, residual, hidden_units, inter_size, n, group_size, stream)
PyObject* ffn(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    void *h, *p[8], *st;
    int   v[4], rc;
    if (n != 14 || !pointer(a[0], &h) || !addresses(a + 1, 8, p) || !numbers(a + 9, 4, v) || !stream_of(a[13], &st)) Py_RETURN_NONE;
    Py_BEGIN_ALLOW_THREADS;
    rc = fn_ffn(static_cast<w4a16_handle*>(h), p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], v[0], v[1], v[2], v[3], st);
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(rc);
}

// (A_dst, Q_dst, workspace, A_src, scales, qzeros, m, k, group_size)
PyObject* convert(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    void *p[6], *st;
    int   v[3], rc;
    if (n != 9 || !addresses(a, 6, p) || !numbers(a + 6, 3, v) || !stream_of(Py_None, &st)) Py_RETURN_NONE;
    Py_BEGIN_ALLOW_THREADS;
    rc = fn_convert(static_cast<uint32_t*>(p[0]), p[1], p[2], static_cast<uint32_t*>(p[3]), p[4], static_cast<uint32_t*>(p[5]), v[0], v[1],
                    v[2], st);
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(rc);
}

// the addresses of `count` triples (qweight, qzeros, scales), tuples each
bool triples(PyObject* const* t, int count, uint32_t** qweight, uint32_t** qzeros, void** scales)
{
    for (int i = 0; i < count; ++i) {
        void* p[3];
        if (!PyTuple_CheckExact(t[i]) || PyTuple_GET_SIZE(t[i]) != 3 || !addresses(PySequence_Fast_ITEMS(t[i]), 3, p)) return false;
        qweight[i] = static_cast<uint32_t*>(p[0]), qzeros[i] = static_cast<uint32_t*>(p[1]), scales[i] = p[2];
    }
    return true;
}

// (4 pairs (A, Q), 7 triples (qweight, qzeros, scales), 7 widths, 4 numbers of rows, size_per_head, group_size), tuples all of them
PyObject* deploy_layer(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    void *    Q[4], *scales[7], *p[2], *st;
    uint32_t *dst[4], *qweight[7], *qzeros[7];
    int       width[7], rows[4], v[2], rc;
    auto      tuple = [](PyObject* o, Py_ssize_t size) { return PyTuple_CheckExact(o) && PyTuple_GET_SIZE(o) == size; };
    bool      ok    = n == 6 && tuple(a[0], 4) && tuple(a[1], 7) && tuple(a[2], 7) && tuple(a[3], 4);
    for (int i = 0; ok && i < 4; ++i) {
        PyObject* const t = PyTuple_GET_ITEM(a[0], i);
        ok                = tuple(t, 2) && addresses(PySequence_Fast_ITEMS(t), 2, p);
        if (ok) dst[i] = static_cast<uint32_t*>(p[0]), Q[i] = p[1];
    }
    ok = ok && triples(PySequence_Fast_ITEMS(a[1]), 7, qweight, qzeros, scales);
    if (!ok || !numbers(PySequence_Fast_ITEMS(a[2]), 7, width) || !numbers(PySequence_Fast_ITEMS(a[3]), 4, rows) || !numbers(a + 4, 2, v) ||
        !stream_of(Py_None, &st))
        Py_RETURN_NONE;
    Py_BEGIN_ALLOW_THREADS;
    rc = fn_deploy_layer(dst, Q, qweight, qzeros, scales, width, rows, v[0], v[1], st);
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(rc);
}

// (writable array of w4a16_gemm_desc, list or tuple of tuples (C, A, B, Q, m, k, type, residual, depends)) -> True: the array is filled
PyObject* describe(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    if (n != 2 || !(PyList_CheckExact(a[1]) || PyTuple_CheckExact(a[1]))) Py_RETURN_NONE;
    Py_buffer buf;
    if (PyObject_GetBuffer(a[0], &buf, PyBUF_WRITABLE) != 0) return nullptr;
    const Py_ssize_t count = PySequence_Fast_GET_SIZE(a[1]);
    bool             ok    = buf.len == count * (Py_ssize_t)sizeof(w4a16_gemm_desc);
    auto*            d     = static_cast<w4a16_gemm_desc*>(buf.buf);
    for (Py_ssize_t i = 0; ok && i < count; ++i, ++d) {
        PyObject* const g = PySequence_Fast_GET_ITEM(a[1], i);
        ok                = PyTuple_CheckExact(g) && PyTuple_GET_SIZE(g) == 9;
        if (!ok) break;
        PyObject* const* const t = PySequence_Fast_ITEMS(g);
        void *                 p[4], *r;
        int                    v[3];
        ok = addresses(t, 4, p) && addresses(t + 7, 1, &r) && numbers(t + 4, 3, v) && PyLong_Check(t[8]);  // (bool is a long)
        if (ok) *d = w4a16_gemm_desc{p[0], p[1], p[2], p[3], r, v[0], v[1], v[2], PyObject_IsTrue(t[8])};
    }
    PyBuffer_Release(&buf);
    if (!ok) Py_RETURN_NONE;
    Py_RETURN_TRUE;
}

// (tensor): its address; None or anything but a plain tensor: None
PyObject* ptr(PyObject*, PyObject* t)
{
    void* p;
    if (t == Py_None || !addresses(&t, 1, &p)) Py_RETURN_NONE;
    return PyLong_FromVoidPtr(p);
}

// (addresses of the five functions above, accessor of the current device, of its current stream, torch.nn.Parameter)
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    void* f[5];
    bool  ok = n == 8;
    for (int i = 0; ok && i < 5; ++i) ok = pointer(a[i], &f[i]);
    if (!ok) {
        PyErr_SetString(PyExc_TypeError, "bind: five addresses, two accessors and a type");
        return nullptr;
    }
    fn_gemm         = reinterpret_cast<decltype(fn_gemm)>(f[0]);
    fn_gemm_static  = reinterpret_cast<decltype(fn_gemm_static)>(f[1]);
    fn_ffn          = reinterpret_cast<decltype(fn_ffn)>(f[2]);
    fn_convert      = reinterpret_cast<decltype(fn_convert)>(f[3]);
    fn_deploy_layer = reinterpret_cast<decltype(fn_deploy_layer)>(f[4]);
    for (int i = 5; i < 8; ++i) Py_INCREF(a[i]);
    get_device = a[5], get_stream = a[6], parameter_type = a[7];
    Py_RETURN_NONE;
}

#define W4A16_FAST(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {W4A16_FAST(bind), W4A16_FAST(gemm), W4A16_FAST(gemm_static), W4A16_FAST(ffn), W4A16_FAST(convert),
                         W4A16_FAST(deploy_layer), W4A16_FAST(describe),
                         {"ptr", ptr, METH_O, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_binding", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__binding()
{
    PyObject* const m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "torch_version", W4A16_TORCH) != 0) {  // whose layout of a tensor is compiled in
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
