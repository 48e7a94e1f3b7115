// slideformer_amd: the host side of LayerAdam's calls on HIP tensors, as a
// CPython module (plain C++17 against torch's headers, no HIP).
//
// A step of a small layer is bound by the host's issue time: in Python the
// checks, the packing of a layer's tensors and ctypes' argument conversion took
// 6 us of a step_chunk (10 us with its launch), 10 of a clip_grad_norm (14) and
// 23 of a twelve-tensor step_with_grad_views (33).  The functions here do the
// same checks on the tensors themselves and call the library's C-ABI through
// the addresses of the library that slideformer_amd._lib has loaded.
//
// update() and update_multi() handle the calls that pass every check, and
// return None for any other, before anything has changed: the caller then takes
// its per-call path, which raises the reference's errors in the reference's
// order or streams host tensors.  The GIL is released around the library calls,
// as ctypes releases it.  Nothing is kept from one call for the next.

#include <Python.h>

#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cstdint>
#include <exception>
#include <vector>

#include "../../include/layer_adam.h"

namespace {

decltype(&la_adam_update) p_update = nullptr;
decltype(&la_adam_update_multi) p_update_multi = nullptr;
decltype(&la_grad_sqnorm) p_sqnorm = nullptr;
decltype(&la_grad_norm_clip) p_norm_clip = nullptr;
decltype(&la_grad_norm_multi) p_norm_multi = nullptr;

int code_of(const at::Tensor& t)
{
    switch (t.scalar_type()) {
    case at::kFloat: return LA_F32;
    case at::kBFloat16: return LA_BF16;
    case at::kHalf: return LA_F16;
    default: return -1;
    }
}

// The (param, grad, state) triples the reference registers, cpu_adam_impl.cpp:181-189.
bool registered(int p, int g, int s)
{
    if (p < 0 || g < 0 || s < 0) return false;
    if (p == LA_F32) return s == LA_F32;
    if (p == LA_BF16) return g != LA_F16 && (s == LA_F32 || (s == LA_BF16 && g == LA_BF16));
    return g != LA_BF16 && (s == LA_F32 || (s == LA_F16 && g == LA_F16));
}

// Whether a tensor answers for itself as torch.Tensor does: a plain tensor or
// Parameter, or a subclass that leaves __torch_function__ and the methods read
// here as they are and does not dispatch to Python (such a one has no memory of
// its own, or hides it).
bool own_answers(PyObject* o)
{
    if (THPVariable_CheckExact(o)) return true;
    if (!THPVariable_Check(o) || THPVariable_Unpack(o).unsafeGetTensorImpl()->is_python_dispatch()) return false;
    PyObject* type = reinterpret_cast<PyObject*>(Py_TYPE(o));
    auto same = [type](PyObject* base, const char* name) {
        PyObject *a = PyObject_GetAttrString(type, name), *b = PyObject_GetAttrString(base, name);
        // a class method is bound anew at every look: what it is bound to counts
        const bool bound = a && b && PyMethod_Check(a) && PyMethod_Check(b);
        const bool equal = a && b && (bound ? PyMethod_GET_FUNCTION(a) == PyMethod_GET_FUNCTION(b) : a == b);
        Py_XDECREF(a);
        Py_XDECREF(b);
        PyErr_Clear();
        return equal;
    };
    if (!same(THPVariableClass, "__torch_function__") && !same(ParameterClass, "__torch_function__")) return false;
    for (const char* name : {"data_ptr", "numel", "is_contiguous", "get_device", "dtype", "is_cuda"})
        if (!same(THPVariableClass, name)) return false;
    return true;
}

// A tensor that answers for itself, with memory of its own on HIP device
// `dev`, contiguous; null otherwise.
const at::Tensor* plain(PyObject* o, int64_t dev)
{
    if (!own_answers(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || t.layout() != at::kStrided || !t.is_cuda() || t.get_device() != dev || !t.has_storage() ||
        !t.is_contiguous())
        return nullptr;
    return &t;
}

// A float32 tensor of at least one element on device `dev`, or None (then *out is null).
bool coefficient(PyObject* o, int64_t dev, const float** out)
{
    *out = nullptr;
    if (o == Py_None) return true;
    if (!own_answers(o)) return false;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || t.layout() != at::kStrided || !t.is_cuda() || t.get_device() != dev || !t.has_storage() ||
        t.scalar_type() != at::kFloat || t.numel() < 1)
        return false;
    *out = static_cast<const float*>(t.data_ptr());
    return true;
}

// id, step, lr, beta1, beta2, eps, weight_decay, bias_correction, device, stream: the scalars of a call.
struct Call {
    int id, bias_correction;
    uint64_t step;
    float lr, beta1, beta2, eps, wd;
    int64_t dev;
    la_stream_t stream;
};
constexpr Py_ssize_t kCallArgs = 10;

// False with an exception set, or without one for a hyper-parameter that is no
// number: anything with a float value is one, as for a ctypes float argument
// (the caller's path then decides about it).
bool parse(PyObject* const* a, Call& c)
{
    float x[5];
    for (int k = 0; k < 5; ++k) {
        const double d = PyFloat_AsDouble(a[2 + k]);
        if (d == -1.0 && PyErr_Occurred()) {
            PyErr_Clear();
            return false;
        }
        x[k] = static_cast<float>(d);
    }
    c.id = static_cast<int>(PyLong_AsLong(a[0]));
    c.step = PyLong_AsUnsignedLongLongMask(a[1]);    // modulo 2^64, as a ctypes uint64 argument takes it
    c.lr = x[0];
    c.beta1 = x[1];
    c.beta2 = x[2];
    c.eps = x[3];
    c.wd = x[4];
    c.bias_correction = PyObject_IsTrue(a[7]);
    c.dev = PyLong_AsLongLong(a[8]);
    c.stream = PyLong_AsVoidPtr(a[9]);
    return !PyErr_Occurred();
}

PyObject* failed(const char* what)
{
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, what);
    return nullptr;
}

// update(*Call, params, grads, exp_avg, exp_avg_sq, bf16_out | None, clip_coef | None) -> rc | None
PyObject* update(PyObject*, PyObject* const* a, Py_ssize_t n)
try {
    if (n != kCallArgs + 6) return PyErr_Format(PyExc_TypeError, "update takes 16 arguments");
    Call c;
    if (!parse(a, c)) {
        if (PyErr_Occurred()) return nullptr;
        Py_RETURN_NONE;
    }
    const at::Tensor *p = plain(a[10], c.dev), *g = plain(a[11], c.dev), *m = plain(a[12], c.dev),
                     *v = plain(a[13], c.dev);
    if (!p || !g || !m || !v) Py_RETURN_NONE;
    const int64_t count = p->numel();
    const int pc = code_of(*p), gc = code_of(*g), sc = code_of(*m);
    if (g->numel() != count || m->numel() != count || v->numel() != count || code_of(*v) != sc ||
        !registered(pc, gc, sc))
        Py_RETURN_NONE;
    uint16_t* out = nullptr;
    if (a[14] != Py_None) {
        const at::Tensor* o = plain(a[14], c.dev);
        if (!o || o->numel() != count || o->scalar_type() != at::kBFloat16) Py_RETURN_NONE;
        out = static_cast<uint16_t*>(o->data_ptr());
    }
    const float* coef;
    if (!coefficient(a[15], c.dev, &coef)) Py_RETURN_NONE;
    void *pp = p->data_ptr(), *mp = m->data_ptr(), *vp = v->data_ptr();
    const void* gp = g->data_ptr();
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = p_update(c.id, c.step, c.lr, c.beta1, c.beta2, c.eps, c.wd, c.bias_correction, pc, pp, gc, gp, sc, mp, vp,
                  static_cast<uint64_t>(count), out, coef, c.stream);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
} catch (const std::exception& e) {
    return failed(e.what());
}

// update_multi(*Call, [(params, grads, exp_avg, exp_avg_sq), ...], clip_coef | None) -> rc | None
PyObject* update_multi(PyObject*, PyObject* const* a, Py_ssize_t n)
try {
    if (n != kCallArgs + 2 || !PyList_Check(a[10]))
        return PyErr_Format(PyExc_TypeError, "update_multi takes 11 arguments and a list");
    Call c;
    if (!parse(a, c)) {
        if (PyErr_Occurred()) return nullptr;
        Py_RETURN_NONE;
    }
    const Py_ssize_t count = PyList_GET_SIZE(a[10]);
    if (count < 1) Py_RETURN_NONE;
    std::vector<la_segment_t> segs(static_cast<size_t>(count));
    // where the update writes: no two tensors may overlap.  The intervals are
    // disjoint exactly if, sorted apart, every end is at or before the next start.
    std::vector<uintptr_t> starts, ends;
    starts.reserve(3 * static_cast<size_t>(count));
    ends.reserve(3 * static_cast<size_t>(count));
    int codes[3] = {};
    for (Py_ssize_t k = 0; k < count; ++k) {
        PyObject* e = PyList_GET_ITEM(a[10], k);
        if (!PyTuple_Check(e) || PyTuple_GET_SIZE(e) != 4) Py_RETURN_NONE;
        const at::Tensor* t[4];
        int code[4];
        for (int j = 0; j < 4; ++j) {
            t[j] = plain(PyTuple_GET_ITEM(e, j), c.dev);
            if (!t[j] || t[j]->numel() != t[0]->numel()) Py_RETURN_NONE;
            code[j] = code_of(*t[j]);
        }
        if (k == 0) {
            if (!registered(code[0], code[1], code[2])) Py_RETURN_NONE;
            std::copy(code, code + 3, codes);
        }
        if (code[0] != codes[0] || code[1] != codes[1] || code[2] != codes[2] || code[3] != codes[2]) Py_RETURN_NONE;
        const uint64_t numel = static_cast<uint64_t>(t[0]->numel());
        segs[k] = {t[0]->data_ptr(), t[1]->data_ptr(), t[2]->data_ptr(), t[3]->data_ptr(), nullptr, numel};
        for (int j : {0, 2, 3}) {
            if (numel == 0) break;
            const uintptr_t at = reinterpret_cast<uintptr_t>(t[j]->data_ptr());
            starts.push_back(at);
            ends.push_back(at + numel * (code[j] == LA_F32 ? 4 : 2));
        }
    }
    std::sort(starts.begin(), starts.end());
    std::sort(ends.begin(), ends.end());
    for (size_t i = 0; i + 1 < starts.size(); ++i)
        if (ends[i] > starts[i + 1]) Py_RETURN_NONE;
    const float* coef;
    if (!coefficient(a[11], c.dev, &coef)) Py_RETURN_NONE;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = p_update_multi(c.id, c.step, c.lr, c.beta1, c.beta2, c.eps, c.wd, c.bias_correction, codes[0], codes[1],
                        codes[2], segs.data(), static_cast<int>(count), coef, c.stream);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
} catch (const std::exception& e) {
    return failed(e.what());
}

// check_grads(grads, device index) -> None | (position, why): the first grad
// that the norm does not take: 0 another device, 1 not contiguous, 2 its type.
PyObject* check_grads(PyObject*, PyObject* const* a, Py_ssize_t n)
try {
    if (n != 2 || !PyList_Check(a[0])) return PyErr_Format(PyExc_TypeError, "check_grads takes a list and a device");
    const int64_t dev = PyLong_AsLongLong(a[1]);
    if (dev == -1 && PyErr_Occurred()) return nullptr;
    for (Py_ssize_t k = 0; k < PyList_GET_SIZE(a[0]); ++k) {
        PyObject* o = PyList_GET_ITEM(a[0], k);
        if (!THPVariable_Check(o)) return PyErr_Format(PyExc_TypeError, "grads must be tensors");
        const at::Tensor& t = THPVariable_Unpack(o);
        if (!t.is_cuda() || t.get_device() != dev) return Py_BuildValue("(ni)", k, 0);
        if (!t.is_contiguous()) return Py_BuildValue("(ni)", k, 1);
        if (code_of(t) < 0) return Py_BuildValue("(ni)", k, 2);
    }
    Py_RETURN_NONE;
} catch (const std::exception& e) {
    return failed(e.what());
}

// norm(grads, workspace, its bytes, sqnorm, accumulate, max_norm, cn | 0, stream) -> rc
// The sum of squares of checked grads into the float64 at `sqnorm` (added to
// it when accumulate): runs of one dtype, at most LA_NORM_MULTI_MAX buffers
// each, one library call per run, later runs adding to the earlier ones;
// la_grad_norm_multi for a run of several buffers, la_grad_sqnorm /
// la_grad_norm_clip for a run of one (the same bits, a smaller launch).  With
// `cn` (address of two fp32: coef, norm) the last call also writes the clip
// coefficient.
PyObject* norm(PyObject*, PyObject* const* a, Py_ssize_t n)
try {
    if (n != 8 || !PyList_Check(a[0])) return PyErr_Format(PyExc_TypeError, "norm takes a list and 7 arguments");
    void* work = PyLong_AsVoidPtr(a[1]);
    const uint64_t bytes = PyLong_AsUnsignedLongLong(a[2]);
    double* sqnorm = static_cast<double*>(PyLong_AsVoidPtr(a[3]));
    const int accumulate = PyObject_IsTrue(a[4]);
    const float max_norm = static_cast<float>(PyFloat_AsDouble(a[5]));
    float* cn = static_cast<float*>(PyLong_AsVoidPtr(a[6]));
    const la_stream_t stream = PyLong_AsVoidPtr(a[7]);
    if (PyErr_Occurred()) return nullptr;
    const Py_ssize_t count = PyList_GET_SIZE(a[0]);
    std::vector<la_grad_buffer_t> bufs(static_cast<size_t>(count));
    std::vector<int> codes(static_cast<size_t>(count));
    for (Py_ssize_t k = 0; k < count; ++k) {
        const at::Tensor& t = THPVariable_Unpack(PyList_GET_ITEM(a[0], k));
        bufs[k] = {t.data_ptr(), static_cast<uint64_t>(t.numel())};
        codes[k] = code_of(t);
    }
    int rc = LA_OK;
    Py_BEGIN_ALLOW_THREADS
    for (Py_ssize_t k = 0, end; k < count && rc == LA_OK; k = end) {
        end = k + 1;
        while (end < count && codes[end] == codes[k] && end - k < LA_NORM_MULTI_MAX) ++end;
        float* coef = end == count ? cn : nullptr;
        const int acc = accumulate || k > 0;
        if (end - k > 1)
            rc = p_norm_multi(codes[k], &bufs[k], static_cast<int>(end - k), work, bytes, sqnorm, acc, max_norm, coef,
                              coef ? coef + 1 : nullptr, stream);
        else if (coef)
            rc = p_norm_clip(codes[k], bufs[k].g, bufs[k].n, work, bytes, sqnorm, acc, max_norm, coef, coef + 1,
                             stream);
        else
            rc = p_sqnorm(codes[k], bufs[k].g, bufs[k].n, work, bytes, sqnorm, acc, stream);
    }
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
} catch (const std::exception& e) {
    return failed(e.what());
}

// bind(addresses of la_adam_update, la_adam_update_multi, la_grad_sqnorm,
// la_grad_norm_clip, la_grad_norm_multi): of the library _lib has loaded.
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    if (n != 5) return PyErr_Format(PyExc_TypeError, "bind takes 5 addresses");
    void* at[5];
    for (int k = 0; k < 5; ++k) {
        at[k] = PyLong_AsVoidPtr(a[k]);
        if (!at[k]) return PyErr_Occurred() ? nullptr : PyErr_Format(PyExc_ValueError, "bind: null address");
    }
    p_update = reinterpret_cast<decltype(p_update)>(at[0]);
    p_update_multi = reinterpret_cast<decltype(p_update_multi)>(at[1]);
    p_sqnorm = reinterpret_cast<decltype(p_sqnorm)>(at[2]);
    p_norm_clip = reinterpret_cast<decltype(p_norm_clip)>(at[3]);
    p_norm_multi = reinterpret_cast<decltype(p_norm_multi)>(at[4]);
    Py_RETURN_NONE;
}

PyCFunction fast(_PyCFunctionFast f) { return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)); }

PyMethodDef methods[] = {{"bind", fast(bind), METH_FASTCALL, nullptr},
                         {"update", fast(update), METH_FASTCALL, nullptr},
                         {"update_multi", fast(update_multi), METH_FASTCALL, nullptr},
                         {"check_grads", fast(check_grads), METH_FASTCALL, nullptr},
                         {"norm", fast(norm), METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host_calls(void) { return PyModule_Create(&module); }
