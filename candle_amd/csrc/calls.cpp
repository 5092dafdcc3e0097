// The matmul-side calls of qhip.py in native code: argument checks, the result tensor, the workspace and the stream of one
// call, then the C ABI (include/candle_qhip.h).  A decode launch of the matmul kernel takes about 5 us of device time; the
// same steps written in Python over ctypes took 10 us of host time per call and bounded it (4096x4096 Q4K, one row, calls
// back to back: 10.5 us), here they take about 3.
//
// The matmuls return None where they do not take their arguments (wrong type, shape, device, layout): qhip.py then words
// the error.  The C functions are handed over by address (`bind`), so that whichever libcandle_qhip.so qhip.py loaded is the
// one that is called.
//
// torch's C++ side throws (a tensor without memory under vmap, grad or a tracer; no memory left; no device): `entry` turns what
// reaches it into the Python exception that torch's own calls raise, so references are held by objects that let go of them.
#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/device_lazy_init.h>

#include <climits>

#include "../../include/candle_qhip.h"

namespace {

struct Abi {
    decltype(&cq_last_error) last_error;
    decltype(&cq_weight_shape) weight_shape;
    decltype(&cq_weight_device) weight_device;
    decltype(&cq_workspace_bytes) workspace_bytes;
    decltype(&cq_qmatmul) qmatmul;
    decltype(&cq_qmatmul_fused) qmatmul_fused;
    decltype(&cq_qmatmul_multi) qmatmul_multi;
    decltype(&cq_grouped_workspace_bytes) grouped_workspace_bytes;
    decltype(&cq_qmatmul_grouped) qmatmul_grouped;
    decltype(&cq_qmatmul_grouped_fused) qmatmul_grouped_fused;
    decltype(&cq_weight_dequantize) weight_dequantize;
    decltype(&cq_weight_dequantize_f16) weight_dequantize_f16;
} g_abi;
PyObject *g_error = nullptr, *g_workspace = nullptr;                     // qhip.QHipError, qhip.Workspace
PyObject *g_s_addr = nullptr, *g_s_buf = nullptr, *g_s_get = nullptr;   // "_addr", "buf", "get"

// An owned reference.
struct Ref {
    PyObject *p = nullptr;
    Ref() = default;
    explicit Ref(PyObject *o) : p(o) {}
    Ref(const Ref &) = delete;
    Ref &operator=(const Ref &) = delete;
    ~Ref() { Py_XDECREF(p); }
    PyObject *release() {
        PyObject *o = p;
        p = nullptr;
        return o;
    }
};

// The weights of one call, any number of them, and their results.
using Weights = c10::SmallVector<const cq_weight *, 16>;
using Results = c10::SmallVector<float *, 16>;

void *stream_now() { return (void *)c10::hip::getCurrentHIPStream().stream(); }

PyObject *fail(int rc) {
    PyErr_Format(g_error, "[%d] %s", rc, g_abi.last_error());
    return nullptr;
}

// The cq_weight behind a qhip.QWeight; null (no Python error) if the object has none.
const cq_weight *weight_of(PyObject *w) {
    PyObject *a = PyObject_GetAttr(w, g_s_addr);
    if (!a) {
        PyErr_Clear();
        return nullptr;
    }
    void *p = PyLong_AsVoidPtr(a);
    Py_DECREF(a);
    if (PyErr_Occurred()) PyErr_Clear();
    return (const cq_weight *)p;
}

bool f32_on_device(PyObject *x) {
    if (!THPVariable_Check(x)) return false;
    const at::Tensor &t = THPVariable_Unpack(x);
    return t.is_cuda() && t.scalar_type() == at::kFloat && t.is_contiguous();
}

// The operand of the fused step `pre`, with the shape rules of qhip._check_pre.  (Without a step nothing reads it.)
bool aux_ok(int pre, const at::Tensor &x, PyObject *aux) {
    if (pre == CQ_PRE_NONE) return true;
    if (!f32_on_device(aux)) return false;
    const at::Tensor &a = THPVariable_Unpack(aux);
    if (pre == CQ_PRE_RMS_NORM) return a.dim() == 1 && a.size(0) == x.size(-1);
    return pre == CQ_PRE_SILU_MUL && a.sizes() == x.sizes();
}

// Its address, after aux_ok.
const float *aux_floats(int pre, PyObject *aux) { return pre == CQ_PRE_NONE ? nullptr : (const float *)THPVariable_Unpack(aux).data_ptr(); }

// At least `need` bytes on x's device out of the caller's workspace: anything with a `get(bytes, device)`, which is spared
// where a qhip.Workspace (and no class derived from it) holds enough already.  *held keeps the buffer alive during the call.
bool workspace(PyObject *ws, size_t need, const at::Tensor &x, PyObject *px, Ref *held, void **ptr, size_t *bytes) {
    if ((PyObject *)Py_TYPE(ws) == g_workspace) {
        held->p = PyObject_GetAttr(ws, g_s_buf);
        if (!held->p) return false;
        const auto fits = [&](const at::Tensor &b) { return (size_t)b.numel() >= need && b.device() == x.device(); };
        if (!THPVariable_Check(held->p) || !fits(THPVariable_Unpack(held->p))) Py_CLEAR(held->p);
    }
    if (!held->p) {
        const Ref dev(PyObject_GetAttrString(px, "device")), n(PyLong_FromSize_t(need));
        held->p = dev.p && n.p ? PyObject_CallMethodObjArgs(ws, g_s_get, n.p, dev.p, nullptr) : nullptr;
        if (!held->p) return false;
        if (!THPVariable_Check(held->p)) {
            PyErr_Format(PyExc_TypeError, "the workspace gave no tensor");
            return false;
        }
    }
    const at::Tensor &b = THPVariable_Unpack(held->p);
    *ptr = b.data_ptr();
    *bytes = (size_t)b.numel();
    return true;
}

at::Tensor empty_f32(at::IntArrayRef sizes, c10::Device dev) { return at::Tensor(at::detail::empty_cuda(sizes, at::kFloat, dev, std::nullopt)); }

// x's shape with its last dimension replaced by n
at::Tensor result_like(const at::Tensor &x, int64_t n) {
    c10::SmallVector<int64_t, 6> sizes(x.sizes().begin(), x.sizes().end());
    sizes.back() = n;
    return empty_f32(sizes, x.device());
}

bool as_int(PyObject *o, int *v) {
    const long l = PyLong_AsLong(o);
    if (l == -1 && PyErr_Occurred()) return false;
    *v = (int)l;
    return true;
}

// qmatmul(w, x, flags, out, workspace, pre, aux, eps)
PyObject *py_qmatmul(PyObject *const *a, Py_ssize_t na) {
    if (na != 8) return PyErr_Format(PyExc_TypeError, "qmatmul takes 8 arguments");
    int flags, pre;
    if (!as_int(a[2], &flags) || !as_int(a[5], &pre)) return nullptr;
    const double eps = pre == CQ_PRE_NONE ? 0.0 : PyFloat_AsDouble(a[7]);
    if (eps == -1.0 && PyErr_Occurred()) return nullptr;
    const cq_weight *w = weight_of(a[0]);
    PyObject *px = a[1], *aux = a[6];
    if (!w || !f32_on_device(px) || (a[3] != Py_None && !THPVariable_Check(a[3]))) Py_RETURN_NONE;
    const at::Tensor &x = THPVariable_Unpack(px);
    int64_t n, k;
    if (g_abi.weight_shape(w, &n, &k) != CQ_OK || x.dim() < 2 || x.size(-1) != k || !aux_ok(pre, x, aux)) Py_RETURN_NONE;
    const int64_t m = k ? x.numel() / k : 0;
    Ref held, out;
    void *ws;
    size_t ws_bytes;
    if (!workspace(a[4], g_abi.workspace_bytes(w, m, flags), x, px, &held, &ws, &ws_bytes)) return nullptr;
    if (a[3] == Py_None) {
        out.p = THPVariable_Wrap(result_like(x, n));
        if (!out.p) return nullptr;
    } else {
        Py_INCREF(out.p = a[3]);
    }
    float *y = (float *)THPVariable_Unpack(out.p).data_ptr();
    const float *xp = (const float *)x.data_ptr(), *ap = aux_floats(pre, aux);
    void *s = stream_now();
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = pre == CQ_PRE_NONE ? g_abi.qmatmul(w, xp, m, y, flags, ws, ws_bytes, s)
                            : g_abi.qmatmul_fused(w, pre, xp, ap, (float)eps, m, y, flags, ws, ws_bytes, s);
    Py_END_ALLOW_THREADS
    return rc == CQ_OK ? out.release() : fail(rc);
}

// The weights of a list; false where it is empty or an element has none.
bool weights_of(PyObject *list, Weights *ws) {
    if (!PyList_Check(list)) return false;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(list); i++) {
        ws->push_back(weight_of(PyList_GET_ITEM(list, i)));
        if (!ws->back()) return false;
    }
    return !ws->empty() && ws->size() <= (size_t)INT_MAX;
}

// qmatmul_multi(weights, x, flags, workspace, pre, aux, eps)
PyObject *py_qmatmul_multi(PyObject *const *a, Py_ssize_t na) {
    if (na != 7) return PyErr_Format(PyExc_TypeError, "qmatmul_multi takes 7 arguments");
    int flags, pre;
    if (!as_int(a[2], &flags) || !as_int(a[4], &pre)) return nullptr;
    const double eps = PyFloat_AsDouble(a[6]);
    if (eps == -1.0 && PyErr_Occurred()) return nullptr;
    Weights ws;
    Results ys;
    PyObject *px = a[1], *aux = a[5];
    if (!weights_of(a[0], &ws) || !f32_on_device(px) || (aux != Py_None && !THPVariable_Check(aux))) Py_RETURN_NONE;
    const at::Tensor &x = THPVariable_Unpack(px);
    int64_t n, k;
    if (g_abi.weight_shape(ws[0], &n, &k) != CQ_OK || x.dim() < 2 || x.size(-1) != k || !aux_ok(pre, x, aux)) Py_RETURN_NONE;
    const int64_t m = k ? x.numel() / k : 0;
    size_t need = 0;
    for (const cq_weight *w : ws) need = std::max(need, g_abi.workspace_bytes(w, m, flags));
    Ref held;
    void *wp;
    size_t ws_bytes;
    if (!workspace(a[3], need, x, px, &held, &wp, &ws_bytes)) return nullptr;
    Ref outs(PyList_New((Py_ssize_t)ws.size()));
    if (!outs.p) return nullptr;
    for (size_t i = 0; i < ws.size(); i++) {
        int64_t ni, ki;
        g_abi.weight_shape(ws[i], &ni, &ki);
        PyObject *o = THPVariable_Wrap(result_like(x, ni));
        if (!o) return nullptr;
        PyList_SET_ITEM(outs.p, (Py_ssize_t)i, o);
        ys.push_back((float *)THPVariable_Unpack(o).data_ptr());
    }
    const float *xp = (const float *)x.data_ptr(), *ap = aux_floats(pre, aux);
    void *s = stream_now();
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = g_abi.qmatmul_multi(ws.data(), (int)ws.size(), pre, xp, ap, (float)eps, m, ys.data(), flags, wp, ws_bytes, s);
    Py_END_ALLOW_THREADS
    return rc == CQ_OK ? outs.release() : fail(rc);
}

struct Buffer {
    Py_buffer b{};
    ~Buffer() { PyBuffer_Release(&b); }   // (nothing where no buffer was taken)
};

// qmatmul_grouped(experts, x, row_ids, offsets (int32 buffer), flags, workspace, pre, aux, eps)
PyObject *py_qmatmul_grouped(PyObject *const *a, Py_ssize_t na) {
    if (na != 9) return PyErr_Format(PyExc_TypeError, "qmatmul_grouped takes 9 arguments");
    int flags, pre;
    if (!as_int(a[4], &flags) || !as_int(a[6], &pre)) return nullptr;
    const double eps = pre == CQ_PRE_NONE ? 0.0 : PyFloat_AsDouble(a[8]);
    if (eps == -1.0 && PyErr_Occurred()) return nullptr;
    Weights ws;
    PyObject *px = a[1], *ids = a[2], *aux = a[7];
    if (!weights_of(a[0], &ws) || !f32_on_device(px) || (ids != Py_None && !THPVariable_Check(ids))) Py_RETURN_NONE;
    const at::Tensor &x = THPVariable_Unpack(px);
    int64_t n, k;
    if (g_abi.weight_shape(ws[0], &n, &k) != CQ_OK || !aux_ok(pre, x, aux)) Py_RETURN_NONE;
    Buffer offs;
    if (PyObject_GetBuffer(a[3], &offs.b, PyBUF_C_CONTIGUOUS) != 0) return nullptr;
    const int32_t *offsets = (const int32_t *)offs.b.buf;
    const Py_ssize_t have = offs.b.len / (Py_ssize_t)sizeof(int32_t);
    if (offs.b.itemsize != sizeof(int32_t) || have < (Py_ssize_t)ws.size() + 1) Py_RETURN_NONE;
    const int64_t total = offsets[have - 1];
    if (total < 0) return PyErr_Format(g_error, "offsets must be non-negative");
    Ref held;
    void *wp;
    size_t ws_bytes;
    if (!workspace(a[5], g_abi.grouped_workspace_bytes(ws.data(), (int)ws.size(), total, flags), x, px, &held, &wp, &ws_bytes)) return nullptr;
    Ref out(THPVariable_Wrap(empty_f32({total, n}, x.device())));
    if (!out.p) return nullptr;
    float *y = (float *)THPVariable_Unpack(out.p).data_ptr();
    const float *xp = (const float *)x.data_ptr(), *ap = aux_floats(pre, aux);
    const int32_t *rid = ids == Py_None ? nullptr : (const int32_t *)THPVariable_Unpack(ids).data_ptr();
    void *s = stream_now();
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = pre == CQ_PRE_NONE ? g_abi.qmatmul_grouped(ws.data(), (int)ws.size(), xp, rid, offsets, y, flags, wp, ws_bytes, s)
                            : g_abi.qmatmul_grouped_fused(ws.data(), (int)ws.size(), pre, xp, ap, (float)eps, rid, offsets, y, flags, wp, ws_bytes, s);
    Py_END_ALLOW_THREADS
    return rc == CQ_OK ? out.release() : fail(rc);
}

// dequantize(w, f16)
PyObject *py_dequantize(PyObject *const *a, Py_ssize_t na) {
    if (na != 2) return PyErr_Format(PyExc_TypeError, "dequantize takes 2 arguments");
    const bool f16 = PyObject_IsTrue(a[1]) == 1;
    const cq_weight *w = weight_of(a[0]);
    int64_t n, k;
    if (const int rc = g_abi.weight_shape(w, &n, &k); rc != CQ_OK) return fail(rc);   // (no weight is an error there)
    torch::utils::device_lazy_init(c10::kCUDA);   // the one call that may come before torch has touched the device
    const c10::Device dev(c10::kCUDA, (c10::DeviceIndex)g_abi.weight_device(w));
    Ref out(THPVariable_Wrap(at::Tensor(at::detail::empty_cuda({n, k}, f16 ? at::kHalf : at::kFloat, dev, std::nullopt))));
    if (!out.p) return nullptr;
    void *p = THPVariable_Unpack(out.p).data_ptr(), *s = stream_now();
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = f16 ? g_abi.weight_dequantize_f16(w, (uint16_t *)p, s) : g_abi.weight_dequantize(w, (float *)p, s);
    Py_END_ALLOW_THREADS
    return rc == CQ_OK ? out.release() : fail(rc);
}

template <typename F> bool take(PyObject *table, const char *name, F *f) {
    PyObject *v = PyDict_GetItemString(table, name);
    if (!v) {
        PyErr_Format(PyExc_KeyError, "%s", name);
        return false;
    }
    *f = (F)PyLong_AsVoidPtr(v);
    return !PyErr_Occurred();
}

// bind({name: address}, error class, workspace class)
PyObject *py_bind(PyObject *const *a, Py_ssize_t na) {
    if (na != 3 || !PyDict_Check(a[0])) return PyErr_Format(PyExc_TypeError, "bind takes a dict and two classes");
#define TAKE(f) take(a[0], "cq_" #f, &g_abi.f)
    if (!(TAKE(last_error) && TAKE(weight_shape) && TAKE(weight_device) && TAKE(workspace_bytes) && TAKE(qmatmul) && TAKE(qmatmul_fused) &&
          TAKE(qmatmul_multi) && TAKE(grouped_workspace_bytes) && TAKE(qmatmul_grouped) && TAKE(qmatmul_grouped_fused) &&
          TAKE(weight_dequantize) && TAKE(weight_dequantize_f16)))
        return nullptr;
#undef TAKE
    Py_INCREF(a[1]);
    Py_XSETREF(g_error, a[1]);
    Py_INCREF(a[2]);
    Py_XSETREF(g_workspace, a[2]);
    Py_RETURN_NONE;
}

template <PyObject *(*F)(PyObject *const *, Py_ssize_t)> PyObject *entry(PyObject *, PyObject *const *a, Py_ssize_t na) {
    try {
        return F(a, na);
    } catch (const std::exception &) {
        torch::translate_exception_to_python(std::current_exception());
        return nullptr;
    }
}

#define FAST(f) (PyCFunction)(void (*)(void))entry<f>, METH_FASTCALL, nullptr
PyMethodDef g_methods[] = {{"bind", FAST(py_bind)},
                           {"qmatmul", FAST(py_qmatmul)},
                           {"qmatmul_multi", FAST(py_qmatmul_multi)},
                           {"qmatmul_grouped", FAST(py_qmatmul_grouped)},
                           {"dequantize", FAST(py_dequantize)},
                           {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls(void) {
    g_s_addr = PyUnicode_InternFromString("_addr");
    g_s_buf = PyUnicode_InternFromString("buf");
    g_s_get = PyUnicode_InternFromString("get");
    return PyModule_Create(&g_module);
}
