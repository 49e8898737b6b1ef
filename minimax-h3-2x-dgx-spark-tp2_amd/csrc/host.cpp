// The host path of the common calls, natively: the argument checks, the output allocations and the C-ABI call of
// ops.quant_rows, ops.gemm, the dispatcher's scaled product, ops.gemm_quant, ops.gemm_swiglu_quant, ops.silu_mul_quant,
// ops.rms_quant and ops.gate_rms_quant (h3_tp2_amd/ops.py, fp8_gemm.py).
//
// Every function takes the call only in its plain form -- exact torch tensors on one GPU, the dtypes, shapes and strides
// that the kernels read in place, no caller-supplied outputs -- and returns None for any other, which the Python path then
// computes or refuses as it always did.  Nothing is kept between calls.  What it saves is the interpreter's and ctypes'
// share of a call: quant + dispatched product of two rows (two calls) 19.8 -> 13.5 us a pass, which the kernels bound.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ops/empty.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "h3fp8.h"

namespace {

constexpr c10::DispatchKeySet kWrappers({c10::DispatchKey::Functionalize, c10::DispatchKey::FuncTorchGradWrapper,
                                         c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::Batched});

// A plain GPU tensor with memory of its own (no subclass, no wrapper of a function transform).
const at::Tensor* plain(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage() ||
        t.unsafeGetTensorImpl()->is_python_dispatch() || t.key_set().has_any(kWrappers))
        return nullptr;
    return &t;
}

// A non-empty 2-D tensor with contiguous rows: its row stride (a single row: at least its width), else -1.
int64_t row_stride(const at::Tensor& t) {
    if (t.dim() != 2 || t.size(0) < 1 || t.size(1) < 1 || (t.size(1) > 1 && t.stride(1) != 1)) return -1;
    return t.size(0) > 1 ? t.stride(0) : std::max<int64_t>(t.size(1), t.stride(0));
}

// An fp32 scale of 1 or n entries that is read in place: pointer and element stride (0: a scalar).
bool scale_of(const at::Tensor& s, int64_t n, const float** p, int64_t* stride) {
    if (s.scalar_type() != at::kFloat || (s.numel() != 1 && s.numel() != n)) return false;
    if (s.numel() == 1) *stride = 0;
    else if (s.dim() == 1 || (s.dim() == 2 && s.size(1) == 1)) *stride = s.stride(0);
    else if (s.dim() == 2 && s.size(0) == 1) *stride = s.stride(1);
    else return false;
    *p = static_cast<const float*>(s.data_ptr());
    return true;
}

bool vector_of(const at::Tensor& t, int64_t n, at::ScalarType dt, const at::Device& dev) {
    return t.dim() == 1 && t.numel() == n && t.scalar_type() == dt && t.device() == dev && t.is_contiguous();
}

at::Tensor empty(int64_t m, int64_t n, at::ScalarType dt, const at::Device& dev) {
    return at::empty({m, n}, at::TensorOptions().dtype(dt).device(dev));
}

void* stream_of(const at::Device& dev) { return c10::hip::getCurrentHIPStream(dev.index()).stream(); }

// The exception of a non-zero status (h3_tp2_amd._lib.fail raises it).
PyObject* failed(const char* fn, int rc) {
    PyObject* lib = PyImport_ImportModule("h3_tp2_amd._lib");
    if (!lib) return nullptr;
    PyObject* r = PyObject_CallMethod(lib, "fail", "si", fn, rc);
    Py_DECREF(lib);
    Py_XDECREF(r);
    if (!PyErr_Occurred()) PyErr_Format(PyExc_RuntimeError, "%s returned %d", fn, rc);
    return nullptr;
}

template <class... T>
PyObject* tuple_of(T&&... t) {
    PyObject* items[] = {THPVariable_Wrap(std::forward<T>(t))...};
    constexpr Py_ssize_t n = sizeof...(T);
    bool ok = true;
    for (PyObject* o : items) ok = ok && o;
    PyObject* r = ok ? PyTuple_New(n) : nullptr;
    for (Py_ssize_t i = 0; i < n; ++i) {
        if (r) PyTuple_SET_ITEM(r, i, items[i]);
        else Py_XDECREF(items[i]);
    }
    return r;
}

#define DECLINE Py_RETURN_NONE

// quant_rows(x)
PyObject* quant_rows(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const at::Tensor* x = n == 1 ? plain(args[0]) : nullptr;
    if (!x || x->scalar_type() != at::kBFloat16) DECLINE;
    const int64_t ldx = row_stride(*x);
    if (ldx < 0) DECLINE;
    const int64_t M = x->size(0), K = x->size(1);
    const at::Device dev = x->device();
    at::Tensor q, s;
    int rc;
    {
        pybind11::gil_scoped_release nogil;
        q = empty(M, K, at::kFloat8_e4m3fn, dev);
        s = empty(M, 1, at::kFloat, dev);
        rc = h3fp8_quant_rows(x->data_ptr(), ldx, M, K, q.data_ptr(), K, static_cast<float*>(s.data_ptr()), stream_of(dev));
    }
    if (rc) return failed("h3fp8_quant_rows", rc);
    return tuple_of(std::move(q), std::move(s));
    END_HANDLE_TH_ERRORS
}

struct Operands {
    const at::Tensor *a, *w;                             // [M, K] and [N, K] (or its [K, N] view), both e4m3
    int64_t M, N, K, lda, ldw;
    const float *sa, *sb;
    int64_t sa_stride, sb_stride;
    at::Device dev{at::kCPU};
};

// a, w, scale_a, scale_b of a product; w_t: the weight comes as its [K, N] view.
bool operands(PyObject* const* args, bool w_t, Operands* o) {
    const at::Tensor* t[4];
    for (int i = 0; i < 4; ++i) {
        t[i] = plain(args[i]);
        if (!t[i] || t[i]->device() != t[0]->device()) return false;
    }
    o->a = t[0];
    o->w = t[1];
    o->dev = t[0]->device();
    if (t[0]->scalar_type() != at::kFloat8_e4m3fn || t[1]->scalar_type() != at::kFloat8_e4m3fn) return false;
    o->lda = row_stride(*t[0]);
    if (o->lda < 0 || t[1]->dim() != 2) return false;
    o->M = t[0]->size(0);
    o->K = t[0]->size(1);
    if (w_t) {
        if (t[1]->size(0) != o->K || t[1]->stride(0) != 1 || t[1]->stride(1) != o->K || t[1]->size(1) < 1) return false;
        o->N = t[1]->size(1);
        o->ldw = o->K;
    } else {
        o->ldw = row_stride(*t[1]);
        if (o->ldw < 0 || t[1]->size(1) != o->K) return false;
        o->N = t[1]->size(0);
    }
    return scale_of(*t[2], o->M, &o->sa, &o->sa_stride) && scale_of(*t[3], o->N, &o->sb, &o->sb_stride);
}

// A bias argument: None, or a vector of n entries; *p its pointer (or null).
bool bias_of(PyObject* arg, int64_t n, at::ScalarType dt, const at::Device& dev, const void** p) {
    *p = nullptr;
    if (arg == Py_None) return true;
    const at::Tensor* b = plain(arg);
    if (!b || !vector_of(*b, n, dt, dev)) return false;
    *p = b->data_ptr();
    return true;
}

PyObject* product(const Operands& o, at::ScalarType dt, const void* bias) {
    const int code = dt == at::kBFloat16 ? H3FP8_DT_BF16 : dt == at::kHalf ? H3FP8_DT_FP16 : H3FP8_DT_F32;
    at::Tensor y;
    int rc;
    {
        pybind11::gil_scoped_release nogil;
        y = empty(o.M, o.N, dt, o.dev);
        rc = h3fp8_gemm(o.a->data_ptr(), o.lda, o.w->data_ptr(), o.ldw, o.sa, o.sa_stride, o.sb, o.sb_stride, bias,
                        y.data_ptr(), o.N, code, o.M, o.N, o.K, nullptr, stream_of(o.dev));
    }
    if (rc) return failed("h3fp8_gemm", rc);
    return THPVariable_Wrap(std::move(y));
}

// scaled_mm(a, b, scale_a, scale_b, out_dtype, bias): b the weight's [K, N] view; per-tensor scales on both sides and
// sizes that are no multiple of 16 are not this path's
PyObject* scaled_mm(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Operands o;
    const void* bias;
    if (n != 6 || !THPDtype_Check(args[4]) || !operands(args, true, &o)) DECLINE;
    const at::ScalarType dt = reinterpret_cast<THPDtype*>(args[4])->scalar_type;
    if ((dt != at::kBFloat16 && dt != at::kHalf) || !o.a->is_contiguous() || o.K % 16 || o.N % 16 ||
        (THPVariable_Unpack(args[2]).numel() == 1 && THPVariable_Unpack(args[3]).numel() == 1) ||
        !bias_of(args[5], o.N, dt, o.dev, &bias))
        DECLINE;
    o.lda = o.K;
    return product(o, dt, bias);
    END_HANDLE_TH_ERRORS
}

// gemm(a, w, scale_a, scale_b, out_dtype, bias)
PyObject* gemm(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Operands o;
    const void* bias;
    if (n != 6 || !THPDtype_Check(args[4]) || !operands(args, false, &o)) DECLINE;
    const at::ScalarType dt = reinterpret_cast<THPDtype*>(args[4])->scalar_type;
    if ((dt != at::kBFloat16 && dt != at::kHalf && dt != at::kFloat) || (dt == at::kFloat && args[5] != Py_None) ||
        !bias_of(args[5], o.N, dt, o.dev, &bias))
        DECLINE;
    return product(o, dt, bias);
    END_HANDLE_TH_ERRORS
}

// gemm_quant(a, w, scale_a, scale_b, bias)
PyObject* gemm_quant(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Operands o;
    const void* bias;
    if (n != 5 || !operands(args, false, &o) || !bias_of(args[4], o.N, at::kBFloat16, o.dev, &bias)) DECLINE;
    at::Tensor y, amax, q, s;
    int rc;
    {
        pybind11::gil_scoped_release nogil;
        y = empty(o.M, o.N, at::kBFloat16, o.dev);
        amax = empty(o.M, 1, at::kFloat, o.dev);
        q = empty(o.M, o.N, at::kFloat8_e4m3fn, o.dev);
        s = empty(o.M, 1, at::kFloat, o.dev);
        rc = h3fp8_gemm_quant(o.a->data_ptr(), o.lda, o.w->data_ptr(), o.ldw, o.sa, o.sa_stride, o.sb, o.sb_stride, bias,
                              y.data_ptr(), o.N, o.M, o.N, o.K, static_cast<float*>(amax.data_ptr()), q.data_ptr(), o.N,
                              static_cast<float*>(s.data_ptr()), stream_of(o.dev));
    }
    if (rc) return failed("h3fp8_gemm_quant", rc);
    return tuple_of(std::move(y), std::move(q), std::move(s));
    END_HANDLE_TH_ERRORS
}

// gemm_swiglu_quant(a, w_gate_up, scale_a, scale_b, bias)
PyObject* gemm_swiglu_quant(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Operands o;
    const void* bias;
    if (n != 5 || !operands(args, false, &o) || o.N % 2 || !bias_of(args[4], o.N, at::kBFloat16, o.dev, &bias)) DECLINE;
    const int64_t F = o.N / 2;
    at::Tensor h, amax, q, s;
    int rc;
    {
        pybind11::gil_scoped_release nogil;
        h = empty(o.M, F, at::kBFloat16, o.dev);
        amax = empty(o.M, 1, at::kFloat, o.dev);
        q = empty(o.M, F, at::kFloat8_e4m3fn, o.dev);
        s = empty(o.M, 1, at::kFloat, o.dev);
        rc = h3fp8_gemm_swiglu_quant(o.a->data_ptr(), o.lda, o.w->data_ptr(), o.ldw, o.sa, o.sa_stride, o.sb, o.sb_stride,
                                     bias, o.M, F, o.K, h.data_ptr(), static_cast<float*>(amax.data_ptr()), q.data_ptr(),
                                     F, static_cast<float*>(s.data_ptr()), stream_of(o.dev));
    }
    if (rc) return failed("h3fp8_gemm_swiglu_quant", rc);
    return tuple_of(std::move(q), std::move(s));
    END_HANDLE_TH_ERRORS
}

// silu_mul_quant(x)
PyObject* silu_mul_quant(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const at::Tensor* x = n == 1 ? plain(args[0]) : nullptr;
    if (!x || x->scalar_type() != at::kBFloat16) DECLINE;
    const int64_t ldx = row_stride(*x);
    if (ldx < 0 || ldx % 8 || x->size(1) % 8) DECLINE;
    const int64_t M = x->size(0), F = x->size(1) / 2;
    const at::Device dev = x->device();
    at::Tensor q, s;
    int rc;
    {
        pybind11::gil_scoped_release nogil;
        q = empty(M, F, at::kFloat8_e4m3fn, dev);
        s = empty(M, 1, at::kFloat, dev);
        rc = h3fp8_silu_mul_quant(x->data_ptr(), ldx, M, F, q.data_ptr(), F, static_cast<float*>(s.data_ptr()),
                                  stream_of(dev));
    }
    if (rc) return failed("h3fp8_silu_mul_quant", rc);
    return tuple_of(std::move(q), std::move(s));
    END_HANDLE_TH_ERRORS
}

// A producer's rows, weight, tables and indices: all plain, on one GPU.
struct Producer {
    const at::Tensor *x, *weight, *indices;
    const at::Tensor* table[3];
    int64_t M, H, ldx, ld_table[3], n_index;
    double eps;
    at::Device dev{at::kCPU};
};

bool producer(PyObject* x, PyObject* weight, PyObject* const* tables, int n_tables, PyObject* indices, PyObject* eps,
              Producer* p) {
    p->x = plain(x);
    p->weight = plain(weight);
    p->indices = plain(indices);
    if (!p->x || !p->weight || !p->indices || !PyFloat_CheckExact(eps)) return false;
    p->eps = PyFloat_AS_DOUBLE(eps);
    p->dev = p->x->device();
    p->ldx = row_stride(*p->x);
    if (p->ldx < 0 || p->x->scalar_type() != at::kBFloat16) return false;
    p->M = p->x->size(0);
    p->H = p->x->size(1);
    p->n_index = INT64_MAX;
    for (int i = 0; i < n_tables; ++i) {
        const at::Tensor* t = p->table[i] = plain(tables[i]);
        if (!t || t->scalar_type() != at::kBFloat16 || t->device() != p->dev) return false;
        p->ld_table[i] = row_stride(*t);
        if (p->ld_table[i] < 0 || t->size(1) != p->H) return false;
        p->n_index = std::min(p->n_index, t->size(0));
    }
    return vector_of(*p->weight, p->H, at::kBFloat16, p->dev) && p->indices->device() == p->dev &&
           p->indices->dim() == 1 && p->indices->size(0) == p->M &&
           (p->indices->scalar_type() == at::kInt || p->indices->scalar_type() == at::kLong);
}

// rms_quant(x, weight, shift, scale, indices, eps)
PyObject* rms_quant(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Producer p;
    if (n != 6 || !producer(args[0], args[1], args + 2, 2, args[4], args[5], &p)) DECLINE;
    at::Tensor q, s;
    int rc;
    {
        pybind11::gil_scoped_release nogil;
        q = empty(p.M, p.H, at::kFloat8_e4m3fn, p.dev);
        s = empty(p.M, 1, at::kFloat, p.dev);
        rc = h3fp8_rms_quant(p.x->data_ptr(), p.ldx, p.weight->data_ptr(), p.table[0]->data_ptr(), p.ld_table[0],
                             p.table[1]->data_ptr(), p.ld_table[1], p.n_index, p.indices->data_ptr(),
                             p.indices->stride(0), (int)p.indices->element_size(), p.M, p.H, (float)p.eps, q.data_ptr(),
                             p.H, static_cast<float*>(s.data_ptr()), nullptr, 0, stream_of(p.dev));
    }
    if (rc) return failed("h3fp8_rms_quant", rc);
    return tuple_of(std::move(q), std::move(s));
    END_HANDLE_TH_ERRORS
}

// gate_rms_quant(residual, gate, branch, weight, shift, scale, indices, eps)
PyObject* gate_rms_quant(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Producer p;
    if (n != 8) DECLINE;
    PyObject* const tables[3] = {args[1], args[4], args[5]};          // gate, shift, scale
    if (!producer(args[0], args[3], tables, 3, args[6], args[7], &p)) DECLINE;
    const at::Tensor* branch = plain(args[2]);
    if (!branch || branch->scalar_type() != at::kBFloat16 || branch->device() != p.dev ||
        branch->sizes() != p.x->sizes())
        DECLINE;
    const int64_t ldb = row_stride(*branch);
    if (ldb < 0) DECLINE;
    at::Tensor res, q, s;
    int rc;
    {
        pybind11::gil_scoped_release nogil;
        res = empty(p.M, p.H, at::kBFloat16, p.dev);
        q = empty(p.M, p.H, at::kFloat8_e4m3fn, p.dev);
        s = empty(p.M, 1, at::kFloat, p.dev);
        rc = h3fp8_gate_rms_quant(p.x->data_ptr(), p.ldx, p.table[0]->data_ptr(), p.ld_table[0], branch->data_ptr(), ldb,
                                  p.weight->data_ptr(), p.table[1]->data_ptr(), p.ld_table[1], p.table[2]->data_ptr(),
                                  p.ld_table[2], p.n_index, p.indices->data_ptr(), p.indices->stride(0),
                                  (int)p.indices->element_size(), p.M, p.H, (float)p.eps, res.data_ptr(), p.H,
                                  q.data_ptr(), p.H, static_cast<float*>(s.data_ptr()), nullptr, 0, stream_of(p.dev));
    }
    if (rc) return failed("h3fp8_gate_rms_quant", rc);
    return tuple_of(std::move(res), std::move(q), std::move(s));
    END_HANDLE_TH_ERRORS
}

#define METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(name)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {METHOD(quant_rows), METHOD(scaled_mm), METHOD(gemm), METHOD(gemm_quant),
                          METHOD(gemm_swiglu_quant), METHOD(silu_mul_quant), METHOD(rms_quant), METHOD(gate_rms_quant),
                          {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host", "the common calls' host path", -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
    if (h3fp8_abi_version() != H3FP8_ABI_VERSION) {
        PyErr_Format(PyExc_ImportError, "libh3fp8 ABI version %d, expected %d", h3fp8_abi_version(), H3FP8_ABI_VERSION);
        return nullptr;
    }
    // torch's C++ interface is that of one version
    PyObject* torch = PyImport_ImportModule("torch");
    PyObject* version = torch ? PyObject_GetAttrString(torch, "__version__") : nullptr;
    PyObject* text = version ? PyObject_Str(version) : nullptr;
    Py_XDECREF(torch);
    Py_XDECREF(version);
    if (!text) return nullptr;
    const bool same = PyUnicode_CompareWithASCIIString(text, H3_TORCH_VERSION) == 0;
    if (!same) PyErr_Format(PyExc_ImportError, "built on torch %s, loaded by torch %U", H3_TORCH_VERSION, text);
    Py_DECREF(text);
    return same ? PyModule_Create(&kModule) : nullptr;
}
