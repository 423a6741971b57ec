// The host side of an operator call in one native call: argument checks on the tensors' own fields, the output and
// workspace allocations and the library's launch, without the Python objects (shape tuples, dictionary keys, ctypes
// conversions) that cost a call more than its two kernel launches. The module extends kea_kernels.lowbit: everything it does
// not take (tensor subclasses and transforms, arguments that would raise) it declines by returning None / False, and the
// caller's Python path, which holds the full checks and their messages, runs instead.
//
// Calls in a row, host bound: Int8MmaLayer.linear at M = 128, N = 4096, K = 1024 (fp16 in and out) 13.2 -> 9.3 us, at one
// row 13.2 -> 9.9, lowbit.quantize + lowbit.gemm with group scales 21.9 -> 12.9, the provider's call on a few rows 18.7 ->
// 11.7; the two HIP launches are about 6 us of each.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/GradMode.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include <cstdint>
#include <list>
#include <unordered_map>

#include "../../include/kea_lowbit.h"

namespace {

// Library entry points, resolved from the loaded libkea_hip.so by bind().
struct Library {
    decltype(&kea_lowbit_project_launch) project_launch = nullptr;
    decltype(&kea_lowbit_gemm) gemm = nullptr;
    decltype(&kea_lowbit_gemm_residual) gemm_residual = nullptr;
    decltype(&kea_quantize) quantize = nullptr;
} lib;

// The tensor behind an exact torch.Tensor whose memory a kernel may read as it is: on a GPU, strided, no transform
// (functorch, lazy negation or conjugation), nothing that autograd would have to record. nullptr otherwise.
const at::Tensor *plain(PyObject *o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor &t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided) return nullptr;
    constexpr c10::DispatchKeySet transforms({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                              c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize,
                                              c10::DispatchKey::Negative, c10::DispatchKey::Conjugate,
                                              c10::DispatchKey::ZeroTensor});
    if (t.key_set().has_any(transforms)) return nullptr;
    if (t.requires_grad() && c10::GradMode::is_enabled()) return nullptr;
    return &t;
}

// Calls made while something records or rewrites operators (dispatch modes, functorch layers, tracing) are not taken.
bool modes_active() {
    const auto &tls = c10::impl::tls_local_dispatch_key_set();
    return tls.included_.has(c10::DispatchKey::Python) || tls.included_.has(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) ||
           tls.included_.has(c10::DispatchKey::Tracer);
}

int code_of(at::ScalarType t) {
    return t == at::kFloat ? KEA_F32 : t == at::kHalf ? KEA_F16 : t == at::kBFloat16 ? KEA_BF16 : -1;
}

void *stream_of(c10::Device d) { return c10::hip::getCurrentHIPStream(d.index()).stream(); }

// ---- Replays: an operator's resolved call layouts ----

constexpr int kMaxDim = 4;

struct Key {
    int64_t tag;                // what the operator does with the input (its own numbering)
    int64_t sizes[kMaxDim], strides[kMaxDim];
    const void *norm_w, *norm_b;
    int64_t norm_size[2];       // elements of each; -1: a call without a LayerNorm
    float eps;
    int8_t dim, dtype, out_dtype, device;
    bool operator==(const Key &o) const {
        if (tag != o.tag || dim != o.dim || dtype != o.dtype || out_dtype != o.out_dtype || device != o.device ||
            norm_w != o.norm_w || norm_b != o.norm_b || norm_size[0] != o.norm_size[0] || norm_size[1] != o.norm_size[1] ||
            eps != o.eps)
            return false;
        for (int i = 0; i < dim; ++i)
            if (sizes[i] != o.sizes[i] || strides[i] != o.strides[i]) return false;
        return true;
    }
};
struct KeyHash {
    size_t operator()(const Key &k) const {
        uint64_t h = (uint64_t)k.tag * 0x9E3779B97F4A7C15ull + (uint64_t)(uintptr_t)k.norm_w + ((uint64_t)k.out_dtype << 56);
        for (int i = 0; i < k.dim; ++i) {
            h = (h ^ (uint64_t)k.sizes[i]) * 0x100000001B3ull;
            h = (h ^ (uint64_t)k.strides[i]) * 0x100000001B3ull;
        }
        return (size_t)(h ^ (h >> 29));
    }
};

struct Entry {
    PyObject *owner;  // the Python entry that frees the plan
    const kea_project_plan *plan;
    int64_t need;
    c10::SmallVector<int64_t, 4> shape;
    bool transposed;
    std::list<Key>::iterator order;
};

struct Replays {
    PyObject_HEAD
    std::unordered_map<Key, Entry, KeyHash> *entries;
    std::list<Key> *order;  // oldest first
    Py_ssize_t limit;
};

// The key of input x; false where the call cannot be kept or replayed. norm: the call has a LayerNorm, whose parameters
// must be there.
bool make_key(const at::Tensor &x, PyObject *out_dtype, int64_t tag, bool norm, PyObject *norm_w, PyObject *norm_b, double eps,
              Key *k) {
    if (x.dim() > kMaxDim || !THPDtype_Check(out_dtype)) return false;
    *k = Key{};
    k->tag = tag;
    k->dim = (int8_t)x.dim();
    for (int i = 0; i < k->dim; ++i) {
        k->sizes[i] = x.size(i);
        k->strides[i] = x.stride(i);
    }
    k->dtype = (int8_t)x.scalar_type();
    k->out_dtype = (int8_t)((THPDtype *)out_dtype)->scalar_type;
    k->device = x.device().index();
    k->norm_size[0] = k->norm_size[1] = -1;
    if (norm) {  // LayerNorm parameters are read in place, where the plan was made for
        const at::Tensor *w[2];
        PyObject *const o[2] = {norm_w, norm_b};
        for (int i = 0; i < 2; ++i) {
            if (!THPVariable_Check(o[i])) return false;
            w[i] = &THPVariable_Unpack(o[i]);
            if (!w[i]->defined() || w[i]->scalar_type() != at::kFloat || w[i]->device() != x.device() ||
                w[i]->layout() != at::kStrided || !w[i]->is_contiguous() || !w[i]->has_storage())
                return false;
        }
        k->norm_w = w[0]->const_data_ptr();
        k->norm_b = w[1]->const_data_ptr();
        k->norm_size[0] = w[0]->numel();
        k->norm_size[1] = w[1]->numel();
        k->eps = (float)eps;
    }
    return true;
}

PyObject *replays_new(PyTypeObject *type, PyObject *args, PyObject *) {
    Py_ssize_t limit;
    if (!PyArg_ParseTuple(args, "n", &limit)) return nullptr;
    auto *self = (Replays *)type->tp_alloc(type, 0);
    if (!self) return nullptr;
    self->entries = new (std::nothrow) std::unordered_map<Key, Entry, KeyHash>;
    self->order = new (std::nothrow) std::list<Key>;
    self->limit = limit;
    if (!self->entries || !self->order) {
        Py_DECREF(self);
        return PyErr_NoMemory();
    }
    return (PyObject *)self;
}

void replays_dealloc(PyObject *o) {
    auto *self = (Replays *)o;
    if (self->entries)
        for (auto &e : *self->entries) Py_DECREF(e.second.owner);
    delete self->entries;
    delete self->order;
    Py_TYPE(o)->tp_free(o);
}

// call(x, out_dtype, tag[, norm_weight, norm_bias, eps]) -> the output, or None where this layout is not kept
PyObject *replays_call(PyObject *o, PyObject *const *args, Py_ssize_t n) {
    auto *self = (Replays *)o;
    if (n != 3 && n != 6) Py_RETURN_NONE;
    const at::Tensor *x = plain(args[0]);
    if (!x || modes_active()) Py_RETURN_NONE;
    const int64_t tag = PyLong_AsLongLong(args[2]);
    const double eps = n == 6 ? PyFloat_AsDouble(args[5]) : 0.0;
    if (PyErr_Occurred()) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    Key k;
    if (!make_key(*x, args[1], tag, n == 6, n == 6 ? args[3] : nullptr, n == 6 ? args[4] : nullptr, eps, &k)) Py_RETURN_NONE;
    const auto it = self->entries->find(k);
    if (it == self->entries->end()) Py_RETURN_NONE;
    try {
        // the plan outlives this call whatever runs meanwhile, and its owner is released however the call ends
        const THPObjectPtr owner(Py_NewRef(it->second.owner));
        const kea_project_plan *plan = it->second.plan;
        const int64_t need = it->second.need;
        const bool transposed = it->second.transposed;
        const auto device = x->device();
        at::Tensor y = at::empty(it->second.shape, at::TensorOptions().device(device).dtype((at::ScalarType)k.out_dtype));
        at::Tensor ws = at::empty({need}, at::TensorOptions().device(device).dtype(at::kByte));
        const int rc = lib.project_launch(plan, x->const_data_ptr(), y.mutable_data_ptr(), ws.mutable_data_ptr(), need,
                                          stream_of(device));
        if (rc != 0) Py_RETURN_NONE;  // the Python path reports it
        return THPVariable_Wrap(transposed ? y.transpose(1, 2) : std::move(y));
    } catch (const std::exception &) {
        Py_RETURN_NONE;  // (an allocation failed: the Python path raises torch's error)
    }
}

// keep(x, out_dtype, tag, norm_weight, norm_bias, eps, owner, plan, need, shape, transposed)
PyObject *replays_keep(PyObject *o, PyObject *args) {
    auto *self = (Replays *)o;
    PyObject *xo, *dtype, *nw, *nb, *owner, *shape;
    long long tag, need;
    unsigned long long plan;
    double eps;
    int transposed;
    if (!PyArg_ParseTuple(args, "OOLOOdOKLO!p", &xo, &dtype, &tag, &nw, &nb, &eps, &owner, &plan, &need, &PyTuple_Type, &shape,
                          &transposed))
        return nullptr;
    const at::Tensor *x = plain(xo);
    Key k;
    if (!x || !make_key(*x, dtype, tag, nw != Py_None || nb != Py_None, nw, nb, eps, &k)) Py_RETURN_NONE;
    Entry e{owner, (const kea_project_plan *)plan, need, {}, transposed != 0, {}};
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(shape); ++i) {
        e.shape.push_back(PyLong_AsLongLong(PyTuple_GET_ITEM(shape, i)));
        if (PyErr_Occurred()) return nullptr;
    }
    THPObjectPtr old;  // released last: that may run other code, which may come back here
    try {
        auto it = self->entries->find(k);
        if (it == self->entries->end() && (Py_ssize_t)self->entries->size() >= self->limit) it = self->entries->find(self->order->front());
        if (it != self->entries->end()) {  // replaced, or the oldest makes room
            old = it->second.owner;
            self->order->erase(it->second.order);
            self->entries->erase(it);
        }
        e.order = self->order->insert(self->order->end(), k);
        self->entries->emplace(k, e);
        Py_INCREF(owner);
    } catch (const std::exception &) {
        return PyErr_NoMemory();
    }
    Py_RETURN_NONE;
}

PyMethodDef replays_methods[] = {
    {"call", (PyCFunction)(void (*)())replays_call, METH_FASTCALL, "call(x, out_dtype, tag[, norm_weight, norm_bias, eps])"},
    {"keep", replays_keep, METH_VARARGS, "keep(x, out_dtype, tag, norm_weight, norm_bias, eps, owner, plan, need, shape, transposed)"},
    {nullptr, nullptr, 0, nullptr}};

PyTypeObject ReplaysType = {PyVarObject_HEAD_INIT(nullptr, 0) "kea_native.Replays", sizeof(Replays)};

// ---- quantize and gemm ----

bool as_int(PyObject *o, int64_t *v) {
    *v = PyLong_AsLongLong(o);
    if (!PyErr_Occurred()) return true;
    PyErr_Clear();
    return false;
}

// An optional tensor argument: false where it is neither None nor a plain tensor on `device`.
bool optional(PyObject *o, c10::Device device, const at::Tensor **t) {
    *t = nullptr;
    if (o == Py_None) return true;
    *t = plain(o);
    return *t && (*t)->device() == device;
}

// quantize(x, xb, xt, xk, t, m, k, parts, norm_w, norm_b, eps, silu, qs_dtype, ldq) -> (q, qs) or None. norm_w / norm_b:
// contiguous FP32 tensors on x's device, or None.
PyObject *native_quantize(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != 14) Py_RETURN_NONE;
    const at::Tensor *x = plain(args[0]), *w, *b;
    if (!x || modes_active() || !THPDtype_Check(args[12])) Py_RETURN_NONE;
    int64_t xb, xt, xk, t, m, k, parts, silu, ldq;
    if (!as_int(args[1], &xb) || !as_int(args[2], &xt) || !as_int(args[3], &xk) || !as_int(args[4], &t) ||
        !as_int(args[5], &m) || !as_int(args[6], &k) || !as_int(args[7], &parts) || !as_int(args[11], &silu) ||
        !as_int(args[13], &ldq) || !optional(args[8], x->device(), &w) || !optional(args[9], x->device(), &b))
        Py_RETURN_NONE;
    const double eps = PyFloat_AsDouble(args[10]);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    const int xc = code_of(x->scalar_type());
    const auto qs_type = ((THPDtype *)args[12])->scalar_type;
    const int qc = code_of(qs_type);
    if ((xc != KEA_F32 && xc != KEA_F16) || (qc != KEA_F32 && qc != KEA_F16) || m < 1 || k < 1 || t < 1 || xb < 0 ||
        xt < 0 || xk < 0 || parts < 1 || parts > 3 || m > INT32_MAX || k > 8192 || ldq < k || (w != nullptr) != (b != nullptr))
        Py_RETURN_NONE;
    for (const at::Tensor *v : {w, b})
        if (v && (v->scalar_type() != at::kFloat || !v->is_contiguous() || v->numel() != k)) Py_RETURN_NONE;
    // the furthest element any row reads lies in x's storage (each factor is below 2^31 or a stride of x's own storage)
    const int64_t bl = (m - 1) / t, rl = (m - 1) % t;
    const int64_t limit = (int64_t)(x->storage().nbytes() / x->element_size());
    if (xb > limit || xt > limit || xk > limit) Py_RETURN_NONE;
    __int128 far = (__int128)bl * xb + (__int128)rl * xt;
    if (bl >= 1) {
        const __int128 other = (__int128)(bl - 1) * xb + (__int128)(t - 1) * xt;
        if (other > far) far = other;
    }
    far += (__int128)(k - 1) * xk + x->storage_offset();
    if (far >= limit) Py_RETURN_NONE;
    try {
        const auto device = x->device();
        at::Tensor q = at::empty({parts, m, ldq}, at::TensorOptions().device(device).dtype(at::kChar));
        at::Tensor qs = at::empty({parts, m}, at::TensorOptions().device(device).dtype(qs_type));
        const int rc = lib.quantize(x->const_data_ptr(), xc, xb, xt, xk, t, m, k, (int)parts,
                                    w ? (const float *)w->const_data_ptr() : nullptr,
                                    b ? (const float *)b->const_data_ptr() : nullptr, (float)eps, (int)(silu != 0),
                                    (int8_t *)q.mutable_data_ptr(), ldq, qs.mutable_data_ptr(), qc, stream_of(device));
        if (rc != 0) Py_RETURN_NONE;
        PyObject *qo = THPVariable_Wrap(std::move(q)), *so = THPVariable_Wrap(std::move(qs));
        PyObject *r = qo && so ? PyTuple_Pack(2, qo, so) : nullptr;
        Py_XDECREF(qo);
        Py_XDECREF(so);
        return r;
    } catch (const std::exception &) {
        Py_RETURN_NONE;
    }
}

// gemm(wbits, q, qs, words, words_needed, n, k, wscale, bias, y, acc_out, m, flags, split, tile, ws_group, workspace_bytes,
// residual, factor) -> True where the checks of lowbit.gemm hold and the launch went out
PyObject *native_gemm(PyObject *, PyObject *const *args, Py_ssize_t count) {
    if (count != 19) Py_RETURN_FALSE;
    const at::Tensor *q = plain(args[1]);
    if (!q || modes_active()) Py_RETURN_FALSE;
    const auto device = q->device();
    const at::Tensor *qs, *words, *ws, *bias, *y, *acc, *res;
    int64_t wbits, words_needed, n, k, m, flags, split, tile, group, need;
    if (!optional(args[2], device, &qs) || !optional(args[3], device, &words) || !optional(args[7], device, &ws) ||
        !optional(args[8], device, &bias) || !optional(args[9], device, &y) || !optional(args[10], device, &acc) ||
        !optional(args[17], device, &res) || !as_int(args[0], &wbits) || !as_int(args[4], &words_needed) ||
        !as_int(args[5], &n) || !as_int(args[6], &k) || !as_int(args[11], &m) || !as_int(args[12], &flags) ||
        !as_int(args[13], &split) || !as_int(args[14], &tile) || !as_int(args[15], &group) || !as_int(args[16], &need))
        Py_RETURN_FALSE;
    const double factor = PyFloat_AsDouble(args[18]);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        Py_RETURN_FALSE;
    }
    if (!qs || !words || !ws || (!y && !acc) || (res && !y)) Py_RETURN_FALSE;
    if (q->scalar_type() != at::kChar || q->dim() != 3 || q->stride(2) != 1 || q->stride(1) != q->size(2)) Py_RETURN_FALSE;
    const int64_t parts = q->size(0), ldq = q->size(2);
    const int sc = code_of(qs->scalar_type()), wc = code_of(ws->scalar_type()), bc = bias ? code_of(bias->scalar_type()) : KEA_F32;
    const int yc = y ? code_of(y->scalar_type()) : KEA_F32;
    auto scale = [](int c) { return c == KEA_F32 || c == KEA_F16; };
    const int64_t groups = group > 0 ? (k + group - 1) / group : 1, ny = (flags & KEA_FLAG_GLU) ? n / 2 : n;
    if ((wbits != 1 && wbits != 2) || parts < 1 || parts > 3 || n < 1 || k < 1 || m < 1 || m > q->size(1) || group < 0 ||
        !scale(sc) || !scale(wc) || !scale(bc) || yc < 0 || qs->dim() != 2 || qs->size(0) != parts || qs->size(1) < m ||
        qs->stride(1) != 1 || !ws->is_contiguous() || ws->numel() < n * groups ||
        (bias && (!bias->is_contiguous() || bias->numel() != n)) || !words->is_contiguous() ||
        words->numel() * (int64_t)words->element_size() < 4 * words_needed ||
        (y && (y->dim() != 2 || y->size(0) < m || y->size(1) < ny || y->stride(1) != 1)) ||
        (acc && (acc->scalar_type() != at::kInt || acc->dim() != 3 || acc->size(0) != parts || acc->size(1) != m ||
                 acc->size(2) < n || acc->stride(2) != 1 || acc->stride(0) != m * acc->stride(1))) ||
        (res && (res->scalar_type() != at::kFloat || res->dim() != 2 || res->size(0) < m || res->size(1) < n ||
                 res->stride(1) != 1)))
        Py_RETURN_FALSE;
    try {
        at::Tensor space;
        if (need > 0) space = at::empty({need}, at::TensorOptions().device(device).dtype(at::kByte));
        void *sp = need > 0 ? space.mutable_data_ptr() : nullptr;
        auto run = [&](auto fn, auto... tail) {
            return fn((int)wbits, (const int8_t *)q->const_data_ptr(), q->stride(0), ldq, (int)parts, qs->const_data_ptr(), sc,
                      qs->stride(0), (const uint32_t *)words->const_data_ptr(), n, k, ws->const_data_ptr(), wc, group,
                      bias ? bias->const_data_ptr() : nullptr, bc, y ? y->mutable_data_ptr() : nullptr, yc,
                      y ? y->stride(0) : 0, acc ? (int32_t *)acc->mutable_data_ptr() : nullptr, acc ? acc->stride(1) : 0, m,
                      (int)flags, (int)split, (int)tile, sp, need, tail...);
        };
        const int rc = res ? run(lib.gemm_residual, (const float *)res->const_data_ptr(), (int64_t)res->stride(0), (float)factor,
                                 stream_of(device))
                           : run(lib.gemm, stream_of(device));
        if (rc == 0) Py_RETURN_TRUE;
    } catch (const std::exception &) {
    }
    Py_RETURN_FALSE;
}

// bind(project_launch, gemm, gemm_residual, quantize): the library's entry points as integers
PyObject *native_bind(PyObject *, PyObject *args) {
    unsigned long long p, g, r, q;
    if (!PyArg_ParseTuple(args, "KKKK", &p, &g, &r, &q)) return nullptr;
    lib.project_launch = (decltype(lib.project_launch))p;
    lib.gemm = (decltype(lib.gemm))g;
    lib.gemm_residual = (decltype(lib.gemm_residual))r;
    lib.quantize = (decltype(lib.quantize))q;
    Py_RETURN_NONE;
}

PyMethodDef module_methods[] = {
    {"bind", native_bind, METH_VARARGS, nullptr},
    {"quantize", (PyCFunction)(void (*)())native_quantize, METH_FASTCALL, nullptr},
    {"gemm", (PyCFunction)(void (*)())native_gemm, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "kea_native", nullptr, -1, module_methods};

}  // namespace

PyMODINIT_FUNC PyInit_kea_native(void) {
    ReplaysType.tp_flags = Py_TPFLAGS_DEFAULT;
    ReplaysType.tp_new = replays_new;
    ReplaysType.tp_dealloc = replays_dealloc;
    ReplaysType.tp_methods = replays_methods;
    if (PyType_Ready(&ReplaysType) < 0) return nullptr;
    PyObject *m = PyModule_Create(&module);
    if (m && PyModule_AddObjectRef(m, "Replays", (PyObject *)&ReplaysType) < 0) Py_CLEAR(m);
    return m;
}
