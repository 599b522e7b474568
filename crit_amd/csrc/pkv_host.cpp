// The host's share of an append's and a window launch's call in native code: a decode step makes two of these calls a layer,
// and their argument handling in Python (35 questions to tensors, a structure of 60 fields) took as long as queueing the
// kernels. A Python extension module of its own beside libcrit_pkv.so, whose C ABI it calls: that library knows no Python.
//
// Both functions take the common forms only and check them all; any other form, and every error, is None, and the caller goes
// the general way, which says what is wrong. With an entry point of 0 nothing is launched and the filled parameters come back
// as bytes, whatever device the tensors are on.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <cmath>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/crit_pkv.h"

namespace {

// An ordinary strided tensor of this very type: no subclass, nothing wrapped by a transform.
const at::Tensor* tensor(PyObject* x) {
    if (!THPVariable_CheckExact(x)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(x);
    static const c10::DispatchKeySet wrapped({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                              c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
                                              c10::DispatchKey::ZeroTensor});
    if (!t.defined() || t.layout() != at::kStrided || !t.has_storage() || t.key_set().has_any(wrapped)) return nullptr;
    return &t;
}
// ... or None.
bool given(PyObject* x, const at::Tensor*& t) {
    t = nullptr;
    return x == Py_None || (t = tensor(x)) != nullptr;
}
void* address(const at::Tensor* t) { return t ? t->data_ptr() : nullptr; }
template <typename T>
T* address_as(const at::Tensor* t) { return static_cast<T*>(address(t)); }

bool whole(PyObject* x, int64_t lo, int64_t hi, int64_t& to) {      // a Python int (and no bool) of lo .. hi
    if (!PyLong_CheckExact(x)) return false;
    int over = 0;
    to = PyLong_AsLongLongAndOverflow(x, &over);
    return !over && to >= lo && to <= hi;
}
bool real(PyObject* x, double& to) {
    if (!PyFloat_CheckExact(x)) return false;
    to = PyFloat_AS_DOUBLE(x);
    return true;
}

// The E4M3 pools' multipliers: a pair of floats, or a [2][kv_heads] FP32 tensor on `device`.
bool multipliers(PyObject* x, int64_t kv_heads, c10::Device device, float& k, float& v, const at::Tensor*& heads) {
    heads = nullptr, k = v = 1.0f;
    if (PyTuple_CheckExact(x)) {
        double a, b;
        if (PyTuple_GET_SIZE(x) != 2 || !real(PyTuple_GET_ITEM(x, 0), a) || !real(PyTuple_GET_ITEM(x, 1), b)) return false;
        k = (float)a, v = (float)b;
        return true;
    }
    heads = tensor(x);
    return heads && heads->scalar_type() == at::kFloat && heads->dim() == 2 && heads->size(0) == 2 && heads->size(1) == kv_heads &&
           heads->is_contiguous() && heads->device() == device;
}

int float_type(at::ScalarType t) {
    return t == at::kFloat ? CRIT_PKV_F32 : t == at::kBFloat16 ? CRIT_PKV_BF16 : t == at::kHalf ? CRIT_PKV_F16 : -1;
}

template <typename Params>
PyObject* launch(int64_t entry, const Params& p, int64_t stream) {
    if (!entry) return PyBytes_FromStringAndSize(reinterpret_cast<const char*>(&p), sizeof(p));
    int code;
    Py_BEGIN_ALLOW_THREADS
    code = reinterpret_cast<int (*)(const Params*, void*)>(entry)(&p, reinterpret_cast<void*>(stream));
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(code);
}

#define NEED(x) \
    if (!(x)) Py_RETURN_NONE

bool head_width(int64_t d) { return d == 16 || d == 32 || d == 64 || d == 128 || d == 256; }

// attend(entry, stream, launch_state, kind, fp16, q, key_pages, value_pages, tables, rows, starts, firsts, columns, page, counts,
// offsets, tokens, key_scales, value_scales, multipliers, scale, partitions, parents, out, lse, workspace)
PyObject* attend(PyObject*, PyObject* const* x, Py_ssize_t n) {
    NEED(n == 26);
    int64_t entry, stream, state, kind, columns, page, tokens = 0, parts;
    NEED(whole(x[0], INT64_MIN, INT64_MAX, entry) && whole(x[1], INT64_MIN, INT64_MAX, stream) && whole(x[2], INT64_MIN, INT64_MAX, state));
    NEED(whole(x[3], 0, 3, kind));
    const bool fp16 = x[4] == Py_True;
    const at::Tensor *q = tensor(x[5]), *kp = tensor(x[6]), *vp = tensor(x[7]), *tables = tensor(x[8]), *rows = tensor(x[9]),
                     *starts = tensor(x[10]), *firsts = tensor(x[11]), *counts, *offsets, *ks, *vs, *heads, *parents, *out = tensor(x[23]), *lse,
                     *work = tensor(x[25]);
    NEED(q && kp && vp && tables && rows && starts && firsts && out && work && given(x[14], counts) && given(x[15], offsets) &&
         given(x[17], ks) && given(x[18], vs) && given(x[22], parents) && given(x[24], lse));
    NEED(whole(x[12], 1, CRIT_PKV_MAX_COLUMNS, columns) && whole(x[13], 1, INT32_MAX, page) && whole(x[21], 1, INT32_MAX, parts));
    NEED((x[16] == Py_None) == (offsets == nullptr) && (!offsets || whole(x[16], 0, (int64_t)1 << 40, tokens)));
    const c10::Device device = q->device();
    NEED(!entry || device.is_cuda());
    NEED(kp->device() == device && vp->device() == device && tables->device() == device);
    NEED(q->dim() == 3 && kp->dim() >= 2 && vp->dim() >= 2 && tables->dim() == 2 && out->dim() == 3 && starts->dim() >= 1);
    const int64_t hq = q->size(1), d = q->size(2), hkv = kp->size(-2), dv = vp->size(-1), n_rows = starts->size(0);
    NEED(head_width(d) && head_width(dv) && kp->size(-1) == d && hkv > 0 && hq % hkv == 0 && n_rows > 0 && n_rows <= INT32_MAX);
    const at::ScalarType want = fp16 ? at::kHalf : at::kBFloat16;
    NEED(q->scalar_type() == want && q->stride(2) == 1 && (kind != 0 || kp->scalar_type() == want) && (!fp16 || kind == 0));
    NEED((kind >= 2) == (ks != nullptr) && (kind < 2 || vs));
    NEED(tables->scalar_type() == at::kInt && tables->stride(1) == 1 && tables->size(1) <= INT32_MAX);
    NEED((rows->scalar_type() == at::kInt || rows->scalar_type() == at::kLong) && starts->scalar_type() == at::kInt && firsts->scalar_type() == at::kLong);
    NEED((!counts || counts->scalar_type() == at::kInt) && (!offsets || offsets->scalar_type() == at::kInt));
    if (parents)
        NEED((!entry || parents->is_cuda()) && parents->dim() == 1 && parents->stride(0) == 1 && parents->numel() >= q->size(0) &&
             (parents->scalar_type() == at::kInt || parents->scalar_type() == at::kLong) && columns <= 64);
    const int out_dtype = float_type(out->scalar_type());
    NEED(out_dtype >= 0 && out->stride(2) == 1 && out->size(2) == dv && (!lse || (lse->scalar_type() == at::kFloat && lse->is_contiguous())));
    double scale = 0.0;
    NEED(x[20] == Py_None || real(x[20], scale));
    if (x[20] == Py_None) scale = std::pow((double)d, -0.5);
    float km, vm;
    NEED(multipliers(x[19], hkv, device, km, vm, heads));
    // The default piece (piece_size() of an engine without tuned values), a whole number of a wavefront's steps.
    const int64_t wider = d > dv ? d : dv, width = wider == 64 ? 128 : wider, fits = (kind == 0 ? 65536 : 196608) / width / 16 * 16;
    const int64_t block = 4 * (64 / (wider / 8));
    const int64_t piece = ((fits < 256 ? 256 : fits > 2048 ? 2048 : fits) + block - 1) / block * block;
    int64_t states, floats;      // (a mistaken count of tokens or partitions may name more than 64 bits hold)
    NEED(!__builtin_mul_overflow(offsets ? tokens : n_rows * columns, hq, &states) && !__builtin_mul_overflow(states, parts, &states) &&
         !__builtin_mul_overflow(states, dv + 2, &floats));
    NEED(work->scalar_type() == at::kFloat && work->is_contiguous() && work->numel() >= floats);
    float* const base = work->data_ptr<float>();

    crit_pkv_attend_params p = {};
    p.q = address(q), p.key_pages = address(kp), p.value_pages = address(vp);
    p.key_scales = address_as<float>(ks), p.value_scales = address_as<float>(vs), p.head_multipliers = address_as<float>(heads);
    p.tables = address_as<int32_t>(tables), p.rows = address_as<int32_t>(rows), p.starts = address_as<int32_t>(starts);
    p.counts = address_as<int32_t>(counts), p.firsts = address_as<int64_t>(firsts), p.offsets = address_as<int32_t>(offsets);
    p.partial_out = base, p.partial_max = base + states * dv, p.partial_sum = base + states * (dv + 1);
    p.out = address(out), p.lse = address_as<float>(lse);
    if (parents && parents->scalar_type() == at::kInt) p.parents = address_as<int32_t>(parents);
    else p.parents64 = address_as<int64_t>(parents);
    p.q_stride_t = q->stride(0), p.q_stride_h = q->stride(1), p.out_stride_t = out->stride(0), p.out_stride_h = out->stride(1);
    p.table_stride = tables->stride(0);
    p.table_width = (int32_t)tables->size(1), p.n_rows = (int32_t)n_rows, p.columns = (int32_t)columns;
    p.heads = (int32_t)hq, p.kv_heads = (int32_t)hkv, p.head_dim = (int32_t)d, p.value_dim = (int32_t)dv, p.page = (int32_t)page;
    p.kind = (int32_t)kind, p.page_dtype = fp16 ? CRIT_PKV_F16 : CRIT_PKV_BF16, p.out_dtype = out_dtype;
    p.partitions = (int32_t)parts, p.piece = (int32_t)piece;
    p.scale = (float)scale, p.key_multiplier = km, p.value_multiplier = vm;
    p.rows_are_64 = rows->scalar_type() == at::kLong, p.window_tokens = tokens;
    p.launch_state = reinterpret_cast<uint32_t*>(state);
    return launch(entry, p, stream);
}

// write(entry, stream, kind, fp16, keys, values, slots, key_pages, value_pages, key_scales, value_scales, multipliers, rope)
PyObject* write(PyObject*, PyObject* const* x, Py_ssize_t n) {
    NEED(n == 13);
    int64_t entry, stream, kind;
    NEED(whole(x[0], INT64_MIN, INT64_MAX, entry) && whole(x[1], INT64_MIN, INT64_MAX, stream) && whole(x[2], 0, 3, kind));
    const bool fp16 = x[3] == Py_True;
    const at::Tensor *keys = tensor(x[4]), *values = tensor(x[5]), *slots = tensor(x[6]), *kp = tensor(x[7]), *vp = tensor(x[8]), *ks, *vs, *heads;
    NEED(keys && values && slots && kp && vp && given(x[9], ks) && given(x[10], vs));
    const c10::Device device = keys->device();
    NEED(!entry || device.is_cuda());
    NEED(keys->dim() == 3 && values->dim() == 3 && keys->size(0) > 0);
    const int64_t tokens = keys->size(0), hkv = keys->size(1), d = keys->size(2), dv = values->size(2);
    const int in_dtype = float_type(keys->scalar_type());
    NEED(in_dtype >= 0 && values->scalar_type() == keys->scalar_type() && keys->stride(2) == 1 && values->stride(2) == 1);
    NEED(slots->scalar_type() == at::kLong && slots->is_contiguous() && kp->is_contiguous() && vp->is_contiguous());
    NEED((kind >= 2) == (ks != nullptr) && (kind < 2 || vs) && (!fp16 || kind == 0));
    NEED(kind != 0 || kp->scalar_type() == (fp16 ? at::kHalf : at::kBFloat16));
    NEED(hkv <= INT32_MAX && d <= INT32_MAX && dv <= INT32_MAX);
    float km, vm;
    NEED(multipliers(x[11], hkv, device, km, vm, heads));

    crit_pkv_write_params p = {};
    if (x[12] != Py_None) {      // (table, positions)
        NEED(PyTuple_CheckExact(x[12]) && PyTuple_GET_SIZE(x[12]) == 2);
        const at::Tensor *table = tensor(PyTuple_GET_ITEM(x[12], 0)), *positions = tensor(PyTuple_GET_ITEM(x[12], 1));
        NEED(table && positions && (d == 64 || d == 128 || d == 256) && dv <= d);
        NEED(table->scalar_type() == at::kFloat && table->dim() == 2 && table->size(1) == d && table->size(0) > 0 && table->is_contiguous() &&
             table->device() == device);
        NEED(positions->scalar_type() == at::kLong && positions->dim() == 1 && positions->size(0) == tokens && positions->is_contiguous() &&
             positions->device() == device);
        p.rope_table = address_as<float>(table), p.rope_positions = address_as<int64_t>(positions), p.rope_rows = table->size(0);
        p.rope_scale = 1.0f;
    }
    p.keys = address(keys), p.values = address(values), p.slots = address_as<int64_t>(slots);
    p.key_pages = address(kp), p.value_pages = address(vp);
    p.key_scales = address_as<float>(ks), p.value_scales = address_as<float>(vs), p.head_multipliers = address_as<float>(heads);
    p.tokens = tokens, p.key_stride_t = keys->stride(0), p.key_stride_h = keys->stride(1);
    p.value_stride_t = values->stride(0), p.value_stride_h = values->stride(1);
    p.kv_heads = (int32_t)hkv, p.head_dim = (int32_t)d, p.value_dim = (int32_t)dv;
    p.kind = (int32_t)kind, p.page_dtype = fp16 ? CRIT_PKV_F16 : CRIT_PKV_BF16, p.in_dtype = in_dtype;
    p.key_multiplier = km, p.value_multiplier = vm;
    return launch(entry, p, stream);
}

// (What a tensor may throw when it is asked: the general way asks again and says so.)
template <PyObject* (*CALL)(PyObject*, PyObject* const*, Py_ssize_t)>
PyObject* guarded(PyObject* self, PyObject* const* x, Py_ssize_t n) {
    try {
        return CALL(self, x, n);
    } catch (...) {
        Py_RETURN_NONE;
    }
}

PyMethodDef methods[] = {
    {"attend", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(guarded<attend>)), METH_FASTCALL, nullptr},
    {"write", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(guarded<write>)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_pkv_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}   // namespace

PyMODINIT_FUNC PyInit__pkv_host() {
    PyObject* m = PyModule_Create(&module);
    // What it was compiled against: the tensors' layout in memory is torch's, and the structures are the C ABI's.
    if (m && (PyModule_AddStringConstant(m, "torch_version", CRIT_TORCH_VERSION) || PyModule_AddIntConstant(m, "abi_version", CRIT_PKV_ABI_VERSION) ||
              PyModule_AddIntConstant(m, "attend_size", sizeof(crit_pkv_attend_params)) || PyModule_AddIntConstant(m, "write_size", sizeof(crit_pkv_write_params)))) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
