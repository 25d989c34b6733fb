// The call path from torch tensors to the C ABI (include/stbl_amd.h) for the calls of a decode or prefill
// step, whose kernels take a few microseconds: stblarge_amd/ops.py's wrappers cost more than that in the
// interpreter (a one-token GEMV 10.5 us a call against 3.5 on the GPU). Each function here takes the
// arguments of one wrapper, and handles the plain case: strided, contiguous, exactly typed device tensors
// of matching shapes. For anything else it returns NotImplemented before doing anything, and the wrapper
// goes its own way, which checks, explains and raises. Outputs are allocated by torch, launches go to the
// current device's current stream, a failure raises _lib.StblError as _lib.check does, and the GIL is
// released around each call into the library, as ctypes does.
//
// The library's functions come from stblarge_amd/_lib.py by address (bind), so both paths use one copy.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include <initializer_list>
#include <vector>

namespace {

using at::Tensor;

// ---- the library ---------------------------------------------------------------------------------------

typedef void *P;
typedef int (*gemv_t)(P, P, P, P, int, int, int, int, P);
typedef int (*gemv_batch_t)(const P *, const P *, const P *, const P *, int, int, int, int, int, P);
typedef void (*mxfp4_batch_t)(const P *, const P *, const P *, int, int, int, P);
typedef int (*expert_ffn_t)(int, P, P, P, int, int, int, float, float, int, int, P, P);
typedef uint64_t (*expert_layout_t)(int, int, int, uint64_t *);
typedef int (*moe_experts_t)(int, P, P, int, int, int, const P *, int, const int *, const float *, int, int, int, float, int,
                             int, P, P);
typedef uint64_t (*moe_work_t)(int, int, int, int);
typedef int (*route_t)(P, P, int, int, int, float, int, P, P, P, P);
typedef int (*gemm_rows_t)(int, int, P, P, P, P, int, int, int, int, int, P, P);
typedef int (*gemm_q_rows_t)(int, int, P, P, P, P, P, int, int, int, int, int, P, P);
typedef uint64_t (*gemm_work_t)(int, int, int);
typedef int (*act_quant_t)(P, int, int, int, int, P, P, P, P);
typedef int (*act_quant_e4m3_t)(P, int, int, int, P, P, P);
typedef int (*last_error_t)(char *, int);

struct Lib {
    gemv_t gemv[2];
    gemv_batch_t gemv_batch[2];
    mxfp4_batch_t mxfp4_batch;
    expert_ffn_t expert_ffn;
    expert_layout_t expert_layout;
    moe_experts_t moe_experts;
    moe_work_t moe_work;
    route_t route;
    gemm_rows_t gemm_rows;
    gemm_q_rows_t gemm_q_rows;
    gemm_work_t gemm_work;
    act_quant_t act_quant;
    act_quant_e4m3_t act_quant_e4m3;
    last_error_t last_error;
    PyObject *error;  // _lib.StblError
} lib;

// ---- arguments -----------------------------------------------------------------------------------------

PyObject *other() { Py_RETURN_NOTIMPLEMENTED; }

// A plain tensor or parameter (no other subclass), or null.
const Tensor *tensor(PyObject *o) { return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }

// A contiguous strided device tensor of type `dt`, of `dims` dimensions if that is not 0, or null.
const Tensor *device(PyObject *o, at::ScalarType dt, int dims) {
    const Tensor *t = tensor(o);
    if (!t || t->layout() != at::kStrided || !t->is_cuda() || t->scalar_type() != dt || !t->is_contiguous()) return nullptr;
    return dims && t->dim() != dims ? nullptr : t;
}

// An int (not a bool, float or numpy scalar), within an int's range.
bool whole(PyObject *o, int *v) {
    if (!PyLong_CheckExact(o)) return false;
    int over = 0;
    const long x = PyLong_AsLongAndOverflow(o, &over);
    if (over || x < INT32_MIN || x > INT32_MAX) return false;
    *v = (int)x;
    return true;
}

bool flag(PyObject *o, int *v) {
    if (!PyBool_Check(o)) return false;
    *v = o == Py_True;
    return true;
}

bool real(PyObject *o, float *v) {
    if (PyFloat_CheckExact(o)) *v = (float)PyFloat_AS_DOUBLE(o);
    else if (int x; whole(o, &x)) *v = (float)x;
    else return false;
    return true;
}

P ptr(const Tensor &t) { return t.data_ptr(); }

P stream() { return (P)c10::hip::getCurrentHIPStream().stream(); }

Tensor empty(at::IntArrayRef shape, at::ScalarType dt, const Tensor &like) {
    return at::empty(shape, at::TensorOptions().dtype(dt).device(like.device()));
}

at::ScalarType out_type(int f32) { return f32 ? at::kFloat : at::kBFloat16; }

// ceil(n / b) x ceil(k / b) fp32 scales of FP8 weights, or k / 32 bytes a row of FP4.
bool weight_shapes(const Tensor &codes, const Tensor &scales, int fmt, int64_t n, int64_t k) {
    if (fmt == 0) return scales.size(0) == n && scales.size(1) == k / 32;
    return scales.size(0) == (n + 127) / 128 && scales.size(1) == (k + 127) / 128;
}

bool weights(PyObject *c, PyObject *s, int fmt, const Tensor **codes, const Tensor **scales, int64_t *n, int64_t *k) {
    *codes = device(c, at::kByte, 2);
    *scales = device(s, fmt == 0 ? at::kByte : at::kFloat, 2);
    if (!*codes || !*scales) return false;
    *n = (*codes)->size(0), *k = (*codes)->size(1) * (fmt == 0 ? 2 : 1);
    return *n <= INT32_MAX && *k <= INT32_MAX && weight_shapes(**codes, **scales, fmt, *n, *k);
}

// Raises as _lib.check does: for a failing status, and for a failure recorded before it. True if it did.
bool failed(int status, const char *what) {
    char msg[256];
    const int code = lib.last_error(msg, sizeof msg);
    if (status == 0 && code == 0) return false;
    PyErr_Format(lib.error, "%s failed: status %d, hipError %d: %s", what, status, code, msg);
    return true;
}

// A tuple of tensors, or null with an error set.
PyObject *tuple(std::initializer_list<const Tensor *> ts) {
    THPObjectPtr all(PyTuple_New((Py_ssize_t)ts.size()));
    if (!all) return nullptr;
    Py_ssize_t i = 0;
    for (const Tensor *t : ts) {
        PyObject *o = THPVariable_Wrap(*t);
        if (!o) return nullptr;
        PyTuple_SET_ITEM(all.get(), i++, o);
    }
    return all.release();
}

#define CALL(status, ...)               \
    do {                                \
        Py_BEGIN_ALLOW_THREADS;         \
        status = __VA_ARGS__;           \
        Py_END_ALLOW_THREADS;           \
    } while (0)

// ---- the wrappers' calls -------------------------------------------------------------------------------

// (fmt, codes, scales, x, out_f32, out)
PyObject *gemv(PyObject *, PyObject *const *a, Py_ssize_t) {
    HANDLE_TH_ERRORS
    int fmt, f32;
    const Tensor *codes, *scales;
    int64_t n, k;
    const Tensor *x = device(a[3], at::kBFloat16, 0);
    if (!whole(a[0], &fmt) || !flag(a[4], &f32) || !weights(a[1], a[2], fmt, &codes, &scales, &n, &k) || !x) return other();
    const int64_t d = x->dim(), m = d == 2 ? x->size(0) : 1;
    if ((d != 2 && d != 1) || m > INT32_MAX || x->size(d - 1) != k) return other();
    Tensor fresh;
    const Tensor *y = &fresh;
    if (a[5] == Py_None) fresh = empty({m, n}, out_type(f32), *codes);
    else if (!(y = tensor(a[5]))) return other();
    int st;
    const P py = ptr(*y), pc = ptr(*codes), ps = ptr(*scales), px = ptr(*x), s = stream();
    CALL(st, lib.gemv[fmt != 0](py, pc, ps, px, (int)m, (int)n, (int)k, f32, s));
    if (failed(st, fmt == 0 ? "gemv_fp4" : "gemv_fp8")) return nullptr;
    if (a[5] != Py_None) return Py_NewRef(a[5]);
    return THPVariable_Wrap(fresh);
    END_HANDLE_TH_ERRORS
}

// (codes, scales, xs, fmt, out_f32, outs): lists
PyObject *gemv_batch(PyObject *, PyObject *const *a, Py_ssize_t) {
    HANDLE_TH_ERRORS
    int fmt, f32;
    if (!PyList_CheckExact(a[0]) || !PyList_CheckExact(a[1]) || !PyList_CheckExact(a[2]) || !whole(a[3], &fmt) || !flag(a[4], &f32) ||
        (fmt != 0 && fmt != 1))
        return other();
    const Py_ssize_t n = PyList_GET_SIZE(a[0]);
    if (n < 1 || n > 64 || PyList_GET_SIZE(a[1]) != n || PyList_GET_SIZE(a[2]) != n) return other();
    const bool given = a[5] != Py_None;
    if (given && (!PyList_CheckExact(a[5]) || PyList_GET_SIZE(a[5]) != n)) return other();
    P c[64], s[64], x[64], y[64];
    int64_t rows = 0, k = 0, m = 0;
    const Tensor *first = nullptr;
    for (Py_ssize_t i = 0; i < n; i++) {
        const Tensor *ci, *si, *xi = device(PyList_GET_ITEM(a[2], i), at::kBFloat16, 0);
        int64_t ri, ki;
        if (!weights(PyList_GET_ITEM(a[0], i), PyList_GET_ITEM(a[1], i), fmt, &ci, &si, &ri, &ki) || !xi) return other();
        const int64_t d = xi->dim(), mi = d == 2 ? xi->size(0) : 1;
        if (i == 0) rows = ri, k = ki, m = mi, first = ci;
        if ((d != 1 && d != 2) || ri != rows || ki != k || mi != m || m > INT32_MAX || xi->size(d - 1) != k) return other();
        c[i] = ptr(*ci), s[i] = ptr(*si), x[i] = ptr(*xi);
        if (given) {
            const Tensor *yi = tensor(PyList_GET_ITEM(a[5], i));
            if (!yi) return other();
            y[i] = ptr(*yi);
        }
    }
    THPObjectPtr ys(given ? Py_NewRef(a[5]) : PyList_New(n));  // freed with its tensors if one cannot be allocated
    if (!ys) return nullptr;
    for (Py_ssize_t i = 0; i < n && !given; i++) {
        const Tensor t = empty({m, rows}, out_type(f32), *first);
        PyObject *o = THPVariable_Wrap(t);
        if (!o) return nullptr;
        y[i] = ptr(t);
        PyList_SET_ITEM(ys.get(), i, o);
    }
    int st;
    const P sp = stream();
    CALL(st, lib.gemv_batch[fmt](y, c, s, x, (int)n, (int)m, (int)rows, (int)k, f32, sp));
    if (failed(st, "gemv_batch")) return nullptr;
    return ys.release();
    END_HANDLE_TH_ERRORS
}

// (ys, ws, xs, rows, k): lists
PyObject *mxfp4_batch(PyObject *, PyObject *const *a, Py_ssize_t) {
    HANDLE_TH_ERRORS
    int rows, k;
    if (!PyList_CheckExact(a[0]) || !PyList_CheckExact(a[1]) || !PyList_CheckExact(a[2]) || !whole(a[3], &rows) || !whole(a[4], &k) ||
        rows < 1 || k < 1)
        return other();
    const Py_ssize_t n = PyList_GET_SIZE(a[0]);
    if (n < 1 || n > 16 || PyList_GET_SIZE(a[1]) != n || PyList_GET_SIZE(a[2]) != n) return other();
    P y[16], w[16], x[16];
    for (Py_ssize_t i = 0; i < n; i++) {
        const Tensor *yi = device(PyList_GET_ITEM(a[0], i), at::kFloat, 0), *wi = device(PyList_GET_ITEM(a[1], i), at::kByte, 0),
                     *xi = device(PyList_GET_ITEM(a[2], i), at::kFloat, 0);
        if (!yi || !wi || !xi || yi->numel() < rows || wi->numel() != (int64_t)rows * (k / 32) * 17 || xi->numel() < k) return other();
        y[i] = ptr(*yi), w[i] = ptr(*wi), x[i] = ptr(*xi);
    }
    const P sp = stream();
    Py_BEGIN_ALLOW_THREADS;
    lib.mxfp4_batch(y, w, x, (int)n, rows, k, sp);
    Py_END_ALLOW_THREADS;
    if (failed(0, "stbl_gemv_mxfp4_batch")) return nullptr;
    return Py_NewRef(a[0]);
    END_HANDLE_TH_ERRORS
}

// (slot, x, fmt, dim, inter, weight, limit, official, out_f32)
PyObject *expert_ffn(PyObject *, PyObject *const *a, Py_ssize_t) {
    HANDLE_TH_ERRORS
    int fmt, dim, inter, official, f32;
    float weight, limit;
    const Tensor *slot = device(a[0], at::kByte, 0), *x = device(a[1], at::kBFloat16, 0);
    if (!slot || !x || !whole(a[2], &fmt) || !whole(a[3], &dim) || !whole(a[4], &inter) || !real(a[5], &weight) ||
        !real(a[6], &limit) || !flag(a[7], &official) || !flag(a[8], &f32) || fmt < 0 || fmt > 2 || dim < 1 || inter < 1)
        return other();
    const int64_t d = x->dim(), m = d == 2 ? x->size(0) : 1;
    if ((d != 1 && d != 2) || m > INT32_MAX || x->size(d - 1) != dim || (uint64_t)slot->numel() < lib.expert_layout(fmt, dim, inter, nullptr))
        return other();
    const Tensor y = empty({m, dim}, out_type(f32), *x), work = empty({m * inter}, at::kBFloat16, *x);
    int st;
    const P py = ptr(y), pl = ptr(*slot), px = ptr(*x), pw = ptr(work), s = stream();
    CALL(st, lib.expert_ffn(fmt, py, pl, px, (int)m, dim, inter, weight, limit, official, f32, pw, s));
    if (failed(st, "expert_ffn")) return nullptr;
    return THPVariable_Wrap(y);
    END_HANDLE_TH_ERRORS
}

// (x, slots, pick, weights, fmt, dim, inter, shared, limit, official, out_f32, work, out, shared_fmt); slots: a
// list of tensors or addresses, pick and weights: lists of t rows of topk
PyObject *moe_experts(PyObject *, PyObject *const *a, Py_ssize_t) {
    HANDLE_TH_ERRORS
    int fmt, dim, inter, shared, official, f32, shared_fmt;
    float limit;
    const Tensor *x = device(a[0], at::kBFloat16, 0);
    if (!x || !PyList_CheckExact(a[1]) || !PyList_CheckExact(a[2]) || !PyList_CheckExact(a[3]) || !whole(a[4], &fmt) ||
        !whole(a[5], &dim) || !whole(a[6], &inter) || !whole(a[7], &shared) || !real(a[8], &limit) || !flag(a[9], &official) ||
        !flag(a[10], &f32) || !whole(a[13], &shared_fmt) || dim < 1 || inter < 1)
        return other();
    const int64_t d = x->dim(), t = d == 2 ? x->size(0) : 1;
    const Py_ssize_t n = PyList_GET_SIZE(a[1]);
    if ((d != 1 && d != 2) || t < 1 || t > 64 || n < 1 || n > 4096 || PyList_GET_SIZE(a[2]) != t || PyList_GET_SIZE(a[3]) != t) return other();
    std::vector<P> slots(n);
    for (Py_ssize_t i = 0; i < n; i++) {
        PyObject *o = PyList_GET_ITEM(a[1], i);
        if (PyLong_CheckExact(o)) {
            slots[i] = PyLong_AsVoidPtr(o);
            if (PyErr_Occurred()) {
                PyErr_Clear();
                return other();
            }
        } else if (const Tensor *s = tensor(o)) {
            slots[i] = ptr(*s);
        } else {
            return other();
        }
    }
    Py_ssize_t topk = -1;
    std::vector<int> pick;
    std::vector<float> w;
    for (int64_t i = 0; i < t; i++) {
        PyObject *p = PyList_GET_ITEM(a[2], i), *q = PyList_GET_ITEM(a[3], i);
        if (!PyList_CheckExact(p) || !PyList_CheckExact(q)) return other();
        if (topk < 0) topk = PyList_GET_SIZE(p);
        if (topk < 1 || topk > 64 || PyList_GET_SIZE(p) != topk || PyList_GET_SIZE(q) != topk) return other();
        for (Py_ssize_t j = 0; j < topk; j++) {
            int v;
            float f;
            if (!whole(PyList_GET_ITEM(p, j), &v) || !real(PyList_GET_ITEM(q, j), &f)) return other();
            pick.push_back(v), w.push_back(f);
        }
    }
    const uint64_t bytes = lib.moe_work((int)t, (int)topk, dim, inter);
    Tensor own;
    const Tensor *work = nullptr;
    if (a[11] != Py_None) {
        if (!(work = tensor(a[11]))) return other();
        if ((uint64_t)work->numel() < bytes) work = nullptr;
    }
    const Tensor *given = nullptr;
    if (a[12] != Py_None && !(given = tensor(a[12]))) return other();
    if (!work) own = empty({(int64_t)bytes}, at::kByte, *x), work = &own;
    Tensor y;
    if (!given) y = empty({t, dim}, out_type(f32), *x);
    int st;
    const P py = ptr(given ? *given : y), px = ptr(*x), pw = ptr(*work), s = stream();
    CALL(st, lib.moe_experts(fmt, py, px, (int)t, dim, inter, slots.data(), (int)n, pick.data(), w.data(), (int)topk, shared,
                             shared_fmt, limit, official, f32, pw, s));
    if (failed(st, "moe_experts")) return nullptr;
    if (given) return Py_NewRef(a[12]);
    return THPVariable_Wrap(y);
    END_HANDLE_TH_ERRORS
}

// (logits, topk, bias, route_scale, score_fn)
PyObject *route(PyObject *, PyObject *const *a, Py_ssize_t) {
    HANDLE_TH_ERRORS
    int topk, fn;
    float scale;
    const Tensor *l = device(a[0], at::kFloat, 2), *bias = nullptr;
    if (!l || !whole(a[1], &topk) || !real(a[3], &scale) || !whole(a[4], &fn) || topk < 1) return other();
    if (a[2] != Py_None && !(bias = device(a[2], at::kFloat, 1))) return other();
    const int64_t t = l->size(0), e = l->size(1);
    if (t > INT32_MAX || e > INT32_MAX) return other();
    const Tensor ids = empty({t, topk}, at::kInt, *l), w = empty({t, topk}, at::kFloat, *l);
    int st;
    const P pl = ptr(*l), pb = bias ? ptr(*bias) : nullptr, pi = ptr(ids), pw = ptr(w), s = stream();
    CALL(st, lib.route(pl, pb, (int)t, (int)e, topk, scale, fn, pi, pw, nullptr, s));
    if (failed(st, "route")) return nullptr;
    return tuple({&ids, &w});
    END_HANDLE_TH_ERRORS
}

constexpr int64_t kMaxRows = 8192;  // of one call

// (packed, codes, scales, x, a_s or None, fmt, act_block, out_f32, work): gemm, or gemm_q with a_s
PyObject *gemm(PyObject *, PyObject *const *a, Py_ssize_t) {
    HANDLE_TH_ERRORS
    int packed, fmt, block, f32;
    const bool q = a[4] != Py_None;
    const Tensor *codes, *scales, *as = nullptr;
    int64_t n, k;
    const Tensor *x = device(a[3], q ? at::kByte : at::kBFloat16, 2);
    if (!x || !whole(a[0], &packed) || !whole(a[5], &fmt) || !whole(a[6], &block) || !flag(a[7], &f32) || block < 1 ||
        !weights(a[1], a[2], fmt, &codes, &scales, &n, &k))
        return other();
    const int64_t m = x->size(0);
    if (m < 1 || m > kMaxRows || x->size(1) != k || k % 128) return other();
    if (q && (!(as = device(a[4], at::kByte, 2)) || as->size(0) != m || as->size(1) != k / block)) return other();
    const uint64_t bytes = lib.gemm_work((int)m, (int)n, (int)k);
    Tensor own;
    const Tensor *work = nullptr;
    if (a[8] != Py_None) {
        if (!(work = tensor(a[8]))) return other();
        if ((uint64_t)work->numel() < bytes) work = nullptr;
    }
    if (!work) own = empty({(int64_t)bytes}, at::kByte, *x), work = &own;
    const Tensor y = empty({m, n}, out_type(f32), *x);
    int st;
    const P py = ptr(y), pc = ptr(*codes), ps = ptr(*scales), px = ptr(*x), pa = q ? ptr(*as) : nullptr, pw = ptr(*work), s = stream();
    if (q) CALL(st, lib.gemm_q_rows(fmt, packed, py, pc, ps, px, pa, (int)m, (int)n, (int)k, block, f32, pw, s));
    else CALL(st, lib.gemm_rows(fmt, packed, py, pc, ps, px, (int)m, (int)n, (int)k, block, f32, pw, s));
    static const char *const names[2][2] = {{"gemm", "gemm_packed"}, {"gemm_q", "gemm_q_packed"}};
    if (failed(st, names[q][packed != 0])) return nullptr;
    return THPVariable_Wrap(y);
    END_HANDLE_TH_ERRORS
}

// (x, block, pow2, want_deq)
PyObject *act_quant(PyObject *, PyObject *const *a, Py_ssize_t) {
    HANDLE_TH_ERRORS
    int block, pow2, want;
    const Tensor *x = device(a[0], at::kBFloat16, 0);
    if (!x || !whole(a[1], &block) || !flag(a[2], &pow2) || !flag(a[3], &want) || block < 1 || x->dim() < 1) return other();
    const int64_t n = x->size(-1), rows = n > 0 ? x->numel() / n : 0;
    if (rows < 1 || rows > INT32_MAX || n > INT32_MAX) return other();
    at::DimVector shape(x->sizes());
    const Tensor codes = empty(shape, at::kByte, *x);
    shape.back() = n / block;
    const Tensor scales = empty(shape, at::kFloat, *x), deq = want ? at::empty_like(*x) : Tensor();
    int st;
    const P px = ptr(*x), pc = ptr(codes), ps = ptr(scales), pd = want ? ptr(deq) : nullptr, s = stream();
    CALL(st, lib.act_quant(px, (int)rows, (int)n, block, pow2, pc, ps, pd, s));
    if (failed(st, "act_quant")) return nullptr;
    return want ? tuple({&codes, &scales, &deq}) : tuple({&codes, &scales});
    END_HANDLE_TH_ERRORS
}

// (x, block)
PyObject *act_quant_e4m3(PyObject *, PyObject *const *a, Py_ssize_t) {
    HANDLE_TH_ERRORS
    int block;
    const Tensor *x = device(a[0], at::kBFloat16, 2);
    if (!x || !whole(a[1], &block) || block < 1) return other();
    const int64_t rows = x->size(0), k = x->size(1);
    if (rows > INT32_MAX || k > INT32_MAX) return other();
    const Tensor codes = empty({rows, k}, at::kByte, *x), scales = empty({rows, k / block}, at::kByte, *x);
    int st;
    const P px = ptr(*x), pc = ptr(codes), ps = ptr(scales), s = stream();
    CALL(st, lib.act_quant_e4m3(px, (int)rows, (int)k, block, pc, ps, s));
    if (failed(st, "act_quant_e4m3")) return nullptr;
    return tuple({&codes, &scales});
    END_HANDLE_TH_ERRORS
}

// (addresses of the library's functions in the order of kNames, StblError)
constexpr const char *kNames[] = {
    "stbl_amd_gemv_fp4", "stbl_amd_gemv_fp8", "stbl_amd_gemv_fp4_batch", "stbl_amd_gemv_fp8_batch", "stbl_gemv_mxfp4_batch",
    "stbl_amd_expert_ffn", "stbl_amd_expert_layout", "stbl_amd_moe_experts", "stbl_amd_moe_work_bytes", "stbl_amd_route",
    "stbl_amd_gemm_rows", "stbl_amd_gemm_q_rows", "stbl_amd_gemm_work_bytes", "stbl_amd_act_quant", "stbl_amd_act_quant_e4m3",
    "stbl_amd_last_error"};
constexpr int kCount = sizeof kNames / sizeof kNames[0];

PyObject *bind(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 2 || !PyList_CheckExact(a[0]) || PyList_GET_SIZE(a[0]) != kCount) {
        PyErr_SetString(PyExc_TypeError, "bind: a list of the functions' addresses, and the error type");
        return nullptr;
    }
    P f[kCount];
    for (int i = 0; i < kCount; i++) {
        f[i] = PyLong_AsVoidPtr(PyList_GET_ITEM(a[0], i));
        if (PyErr_Occurred()) return nullptr;
    }
    Py_XDECREF(lib.error);
    lib = {{(gemv_t)f[0], (gemv_t)f[1]}, {(gemv_batch_t)f[2], (gemv_batch_t)f[3]}, (mxfp4_batch_t)f[4], (expert_ffn_t)f[5],
           (expert_layout_t)f[6], (moe_experts_t)f[7], (moe_work_t)f[8], (route_t)f[9], (gemm_rows_t)f[10], (gemm_q_rows_t)f[11],
           (gemm_work_t)f[12], (act_quant_t)f[13], (act_quant_e4m3_t)f[14], (last_error_t)f[15], Py_NewRef(a[1])};
    Py_RETURN_NONE;
}

PyObject *names(PyObject *, PyObject *const *, Py_ssize_t) {
    PyObject *l = PyList_New(kCount);
    for (int i = 0; l && i < kCount; i++) PyList_SET_ITEM(l, i, PyUnicode_FromString(kNames[i]));
    return l;
}

// Fixed argument counts: a call with another number is a mistake in ops.py.
template <PyObject *(*F)(PyObject *, PyObject *const *, Py_ssize_t), int N>
PyObject *fixed(PyObject *self, PyObject *const *a, Py_ssize_t n) {
    if (n != N) return PyErr_Format(PyExc_TypeError, "%d arguments needed, got %zd", N, n);
    return F(self, a, n);
}

#define METHOD(f, n) {#f, (PyCFunction)(void (*)(void))fixed<f, n>, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {METHOD(bind, 2),        METHOD(names, 0),       METHOD(gemv, 6),  METHOD(gemv_batch, 6),
                         METHOD(mxfp4_batch, 5), METHOD(expert_ffn, 9),  METHOD(moe_experts, 14),
                         METHOD(route, 5),       METHOD(gemm, 9),        METHOD(act_quant, 4),
                         METHOD(act_quant_e4m3, 2), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_bind", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__bind() {
    PyObject *m = PyModule_Create(&module);
    // the Python and torch of the build: both are used by their in-memory layouts, so _lib.py binds no other's
    if (m && PyModule_AddStringConstant(m, "built_for", STBL_BUILT_FOR) < 0) Py_CLEAR(m);
    return m;
}
