// The host side of the Python functions in mdx/ops.py and mdx/layers.py: argument checks, output and workspace
// allocation, the C ABI call -- in one extension-module function each, so that a call costs the host a few
// microseconds instead of the 15 to 40 that the same steps take as Python statements around ctypes (a decode layer of one
// sequence keeps the GPU busy for 20).  Nothing here computes, synchronises (the sampler's step apart, whose results are
// host values) or falls back: every function ends in libmdx.so or raises.
//
// Functions take their arguments by position (METH_FASTCALL); the signatures with names, defaults and documentation are the
// Python ones.  What the Python statements used to `assert` raises AssertionError, tensors off the GPU and refusals of
// the library raise mdx.MdxError, as before.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/zeros.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/autograd/python_variable.h>
#include <cmath>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <utility>
#include <vector>
#include "../../include/mdx.h"

namespace {

using at::Tensor;

PyObject* g_mdx_error = nullptr;          // mdx.MdxError

struct PyRaise { PyObject* type; std::string text; };
struct PyPending {};                      // a Python exception is already set

[[noreturn]] void raise_mdx(std::string text) { throw PyRaise{g_mdx_error, std::move(text)}; }
[[noreturn]] void raise_assert(const char* text) { throw PyRaise{PyExc_AssertionError, text}; }

#define NEED(cond) do { if (!(cond)) raise_assert(#cond); } while (0)

void check(int rc, const char* what) {
    if (rc == MDX_OK) return;
    const char* msg = mdx_last_error();
    raise_mdx(std::string(what) + " failed (" + std::to_string(rc) + "): " + (msg ? msg : ""));
}

// ---- arguments ----------------------------------------------------------------------------------
const Tensor& tensor(PyObject* o) {
    if (!THPVariable_Check(o)) throw PyRaise{PyExc_TypeError, std::string("expected a tensor, got ") + Py_TYPE(o)->tp_name};
    return THPVariable_Unpack(o);
}
const Tensor& optional_tensor(PyObject* o) {
    static const Tensor none;
    return o == Py_None ? none : tensor(o);
}
int64_t integer(PyObject* o) {
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) throw PyPending{};
    return v;
}
// int(o): what has a value as an integer, a float or a tensor of one element say, is taken for it (towards zero)
template <typename F> auto as_int(PyObject* o, F value) {
    PyObject* whole = PyNumber_Long(o);
    if (!whole) throw PyPending{};
    const auto v = value(whole);
    Py_DECREF(whole);
    if (PyErr_Occurred()) throw PyPending{};
    return v;
}
int64_t to_int(PyObject* o) { return as_int(o, PyLong_AsLongLong); }
uint64_t to_int_mod64(PyObject* o) { return as_int(o, PyLong_AsUnsignedLongLongMask); }
// None or nothing: `otherwise`
int64_t to_int_or(PyObject* o, int64_t otherwise) {
    const int given = PyObject_IsTrue(o);
    if (given < 0) throw PyPending{};
    return given ? to_int(o) : otherwise;
}
double real(PyObject* o) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw PyPending{};
    return v;
}
float scale_or_default(PyObject* o, int64_t d) { return o == Py_None ? (float)(1.0 / std::sqrt((double)d)) : (float)real(o); }

void need_gpu(std::initializer_list<const Tensor*> ts) {
    for (const Tensor* t : ts)
        if (t->defined() && !t->is_cuda()) raise_mdx("mdx ops run on the GPU only: got a tensor on " + t->device().str());
}

int dtype_of(const Tensor& t) {
    switch (t.scalar_type()) {
        case at::kBFloat16: return MDX_BF16;
        case at::kHalf: return MDX_F16;
        case at::kFloat: return MDX_F32;
        default: throw PyRaise{PyExc_KeyError, std::string("dtype ") + c10::toString(t.scalar_type())};
    }
}

Tensor int32_list(const Tensor& t, const char* what) {
    if (t.scalar_type() != at::kInt) raise_mdx(std::string(what) + " must be int32, got " + c10::toString(t.scalar_type()));
    return t.is_contiguous() ? t : t.contiguous();
}

template <typename... I> Tensor make(const Tensor& like, at::ScalarType type, I... sizes) {
    const int64_t s[] = {(int64_t)sizes...};
    return at::empty(s, at::TensorOptions().dtype(type).device(like.device()));
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
void* ptr(const Tensor& t) { return t.data_ptr(); }
void* ptr_or_null(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

PyObject* wrap(Tensor t) { return THPVariable_Wrap(std::move(t)); }
template <typename... T> PyObject* wrap_tuple(T... t) {
    PyObject* items[] = {wrap(std::move(t))...};
    const Py_ssize_t n = sizeof...(T);
    PyObject* tuple = PyTuple_New(n);
    for (Py_ssize_t i = 0; i < n; ++i) PyTuple_SET_ITEM(tuple, i, items[i]);
    return tuple;
}

// A tensor [..., width] as rows: the tensor (a copy where no row stride describes it), their number and stride.
struct Rows { Tensor t; int64_t n, stride; };
Rows rows_of(const Tensor& x, int64_t width) {
    if (x.dim() == 2) return {x, x.size(0), x.stride(0)};
    if (x.is_contiguous()) return {x, width ? x.numel() / width : 0, width};
    Tensor r = x.reshape({-1, width});
    return {r, r.size(0), r.stride(0)};
}

template <typename F> PyObject* guarded(F f) {
    try {
        return f();
    } catch (const PyRaise& e) {
        PyErr_SetString(e.type, e.text.c_str());
    } catch (const PyPending&) {
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
    }
    return nullptr;
}
#define ARGS(count) do { if (n != (count)) { PyErr_Format(PyExc_TypeError, "%s: %d arguments expected, %zd given", __func__, (int)(count), n); return nullptr; } } while (0)

// ---- store_kvcache --------------------------------------------------------------------------------
// [b, s, h, d] as rows [(b s), h, d] (a copy where the first two dimensions do not merge)
Tensor token_rows(const Tensor& t) {
    if (t.size(0) == 1 || t.stride(0) == t.size(1) * t.stride(1))
        return t.as_strided({t.size(0) * t.size(1), t.size(2), t.size(3)}, {t.stride(1), t.stride(2), t.stride(3)});
    return t.flatten(0, 1);
}

// What store() asks of its arguments; the slots as a dense int32 tensor.
Tensor check_store(const Tensor& key, const Tensor& value, const Tensor& k_cache, const Tensor& v_cache, const Tensor& slot_mapping) {
    NEED(key.dim() == 3 && value.dim() == 3);
    const int64_t N = key.size(0), heads = key.size(1), d = key.size(2), D = heads * d;
    NEED(D > 0);
    NEED(key.stride(2) == 1 && value.stride(2) == 1);
    NEED(key.stride(1) == d && value.stride(1) == d);
    NEED(k_cache.dim() > 1 && v_cache.dim() > 1 && k_cache.stride(1) == D && v_cache.stride(1) == D);
    NEED(slot_mapping.numel() == N);
    NEED(key.scalar_type() == value.scalar_type() && key.scalar_type() == k_cache.scalar_type() && key.scalar_type() == v_cache.scalar_type());
    NEED(k_cache.is_contiguous() && v_cache.is_contiguous());
    return int32_list(slot_mapping, "slot_mapping");
}

void store(const Tensor& key, const Tensor& value, const Tensor& k_cache, const Tensor& v_cache, const Tensor& slot_mapping, void* stream) {
    need_gpu({&key, &value, &k_cache, &v_cache, &slot_mapping});
    const Tensor slots = check_store(key, value, k_cache, v_cache, slot_mapping);
    const int64_t N = key.size(0), D = key.size(1) * key.size(2);
    check(mdx_store_kvcache(ptr(key), ptr(value), key.stride(0), value.stride(0), ptr(k_cache), ptr(v_cache),
                            static_cast<const int32_t*>(ptr(slots)), N, D, (int32_t)key.element_size(), k_cache.numel() / D, stream),
          "store_kvcache");
}

// k of four dimensions, and v with it, as rows
void store_maybe4d(const Tensor& k, const Tensor& v, const Tensor& k_cache, const Tensor& v_cache, const Tensor& slot_mapping, void* stream) {
    const bool four = k.dim() == 4;
    NEED(!four || v.dim() == 4);
    store(four ? token_rows(k) : k, four ? token_rows(v) : v, k_cache, v_cache, slot_mapping, stream);
}

PyObject* store_kvcache(PyObject*, PyObject* const* a, Py_ssize_t n) {
    ARGS(5);
    return guarded([&]() -> PyObject* {
        const Tensor& key = tensor(a[0]);
        need_gpu({&key});
        if (key.dim() != 3) throw PyRaise{PyExc_ValueError, "store_kvcache: key must be [N, heads, d]"};
        store(key, tensor(a[1]), tensor(a[2]), tensor(a[3]), tensor(a[4]), stream_of(key));
        Py_RETURN_NONE;
    });
}

PyObject* store_kvcache_maybe4d(PyObject*, PyObject* const* a, Py_ssize_t n) {
    ARGS(5);
    return guarded([&]() -> PyObject* {
        const Tensor& key = tensor(a[0]);
        need_gpu({&key});
        store_maybe4d(key, tensor(a[1]), tensor(a[2]), tensor(a[3]), tensor(a[4]), stream_of(key));
        Py_RETURN_NONE;
    });
}

// ---- the launches either side of attention ----------------------------------------------------------
// qkv, q_weight, k_weight, eps, cos, sin, positions, Hq, Hkv, d, k_cache | None, v_cache | None, slot_mapping | None, want_k
PyObject* qk_norm_rope_store(PyObject*, PyObject* const* a, Py_ssize_t n) {
    ARGS(14);
    return guarded([&]() -> PyObject* {
        const Tensor &qkv = tensor(a[0]), &qw = tensor(a[1]), &kw = tensor(a[2]), &cos = tensor(a[4]), &sin = tensor(a[5]), &positions = tensor(a[6]);
        const Tensor &k_cache = optional_tensor(a[10]), &v_cache = optional_tensor(a[11]), &slot_mapping = optional_tensor(a[12]);
        const int64_t hq = integer(a[7]), hkv = integer(a[8]), d = integer(a[9]);
        const bool want_k = PyObject_IsTrue(a[13]) == 1;
        need_gpu({&qkv, &qw, &kw, &cos, &sin, &positions, &k_cache, &v_cache, &slot_mapping});
        const int64_t width = (hq + 2 * hkv) * d;
        NEED(qkv.dim() >= 1 && qkv.size(-1) == width && qkv.stride(-1) == 1);
        const Rows x = rows_of(qkv, width);
        NEED(positions.numel() == x.n && positions.scalar_type() == at::kLong && cos.scalar_type() == at::kFloat && sin.scalar_type() == at::kFloat);
        const Tensor pos = positions.is_contiguous() ? positions : positions.contiguous();
        std::vector<int64_t> shape(qkv.sizes().begin(), qkv.sizes().end() - 1);
        shape.push_back(hq);
        shape.push_back(d);
        const auto options = at::TensorOptions().dtype(qkv.scalar_type()).device(qkv.device());
        Tensor q = at::empty(shape, options), k;
        shape[shape.size() - 2] = hkv;
        if (want_k) k = at::empty(shape, options);
        const bool caches = k_cache.defined() && k_cache.numel() > 0;
        Tensor slots;
        int64_t num_slots = 0;
        if (caches) {
            NEED(v_cache.defined() && k_cache.is_contiguous() && v_cache.is_contiguous());
            NEED(slot_mapping.defined() && slot_mapping.numel() == x.n);
            slots = int32_list(slot_mapping, "slot_mapping");
            NEED(hkv > 0 && d > 0);
            num_slots = k_cache.numel() / (hkv * d);
        }
        check(mdx_qk_norm_rope_store(ptr(x.t), x.stride, ptr(qw), ptr(kw), (float)real(a[3]), static_cast<const float*>(ptr(cos)),
                                     static_cast<const float*>(ptr(sin)), cos.size(0), static_cast<const int64_t*>(ptr(pos)), ptr(q), hq * d,
                                     ptr_or_null(k), want_k ? hkv * d : 0, caches ? ptr(k_cache) : nullptr, caches ? ptr(v_cache) : nullptr,
                                     static_cast<const int32_t*>(ptr_or_null(slots)), num_slots, x.n, (int32_t)hq, (int32_t)hkv, (int32_t)d,
                                     dtype_of(qkv), stream_of(qkv)),
              "qk_norm_rope_store");
        // v stays where it is: a strided view of qkv
        std::vector<int64_t> strides(qkv.strides().begin(), qkv.strides().end() - 1);
        strides.push_back(d);
        strides.push_back(1);
        Tensor v = qkv.as_strided(shape, strides, qkv.storage_offset() + (hq + hkv) * d);
        PyObject* t = PyTuple_New(3);
        PyTuple_SET_ITEM(t, 0, wrap(std::move(q)));
        if (want_k) PyTuple_SET_ITEM(t, 1, wrap(std::move(k)));
        else { Py_INCREF(Py_None); PyTuple_SET_ITEM(t, 1, Py_None); }
        PyTuple_SET_ITEM(t, 2, wrap(std::move(v)));
        return t;
    });
}

// x, weight, eps, residual | None
PyObject* rms_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
    ARGS(4);
    return guarded([&]() -> PyObject* {
        const Tensor &x = tensor(a[0]), &w = tensor(a[1]), &residual = optional_tensor(a[3]);
        need_gpu({&x, &w, &residual});
        NEED(x.dim() >= 1);
        const int64_t hidden = x.size(-1);
        NEED(x.stride(-1) == 1 && w.dim() == 1 && w.size(0) == hidden && w.is_contiguous() && w.scalar_type() == x.scalar_type());
        const Rows r = rows_of(x, hidden);
        const auto options = at::TensorOptions().dtype(x.scalar_type()).device(x.device());
        Tensor out = at::empty(x.sizes(), options), r_out;
        Rows res{Tensor(), 0, 0};
        if (residual.defined()) {
            NEED(residual.sizes() == x.sizes() && residual.scalar_type() == w.scalar_type() && residual.stride(-1) == 1);
            res = rows_of(residual, hidden);
            r_out = at::empty(x.sizes(), options);
        }
        check(mdx_add_rms_norm(ptr(r.t), r.stride, ptr_or_null(res.t), res.stride, ptr_or_null(r_out), residual.defined() ? hidden : 0, ptr(w),
                               (float)real(a[2]), ptr(out), hidden, r.n, (int32_t)hidden, dtype_of(w), stream_of(x)),
              "rms_norm");
        if (!residual.defined()) return wrap(std::move(out));
        return wrap_tuple(std::move(out), std::move(r_out));
    });
}

PyObject* silu_and_mul(PyObject*, PyObject* const* a, Py_ssize_t n) {
    ARGS(1);
    return guarded([&]() -> PyObject* {
        const Tensor& x = tensor(a[0]);
        need_gpu({&x});
        NEED(x.dim() >= 1 && x.size(-1) % 2 == 0 && x.stride(-1) == 1);
        const int64_t inter = x.size(-1) / 2;
        const Rows r = rows_of(x, 2 * inter);
        std::vector<int64_t> shape(x.sizes().begin(), x.sizes().end());
        shape.back() = inter;
        Tensor out = at::empty(shape, at::TensorOptions().dtype(x.scalar_type()).device(x.device()));
        check(mdx_silu_and_mul(ptr(r.t), r.stride, ptr(out), inter, r.n, (int32_t)inter, dtype_of(x), stream_of(x)), "silu_and_mul");
        return wrap(std::move(out));
    });
}

// ---- linear layers of a decode pass -----------------------------------------------------------------
// The kernels' rows: bf16, 16-byte aligned, dense along k.  (What is not, as a weight that is a view at an odd offset, takes the library's product.)
bool rows_covered(const Rows& r, int64_t k) {
    return r.t.scalar_type() == at::kBFloat16 && r.t.stride(-1) == 1 && r.stride >= k && r.stride % 8 == 0 && reinterpret_cast<uintptr_t>(ptr(r.t)) % 16 == 0;
}

// x and W for the calls whose row strides end below 2^28 elements
bool operands_covered(const Rows& x, const Rows& w, int64_t k) {
    constexpr int64_t kStrides = (int64_t)1 << 28;
    return rows_covered(x, k) && rows_covered(w, k) && x.stride < kStrides && w.stride < kStrides;
}

// x [.., k], w [n, k] -> fp32 partial sums [splits, .., n], or None where the shape is not covered
PyObject* linear_partials(PyObject*, PyObject* const* a, Py_ssize_t n) {
    ARGS(2);
    return guarded([&]() -> PyObject* {
        const Tensor &x = tensor(a[0]), &w = tensor(a[1]);
        need_gpu({&x, &w});
        NEED(x.dim() >= 2 && w.dim() == 2 && x.size(-1) == w.size(1));
        const int64_t k = w.size(1), cols = w.size(0), rows = k ? x.numel() / k : 0;
        const int32_t splits = mdx_decode_linear_splits(rows, cols, k);
        if (splits == 0) Py_RETURN_NONE;
        const Rows r = rows_of(x, k);
        if (!rows_covered(r, k) || !rows_covered(rows_of(w, k), k)) Py_RETURN_NONE;
        std::vector<int64_t> shape{splits};
        shape.insert(shape.end(), x.sizes().begin(), x.sizes().end() - 1);
        shape.push_back(cols);
        Tensor p = at::empty(shape, at::TensorOptions().dtype(at::kFloat).device(x.device()));
        check(mdx_decode_linear_partials(ptr(r.t), r.stride, ptr(w), w.stride(0), static_cast<float*>(ptr(p)), rows, cols, k, stream_of(x)), "linear_partials");
        return wrap(std::move(p));
    });
}

// x [.., k], w [2 n, k] -> silu_and_mul(x . w^T) [.., n], or None where the shape is not covered
PyObject* linear_silu(PyObject*, PyObject* const* a, Py_ssize_t n) {
    ARGS(2);
    return guarded([&]() -> PyObject* {
        const Tensor &x = tensor(a[0]), &w = tensor(a[1]);
        need_gpu({&x, &w});
        NEED(x.dim() >= 2 && w.dim() == 2 && x.size(-1) == w.size(1) && w.size(0) % 2 == 0);
        const int64_t k = w.size(1), cols = w.size(0) / 2, rows = k ? x.numel() / k : 0;
        if (!mdx_decode_linear_silu_supported(rows, cols, k)) Py_RETURN_NONE;
        const Rows r = rows_of(x, k);
        if (!rows_covered(r, k) || !rows_covered(rows_of(w, k), k)) Py_RETURN_NONE;
        std::vector<int64_t> shape(x.sizes().begin(), x.sizes().end());
        shape.back() = cols;
        Tensor y = at::empty(shape, at::TensorOptions().dtype(at::kBFloat16).device(x.device()));
        check(mdx_decode_linear_silu(ptr(r.t), r.stride, ptr(w), w.stride(0), ptr(y), cols, rows, cols, k, stream_of(x)), "linear_silu");
        return wrap(std::move(y));
    });
}

// x [.., k], w [n, k], partials_ok -> the product [.., n] in bf16, or (partials_ok, where that is the faster) its fp32 partial sums
// [splits, .., n]; None where the library's product is the better one or the shape is not covered
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
    ARGS(3);
    return guarded([&]() -> PyObject* {
        const Tensor &x = tensor(a[0]), &w = tensor(a[1]);
        need_gpu({&x, &w});
        NEED(x.dim() >= 2 && w.dim() == 2 && x.size(-1) == w.size(1));
        const int64_t k = w.size(1), cols = w.size(0), rows = k ? x.numel() / k : 0;
        const int32_t splits = mdx_linear_splits(rows, cols, k);
        if (splits < 0) Py_RETURN_NONE;
        const Rows r = rows_of(x, k);
        if (!operands_covered(r, rows_of(w, k), k)) Py_RETURN_NONE;
        const bool cut = splits > 0 && PyObject_IsTrue(a[2]) == 1;
        std::vector<int64_t> shape;
        if (cut) shape.push_back(splits);
        shape.insert(shape.end(), x.sizes().begin(), x.sizes().end() - 1);
        shape.push_back(cols);
        Tensor y = at::empty(shape, at::TensorOptions().dtype(cut ? at::kFloat : at::kBFloat16).device(x.device()));
        if (cut) check(mdx_linear_partials(ptr(r.t), r.stride, ptr(w), w.stride(0), static_cast<float*>(ptr(y)), rows, cols, k, stream_of(x)), "linear");
        else check(mdx_linear(ptr(r.t), r.stride, ptr(w), w.stride(0), ptr(y), cols, rows, cols, k, stream_of(x)), "linear");
        return wrap(std::move(y));
    });
}

// x [.., k], w [2 n, k] -> silu_and_mul(x . w^T) [.., n], or None as above
PyObject* linear_gated(PyObject*, PyObject* const* a, Py_ssize_t n) {
    ARGS(2);
    return guarded([&]() -> PyObject* {
        const Tensor &x = tensor(a[0]), &w = tensor(a[1]);
        need_gpu({&x, &w});
        NEED(x.dim() >= 2 && w.dim() == 2 && x.size(-1) == w.size(1) && w.size(0) % 2 == 0);
        const int64_t k = w.size(1), cols = w.size(0) / 2, rows = k ? x.numel() / k : 0;
        if (!mdx_linear_silu_supported(rows, cols, k)) Py_RETURN_NONE;
        const Rows r = rows_of(x, k);
        if (!operands_covered(r, rows_of(w, k), k)) Py_RETURN_NONE;
        std::vector<int64_t> shape(x.sizes().begin(), x.sizes().end());
        shape.back() = cols;
        Tensor y = at::empty(shape, at::TensorOptions().dtype(at::kBFloat16).device(x.device()));
        check(mdx_linear_silu(ptr(r.t), r.stride, ptr(w), w.stride(0), ptr(y), cols, rows, cols, k, stream_of(x)), "linear_gated");
        return wrap(std::move(y));
    });
}

// x [.., k], w [(hq + 2 hkv) d, k], q/k weights, eps, cos, sin, positions, hq, hkv, d, caches and slots (or None), want_kv
// -> (q [.., hq, d], k, v [.., hkv, d] or None), or None where the shape is not covered
PyObject* linear_qk_norm_rope_store(PyObject*, PyObject* const* a, Py_ssize_t n) {
    ARGS(15);
    return guarded([&]() -> PyObject* {
        const Tensor &x = tensor(a[0]), &w = tensor(a[1]), &qw = tensor(a[2]), &kw = tensor(a[3]), &cos = tensor(a[5]), &sin = tensor(a[6]), &positions = tensor(a[7]);
        const int64_t hq = integer(a[8]), hkv = integer(a[9]), d = integer(a[10]);
        const Tensor &k_cache = optional_tensor(a[11]), &v_cache = optional_tensor(a[12]), &slot_mapping = optional_tensor(a[13]);
        const bool want_kv = PyObject_IsTrue(a[14]) == 1;
        need_gpu({&x, &w, &qw, &kw, &cos, &sin, &positions, &k_cache, &v_cache, &slot_mapping});
        NEED(x.dim() >= 2 && w.dim() == 2 && x.size(-1) == w.size(1) && hq > 0 && hkv > 0 && d > 0 && w.size(0) == (hq + 2 * hkv) * d);
        const int64_t k = w.size(1), rows = k ? x.numel() / k : 0;
        if (!mdx_linear_qk_norm_rope_store_supported(rows, (int32_t)hq, (int32_t)hkv, (int32_t)d, k)) Py_RETURN_NONE;
        const Rows r = rows_of(x, k);
        if (!operands_covered(r, rows_of(w, k), k)) Py_RETURN_NONE;
        NEED(qw.scalar_type() == at::kBFloat16 && kw.scalar_type() == at::kBFloat16 && qw.numel() == d && kw.numel() == d && qw.is_contiguous() && kw.is_contiguous());
        NEED(positions.numel() == rows && positions.scalar_type() == at::kLong && cos.scalar_type() == at::kFloat && sin.scalar_type() == at::kFloat);
        const Tensor pos = positions.is_contiguous() ? positions : positions.contiguous();
        const bool caches = k_cache.defined() && k_cache.numel() > 0;
        Tensor slots;
        if (caches) {
            NEED(v_cache.defined() && k_cache.is_contiguous() && v_cache.is_contiguous() && k_cache.scalar_type() == at::kBFloat16 && v_cache.scalar_type() == at::kBFloat16);
            NEED(slot_mapping.defined() && slot_mapping.numel() == rows);
            slots = int32_list(slot_mapping, "slot_mapping");
        }
        std::vector<int64_t> shape(x.sizes().begin(), x.sizes().end() - 1);
        shape.push_back(hq);
        shape.push_back(d);
        const auto options = at::TensorOptions().dtype(at::kBFloat16).device(x.device());
        Tensor q = at::empty(shape, options), ko, vo;
        shape[shape.size() - 2] = hkv;
        if (want_kv) { ko = at::empty(shape, options); vo = at::empty(shape, options); }
        check(mdx_linear_qk_norm_rope_store(ptr(r.t), r.stride, ptr(w), w.stride(0), ptr(qw), ptr(kw), (float)real(a[4]), static_cast<const float*>(ptr(cos)),
                                            static_cast<const float*>(ptr(sin)), cos.size(0), static_cast<const int64_t*>(ptr(pos)), ptr(q), hq * d,
                                            ptr_or_null(ko), hkv * d, ptr_or_null(vo), hkv * d, caches ? ptr(k_cache) : nullptr, caches ? ptr(v_cache) : nullptr,
                                            static_cast<const int32_t*>(ptr_or_null(slots)), caches ? k_cache.numel() / (hkv * d) : 0, rows, (int32_t)hq,
                                            (int32_t)hkv, (int32_t)d, k, stream_of(x)),
              "linear_qk_norm_rope_store");
        PyObject* t = PyTuple_New(3);
        PyTuple_SET_ITEM(t, 0, wrap(std::move(q)));
        for (int i = 1; i < 3; ++i) {
            if (want_kv) PyTuple_SET_ITEM(t, i, wrap(std::move(i == 1 ? ko : vo)));
            else { Py_INCREF(Py_None); PyTuple_SET_ITEM(t, i, Py_None); }
        }
        return t;
    });
}

void need_partials(const Tensor& p) { NEED(p.dim() >= 3 && p.scalar_type() == at::kFloat && p.is_contiguous()); }

// partials [splits, .., hidden], weight, eps, residual [.., hidden] -> normed, new residual
PyObject* rms_norm_partials(PyObject*, PyObject* const* a, Py_ssize_t n) {
    ARGS(4);
    return guarded([&]() -> PyObject* {
        const Tensor &p = tensor(a[0]), &w = tensor(a[1]), &residual = tensor(a[3]);
        need_gpu({&p, &w, &residual});
        need_partials(p);
        const int64_t hidden = p.size(-1);
        NEED(residual.sizes() == p.sizes().slice(1) && residual.stride(-1) == 1 && w.dim() == 1 && w.size(0) == hidden && w.is_contiguous() &&
             w.scalar_type() == residual.scalar_type());
        const Rows res = rows_of(residual, hidden);
        const auto options = at::TensorOptions().dtype(w.scalar_type()).device(p.device());
        Tensor out = at::empty(residual.sizes(), options), r_out = at::empty(residual.sizes(), options);
        check(mdx_add_rms_norm_partials(static_cast<const float*>(ptr(p)), (int32_t)p.size(0), ptr(res.t), res.stride, ptr(r_out), hidden, ptr(w),
                                        (float)real(a[2]), ptr(out), hidden, res.n, (int32_t)hidden, dtype_of(w), stream_of(p)), "rms_norm");
        return wrap_tuple(std::move(out), std::move(r_out));
    });
}

// partials [splits, .., (Hq + 2 Hkv) d], q_weight, k_weight, eps, cos, sin, positions, Hq, Hkv, d, k_cache, v_cache, slot_mapping -> q [.., Hq, d]
PyObject* qk_norm_rope_store_partials(PyObject*, PyObject* const* a, Py_ssize_t n) {
    ARGS(13);
    return guarded([&]() -> PyObject* {
        const Tensor &p = tensor(a[0]), &qw = tensor(a[1]), &kw = tensor(a[2]), &cos = tensor(a[4]), &sin = tensor(a[5]), &positions = tensor(a[6]);
        const Tensor &k_cache = tensor(a[10]), &v_cache = tensor(a[11]), &slot_mapping = tensor(a[12]);
        const int64_t hq = integer(a[7]), hkv = integer(a[8]), d = integer(a[9]);
        need_gpu({&p, &qw, &kw, &cos, &sin, &positions, &k_cache, &v_cache, &slot_mapping});
        need_partials(p);
        const int64_t width = (hq + 2 * hkv) * d;
        NEED(p.size(0) > 0 && hq >= 0 && hkv > 0 && d > 0);
        const int64_t rows = p.numel() / p.size(0) / width;
        NEED(p.size(-1) == width && positions.numel() == rows && positions.scalar_type() == at::kLong && cos.scalar_type() == at::kFloat && sin.scalar_type() == at::kFloat);
        NEED(k_cache.is_contiguous() && v_cache.is_contiguous() && k_cache.scalar_type() == qw.scalar_type() && slot_mapping.numel() == rows);
        const Tensor pos = positions.is_contiguous() ? positions : positions.contiguous(), slots = int32_list(slot_mapping, "slot_mapping");
        std::vector<int64_t> shape(p.sizes().begin() + 1, p.sizes().end() - 1);
        shape.push_back(hq);
        shape.push_back(d);
        Tensor q = at::empty(shape, at::TensorOptions().dtype(qw.scalar_type()).device(p.device()));
        check(mdx_qk_norm_rope_store_partials(static_cast<const float*>(ptr(p)), (int32_t)p.size(0), ptr(qw), ptr(kw), (float)real(a[3]),
                                              static_cast<const float*>(ptr(cos)), static_cast<const float*>(ptr(sin)), cos.size(0),
                                              static_cast<const int64_t*>(ptr(pos)), ptr(q), hq * d, ptr(k_cache), ptr(v_cache),
                                              static_cast<const int32_t*>(ptr(slots)), k_cache.numel() / (hkv * d), rows, (int32_t)hq, (int32_t)hkv,
                                              (int32_t)d, dtype_of(qw), stream_of(p)), "qk_norm_rope_store");
        return wrap(std::move(q));
    });
}

// ---- staircase prefill ------------------------------------------------------------------------------
// The result as [N, Hq, d], or flattened to [N, Hq * d].  With caches, k and v are stored into them too.
struct Caches { const Tensor &k, &v, &slot_mapping; };
Tensor staircase(const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& cu_q_, const Tensor& cu_k_, int64_t S, PyObject* max_seqlen,
                 PyObject* scale, bool flat, const Caches* caches = nullptr) {
    need_gpu({&q_, &k_, &v_, &cu_q_, &cu_k_});
    NEED(q_.dim() == 3 && k_.dim() == 3 && v_.dim() == 3);
    NEED(q_.size(0) == k_.size(0) && q_.size(0) == v_.size(0));
    NEED(k_.size(1) == v_.size(1) && k_.size(2) == v_.size(2));
    NEED(q_.size(2) == k_.size(2));
    NEED(k_.size(1) > 0 && q_.size(1) % k_.size(1) == 0);
    NEED(S >= 1 && S <= 128 && (S & (S - 1)) == 0);
    NEED(q_.scalar_type() == k_.scalar_type() && q_.scalar_type() == v_.scalar_type());
    const int64_t total = q_.size(0), hq = q_.size(1), hkv = k_.size(1), d = q_.size(2);
    // strided views (e.g. slices of a fused QKV projection) are read in place
    const Tensor q = q_.stride(2) == 1 ? q_ : q_.contiguous(), k = k_.stride(2) == 1 ? k_ : k_.contiguous(), v = v_.stride(2) == 1 ? v_ : v_.contiguous();
    Tensor o = flat ? make(q, q.scalar_type(), total, hq * d) : make(q, q.scalar_type(), total, hq, d);
    const Tensor cu_q = int32_list(cu_q_, "cu_seqlens_q"), cu_k = int32_list(cu_k_, "cu_seqlens_k");
    auto call = [&](auto fn, auto... more) {
        return fn(ptr(q), ptr(k), ptr(v), ptr(o), q.stride(0), q.stride(1), k.stride(0), k.stride(1), v.stride(0), v.stride(1), hq * d, d,
                  static_cast<const int32_t*>(ptr(cu_q)), static_cast<const int32_t*>(ptr(cu_k)), (int32_t)(cu_k.numel() - 1),
                  (int32_t)to_int_or(max_seqlen, total), total, (int32_t)hq, (int32_t)hkv, (int32_t)d, (int32_t)S, scale_or_default(scale, d),
                  dtype_of(q), more...);
    };
    if (caches) {
        need_gpu({&caches->k, &caches->v, &caches->slot_mapping});
        const Tensor slots = check_store(k_, v_, caches->k, caches->v, caches->slot_mapping);
        check(call(mdx_staircase_attn_store, ptr(caches->k), ptr(caches->v), static_cast<const int32_t*>(ptr(slots)), caches->k.numel() / (hkv * d), stream_of(q)),
              "attention");
        return o;
    }
    check(call(mdx_staircase_attn_varlen, stream_of(q)),
          "sparse_attn_varlen");
    return o;
}

// q, k, v, cu_seqlens_q, cu_seqlens_k, staircase_size, max_seqlen (None or 0: the token count), softmax_scale | None
PyObject* sparse_attn_varlen(PyObject*, PyObject* const* a, Py_ssize_t n) {
    ARGS(8);
    return guarded([&]() -> PyObject* {
        return wrap(staircase(tensor(a[0]), tensor(a[1]), tensor(a[2]), tensor(a[3]), tensor(a[4]), integer(a[5]), a[6], a[7], false));
    });
}

// ---- paged decode -----------------------------------------------------------------------------------
// The arrival counters of mdx_paged_block_attn_single_launch and of the unmask step that this module keeps: two buffers per device and
// stream, zero when created, left zero by every launch.  Eager launches on one stream run one after the other, so they can
// share one; a HIP graph keeps using the buffer that it was captured with wherever and beside whatever it is replayed, which
// is why captured calls have the other one, and why a buffer, once handed out, is never replaced or freed: it has its full size from the
// start.  (Several graphs captured on one stream share theirs: they run one after the other, or with counters of the caller's.)  None (undefined)
// when the request does not fit it, or while a graph is being captured and that stream has no buffers yet (they could not be
// zeroed outside the graph): the caller then takes the two-launch entry point -- run the forward once on the capture
// stream before capturing.
bool capturing(const Tensor& like) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(static_cast<hipStream_t>(stream_of(like)), &status) != hipSuccess || status != hipStreamCaptureStatusNone;
}
constexpr int64_t kCounterFloats = 64 * 256;   // the single-launch path exists for up to 64 sequences; 256 head groups is far beyond any model
struct KeptCounters { Tensor eager, captured; };
KeptCounters kept_counters_of(const Tensor& like, bool create) {
    static auto* kept = new std::map<std::pair<int, void*>, KeptCounters>();      // (never destroyed: the driver may be gone at exit)
    static std::mutex lock;
    const std::pair<int, void*> key{like.device().index(), stream_of(like)};
    if (key.second == static_cast<void*>(hipStreamPerThread)) return {};          // (one handle for as many streams as there are threads)
    std::lock_guard<std::mutex> guard(lock);
    auto it = kept->find(key);
    if (it != kept->end()) return it->second;
    if (!create) return {};
    const Tensor both = at::zeros({2, kCounterFloats}, at::TensorOptions().dtype(at::kFloat).device(like.device()));
    return kept->emplace(key, KeptCounters{both[0], both[1]}).first->second;
}
Tensor counters_for(const Tensor& like, int64_t bytes, bool captured) {
    if (bytes > kCounterFloats * 4) return Tensor();
    const KeptCounters kept = kept_counters_of(like, !captured);
    return captured ? kept.captured : kept.eager;
}

// The kept counters of calls that can do without: eager ones only.
Tensor eager_counters(const Tensor& like, int64_t bytes) { return capturing(like) ? Tensor() : counters_for(like, bytes, false); }

// a tensor of the device -> the counters kept for the current stream (eager calls', captured calls'), or None
PyObject* kept_counters(PyObject*, PyObject* const* a, Py_ssize_t n) {
    ARGS(1);
    return guarded([&]() -> PyObject* {
        need_gpu({&tensor(a[0])});
        const KeptCounters kept = kept_counters_of(tensor(a[0]), false);
        if (!kept.eager.defined()) Py_RETURN_NONE;
        return wrap_tuple(kept.eager, kept.captured);
    });
}

// counters: None = single launch with this module's counters, False = two launches, a tensor = the caller's.
// The result as [bs, Sq, Hq, d], or flattened to [bs, Sq, Hq * d].
Tensor paged(const Tensor& q_, const Tensor& k_cache, const Tensor& v_cache, const Tensor& lens_, const Tensor& bt_, PyObject* scale,
             PyObject* counters_arg, bool flat, const Tensor* next = nullptr, const Tensor* then = nullptr) {
    need_gpu({&q_, &k_cache, &v_cache, &lens_, &bt_});
    NEED(q_.dim() == 4 && k_cache.dim() == 4 && v_cache.sizes() == k_cache.sizes());
    NEED(q_.scalar_type() == k_cache.scalar_type() && q_.scalar_type() == v_cache.scalar_type());
    const int64_t bs = q_.size(0), sq = q_.size(1), hq = q_.size(2), d = q_.size(3);
    const int64_t num_pages = k_cache.size(0), page = k_cache.size(1), hkv = k_cache.size(2);
    const Tensor q = q_.stride(3) == 1 ? q_ : q_.contiguous();
    NEED(k_cache.stride(3) == 1 && v_cache.strides() == k_cache.strides());
    const Tensor bt = int32_list(bt_, "block_table"), lens = int32_list(lens_, "cache_seqlens");
    NEED(bt.dim() == 2 && bt.size(0) == bs && lens.numel() == bs);
    Tensor o = flat ? make(q, q.scalar_type(), bs, sq, hq * d) : make(q, q.scalar_type(), bs, sq, hq, d);
    const bool f32_arithmetic = q.scalar_type() == at::kFloat || d > 128 || d % 16 != 0;
    const int64_t bytes = f32_arithmetic
        ? mdx_paged_block_attn_f32_workspace_bytes((int32_t)bs, (int32_t)sq, (int32_t)hq, (int32_t)d, (int32_t)bt.size(1), (int32_t)page)
        : mdx_paged_block_attn_workspace_bytes((int32_t)bs, (int32_t)sq, (int32_t)hq, (int32_t)hkv, (int32_t)d, (int32_t)bt.size(1), (int32_t)page);
    const Tensor ws = bytes > 0 ? make(q, at::kByte, bytes) : Tensor();
    Tensor counters;
    if (counters_arg == Py_None) {         // more than 64 sequences never take the single-launch path
        // Launches that may do without (mdx_paged_block_attn_needs_counters) leave the kept buffers out of graphs: two graphs captured on one
        // stream may be replayed beside each other.
        const bool captured = bs <= 64 && capturing(q);
        if (bs <= 64 && (!captured || mdx_paged_block_attn_needs_counters((int32_t)bs, (int32_t)sq, (int32_t)hq, (int32_t)hkv, (int32_t)bt.size(1), (int32_t)page)))
            counters = counters_for(q, mdx_paged_block_attn_counter_bytes((int32_t)bs, (int32_t)hq, (int32_t)hkv), captured);
    } else if (counters_arg != Py_False) {
        counters = tensor(counters_arg);
        NEED(counters.scalar_type() == at::kFloat && counters.is_contiguous() && counters.device() == q.device());
    }
    auto call = [&](auto fn, auto... more) {
        return fn(ptr(q), ptr(o), ptr(k_cache), ptr(v_cache), q.stride(0), q.stride(1), q.stride(2), sq * hq * d, hq * d, d,
                  k_cache.stride(0), k_cache.stride(1), k_cache.stride(2), static_cast<const int32_t*>(ptr(bt)), bt.stride(0),
                  static_cast<const int32_t*>(ptr(lens)), (int32_t)bs, (int32_t)sq, (int32_t)hq, (int32_t)hkv, (int32_t)d, (int32_t)bt.size(1),
                  (int32_t)page, num_pages, scale_or_default(scale, d), dtype_of(q), ptr_or_null(ws), bytes, more...);
    };
    if (next) {                             // (what does not lie in one piece of whole 16 bytes is not read ahead)
        auto bytes_of = [&](const Tensor& t) -> int64_t {
            return t.is_contiguous() && t.device() == q.device() && reinterpret_cast<uintptr_t>(ptr(t)) % 16 == 0 ? t.nbytes() / 16 * 16 : 0;
        };
        const int64_t n0 = bytes_of(*next), n1 = bytes_of(*then);
        check(call(mdx_paged_block_attn_read_ahead, ptr_or_null(counters), counters.defined() ? counters.numel() * 4 : 0, n0 ? ptr(*next) : nullptr, n0,
                   n1 ? ptr(*then) : nullptr, n1, stream_of(q)), "flash_attn_with_kvcache");
        return o;
    }
    check(counters.defined() ? call(mdx_paged_block_attn_single_launch, ptr(counters), counters.numel() * 4, stream_of(q))
                             : call(mdx_paged_block_attn, stream_of(q)),
          "flash_attn_with_kvcache");
    return o;
}

// q, k_cache, v_cache, cache_seqlens, block_table, softmax_scale | None, counters
PyObject* flash_attn_with_kvcache(PyObject*, PyObject* const* a, Py_ssize_t n) {
    ARGS(7);
    return guarded([&]() -> PyObject* {
        return wrap(paged(tensor(a[0]), tensor(a[1]), tensor(a[2]), tensor(a[3]), tensor(a[4]), a[5], a[6], false));
    });
}

// q, k_cache, v_cache, cache_seqlens, block_table, softmax_scale | None, the weights of the two products behind the call, counters
PyObject* flash_attn_with_kvcache_read_ahead(PyObject*, PyObject* const* a, Py_ssize_t n) {
    ARGS(9);
    return guarded([&]() -> PyObject* {
        const Tensor &next = tensor(a[6]), &then = tensor(a[7]);
        return wrap(paged(tensor(a[0]), tensor(a[1]), tensor(a[2]), tensor(a[3]), tensor(a[4]), a[5], a[8], false, &next, &then));
    });
}

// ---- the attention layer --------------------------------------------------------------------------
// q, k, v, k_cache, v_cache, slot_mapping, cu_seqlens_q, cu_seqlens_k, block_size, max_seqlen, scale -> o [N, Hq * d]
PyObject* attention_prefill(PyObject*, PyObject* const* a, Py_ssize_t n) {
    ARGS(11);
    return guarded([&]() -> PyObject* {
        const Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]), &k_cache = tensor(a[3]), &v_cache = tensor(a[4]);
        const bool have_cache = k_cache.numel() > 0 && v_cache.numel() > 0;
        need_gpu({&q});
        const Tensor &cu_q = tensor(a[6]), &cu_k = tensor(a[7]);
        const int64_t S = integer(a[8]);
        if (!have_cache) return wrap(staircase(q, k, v, cu_q, cu_k, S, a[9], a[10], true));
        const Caches caches{k_cache, v_cache, tensor(a[5])};
        return wrap(staircase(q, k, v, cu_q, cu_k, S, a[9], a[10], true, &caches));
    });
}

// q, k, v, k_cache, v_cache, slot_mapping, context_lens, block_tables, scale, counters -> o [bs, Sq, Hq * d]
PyObject* attention_decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
    ARGS(10);
    return guarded([&]() -> PyObject* {
        const Tensor &q = tensor(a[0]), &k_cache = tensor(a[3]), &v_cache = tensor(a[4]);
        if (k_cache.numel() > 0 && v_cache.numel() > 0) {
            need_gpu({&q});
            store_maybe4d(tensor(a[1]), tensor(a[2]), k_cache, v_cache, tensor(a[5]), stream_of(q));
        }
        return wrap(paged(q, k_cache, v_cache, tensor(a[6]), tensor(a[7]), a[8], a[9], true));
    });
}

// ---- unmask step --------------------------------------------------------------------------------------
struct Logits { Tensor t; int64_t rows, vocab, stride; };
Logits logits_of(const Tensor& l_) {
    const Tensor l = l_.stride(-1) == 1 ? l_ : l_.contiguous();
    const int64_t vocab = l.size(-1);
    const Rows r = rows_of(l, vocab);
    return {r.t, r.n, vocab, r.stride};
}

Tensor temperatures_of(const Tensor& t) {
    if (!t.defined()) return t;
    Tensor f = t.scalar_type() == at::kFloat ? t : t.to(at::kFloat);
    return f.is_contiguous() ? f : f.contiguous();
}

// Noise of a step: a tensor, a generator's coordinates, or none.
struct Noise {
    Tensor tensor;
    bool seeded = false;
    uint64_t seed = 0, offset = 0;
    Tensor offset_dev, row_ids;
    const float* data() const { return tensor.defined() ? static_cast<const float*>(ptr(tensor)) : nullptr; }
};

// noise | None, seed | None, offset, offset_dev | None, row_ids | None
Noise noise_of(PyObject* const* a, int64_t rows, int64_t vocab) {
    Noise z;
    const Tensor& t = optional_tensor(a[0]);
    z.seeded = a[1] != Py_None;
    if (t.defined() && z.seeded) raise_assert("either a noise tensor or a seed");
    if (t.defined()) {
        z.tensor = t.reshape({rows, vocab});
        if (z.tensor.scalar_type() != at::kFloat) z.tensor = z.tensor.to(at::kFloat);
        if (!z.tensor.is_contiguous()) z.tensor = z.tensor.contiguous();
    }
    if (z.seeded) {
        z.seed = to_int_mod64(a[1]);
        z.offset = to_int_mod64(a[2]);
        z.offset_dev = optional_tensor(a[3]);
        z.row_ids = optional_tensor(a[4]);
        if (z.offset_dev.defined()) NEED(z.offset_dev.scalar_type() == at::kLong && z.offset_dev.numel() == 1 && z.offset_dev.is_cuda());
        if (z.row_ids.defined()) NEED(z.row_ids.scalar_type() == at::kLong && z.row_ids.numel() == rows && z.row_ids.is_contiguous() && z.row_ids.is_cuda());
    }
    return z;
}

// logits, temperatures | None, noise (5 arguments: see noise_of) -> x0, x0_p
PyObject* confidence_argmax(PyObject*, PyObject* const* a, Py_ssize_t n) {
    ARGS(7);
    return guarded([&]() -> PyObject* {
        const Tensor &logits = tensor(a[0]), temps = optional_tensor(a[1]);
        need_gpu({&logits, &temps, &optional_tensor(a[2])});
        const Logits l = logits_of(logits);
        const Tensor t = temperatures_of(temps);
        int64_t per_temp = 1;
        if (t.defined()) {
            NEED(t.numel() > 0 && l.rows % t.numel() == 0);
            per_temp = l.rows / t.numel();
        }
        const Noise z = noise_of(a + 2, l.rows, l.vocab);
        const auto lead = logits.sizes().slice(0, logits.dim() - 1);
        Tensor x0 = at::empty(lead, at::TensorOptions().dtype(at::kLong).device(logits.device()));
        Tensor x0_p = at::empty(lead, at::TensorOptions().dtype(at::kFloat).device(logits.device()));
        const int64_t bytes = mdx_confidence_argmax_workspace_bytes(l.rows, l.vocab);
        const Tensor ws = bytes > 0 ? make(logits, at::kByte, bytes) : Tensor();
        const float* tp = static_cast<const float*>(ptr_or_null(t));
        int64_t* x0p = static_cast<int64_t*>(ptr(x0));
        float* pp = static_cast<float*>(ptr(x0_p));
        if (z.seeded)
            check(mdx_confidence_argmax_gumbel(ptr(l.t), l.stride, dtype_of(logits), tp, (int32_t)per_temp, z.seed, z.offset,
                                               static_cast<const int64_t*>(ptr_or_null(z.offset_dev)), static_cast<const int64_t*>(ptr_or_null(z.row_ids)),
                                               x0p, pp, l.rows, l.vocab, ptr_or_null(ws), bytes, stream_of(logits)), "confidence_argmax");
        else
            check(mdx_confidence_argmax(ptr(l.t), l.stride, dtype_of(logits), tp, (int32_t)per_temp, z.data(), z.data() ? l.vocab : 0, x0p, pp,
                                        l.rows, l.vocab, ptr_or_null(ws), bytes, stream_of(logits)), "confidence_argmax");
        return wrap_tuple(std::move(x0), std::move(x0_p));
    });
}

// x, weight, temperatures | None, rows_per_temp | None, row_ids | None -> x0, x0_p
PyObject* lm_head_confidence(PyObject*, PyObject* const* a, Py_ssize_t n) {
    ARGS(5);
    return guarded([&]() -> PyObject* {
        const Tensor &x_ = tensor(a[0]), &w = tensor(a[1]), temps = optional_tensor(a[2]), ids = optional_tensor(a[4]);
        need_gpu({&x_, &w, &temps, &ids});
        if (x_.scalar_type() != at::kBFloat16 || w.scalar_type() != at::kBFloat16) raise_assert("lm_head_confidence: bf16 only");
        NEED(x_.dim() >= 1);
        const Tensor x = x_.stride(-1) == 1 ? x_ : x_.contiguous();
        const int64_t hidden = x.size(-1);
        const Rows r = rows_of(x, hidden);
        NEED(w.dim() == 2 && w.stride(1) == 1 && w.size(1) == hidden);
        const int64_t vocab = w.size(0);
        const Tensor t = temperatures_of(temps);
        int64_t per_temp = 1;
        if (t.defined()) {
            if (a[3] == Py_None) {
                NEED(t.numel() > 0 && r.n % t.numel() == 0);
                per_temp = r.n / t.numel();
            } else {
                per_temp = to_int(a[3]);
            }
        }
        if (ids.defined()) NEED(ids.scalar_type() == at::kLong && ids.is_contiguous() && ids.numel() >= r.n);
        const auto lead = x.sizes().slice(0, x.dim() - 1);
        Tensor x0 = at::empty(lead, at::TensorOptions().dtype(at::kLong).device(x.device()));
        Tensor x0_p = at::empty(lead, at::TensorOptions().dtype(at::kFloat).device(x.device()));
        const int64_t bytes = mdx_lm_head_confidence_workspace_bytes(r.n, vocab);
        const Tensor ws = make(x, at::kByte, bytes > 16 ? bytes : 16);
        check(mdx_lm_head_confidence(ptr(r.t), r.stride, ptr(w), w.stride(0), static_cast<const float*>(ptr_or_null(t)), (int32_t)per_temp,
                                     static_cast<const int64_t*>(ptr_or_null(ids)), static_cast<int64_t*>(ptr(x0)), static_cast<float*>(ptr(x0_p)),
                                     r.n, vocab, hidden, ptr(ws), bytes, stream_of(x)), "lm_head_confidence");
        return wrap_tuple(std::move(x0), std::move(x0_p));
    });
}

// `out` may be `logits` itself; undefined: a new tensor.
Tensor filter(const Tensor& logits, int64_t top_k, double top_p, const Tensor& temps, const Tensor& out_) {
    need_gpu({&logits, &temps, &out_});
    const Logits l = logits_of(logits);
    Tensor out = out_.defined() ? out_ : at::empty(logits.sizes(), at::TensorOptions().dtype(logits.scalar_type()).device(logits.device()));
    NEED(out.sizes() == logits.sizes() && out.scalar_type() == logits.scalar_type());
    if (out.stride(-1) != 1) raise_assert("out must have unit stride along the vocabulary");
    const Tensor o2 = out.dim() == 2 ? out : out.view({-1, l.vocab});           // raises if that would need a copy
    const Tensor t = temperatures_of(temps);
    int64_t per_temp = 1;
    if (t.defined()) {
        NEED(t.numel() > 0 && l.rows % t.numel() == 0);
        per_temp = l.rows / t.numel();
    }
    check(mdx_filter_logits(ptr(l.t), l.stride, dtype_of(logits), static_cast<const float*>(ptr_or_null(t)), (int32_t)per_temp, (int32_t)top_k,
                            (float)top_p, ptr(o2), o2.stride(0), l.rows, l.vocab, stream_of(logits)), "filter_logits");
    return out;
}

// logits, top_k, top_p, temperatures | None, out | None
PyObject* filter_logits(PyObject*, PyObject* const* a, Py_ssize_t n) {
    ARGS(5);
    return guarded([&]() -> PyObject* {
        return wrap(filter(tensor(a[0]), to_int(a[1]), real(a[2]), optional_tensor(a[3]), optional_tensor(a[4])));
    });
}

// x0, x0_p, tokens, mask_token_id, threshold, k -> transfer, count
PyObject* select_transfer(PyObject*, PyObject* const* a, Py_ssize_t n) {
    ARGS(6);
    return guarded([&]() -> PyObject* {
        const Tensor &x0 = tensor(a[0]), &p = tensor(a[1]), &tokens = tensor(a[2]);
        need_gpu({&x0, &p, &tokens});
        NEED(tokens.scalar_type() == at::kLong && x0.scalar_type() == at::kLong && p.scalar_type() == at::kFloat);
        NEED(tokens.is_contiguous() && x0.is_contiguous() && p.is_contiguous());
        NEED(tokens.dim() == 2);
        const int64_t bs = tokens.size(0), S = tokens.size(1);
        Tensor transfer = make(tokens, at::kBool, bs, S), count = make(tokens, at::kInt, bs);
        check(mdx_select_transfer(static_cast<const int64_t*>(ptr(x0)), static_cast<const float*>(ptr(p)), static_cast<int64_t*>(ptr(tokens)),
                                  to_int(a[3]), (float)real(a[4]), (int32_t)to_int(a[5]), static_cast<uint8_t*>(ptr(transfer)),
                                  static_cast<int32_t*>(ptr(count)), (int32_t)bs, (int32_t)S, stream_of(tokens)), "select_transfer");
        return wrap_tuple(std::move(transfer), std::move(count));
    });
}

struct Filter { int64_t top_k; double top_p; bool on() const { return top_k > 0 || top_p < 1.0; } };

void step(const Tensor& logits, int64_t bs, int64_t S, int64_t* tokens, int64_t mask_id, float threshold, int32_t k, const Tensor& temps,
          const Filter& f, const Noise& z, int64_t* x0, float* x0_p, uint8_t* transfer, int32_t* count) {
    const Logits l = logits_of(logits);
    NEED(l.rows == bs * S);
    const Tensor t = temperatures_of(temps);
    if (t.defined()) NEED(t.numel() == bs);
    if (f.on()) {
        const int64_t bytes = mdx_unmask_step_filtered_workspace_bytes(l.rows, l.vocab, (int32_t)f.top_k);
        const Tensor ws = make(logits, at::kByte, bytes);
        check(mdx_unmask_step_filtered(ptr(l.t), l.stride, dtype_of(logits), static_cast<const float*>(ptr_or_null(t)), (int32_t)f.top_k, (float)f.top_p,
                                       z.data(), z.data() ? l.vocab : 0, z.seeded ? 1 : 0, z.seed, z.offset,
                                       static_cast<const int64_t*>(ptr_or_null(z.offset_dev)), tokens, mask_id, threshold, k, x0, x0_p, transfer, count,
                                       (int32_t)bs, (int32_t)S, l.vocab, ptr(ws), bytes, stream_of(logits)), "unmask_step");
        return;
    }
    const int64_t bytes = mdx_confidence_argmax_workspace_bytes(l.rows, l.vocab);
    const Tensor ws = bytes > 0 ? make(logits, at::kByte, bytes) : Tensor();
    const bool one = mdx_unmask_step_single_launch_pays((int32_t)bs, (int32_t)S, l.vocab, z.seeded ? 1 : 0) != 0;
    const Tensor counters = one ? eager_counters(logits, mdx_unmask_step_counter_bytes((int32_t)bs, (int32_t)S)) : Tensor();
    check(mdx_unmask_step_single_launch(ptr(l.t), l.stride, dtype_of(logits), static_cast<const float*>(ptr_or_null(t)), z.data(), z.data() ? l.vocab : 0,
                                        z.seeded ? 1 : 0, z.seed, z.offset, static_cast<const int64_t*>(ptr_or_null(z.offset_dev)), tokens, mask_id,
                                        threshold, k, x0, x0_p, transfer, count, (int32_t)bs, (int32_t)S, l.vocab, ptr_or_null(ws), bytes,
                                        ptr_or_null(counters), counters.defined() ? counters.nbytes() : 0, stream_of(logits)), "unmask_step");
}

// logits, tokens, mask_token_id, threshold, k, temperatures | None, top_k, top_p, noise (5: see noise_of) -> x0, x0_p, transfer, count
PyObject* unmask_step(PyObject*, PyObject* const* a, Py_ssize_t n) {
    ARGS(13);
    return guarded([&]() -> PyObject* {
        const Tensor &logits = tensor(a[0]), &tokens = tensor(a[1]), &temps = optional_tensor(a[5]);
        need_gpu({&logits, &tokens, &temps, &optional_tensor(a[8])});
        const Filter f{to_int(a[6]), real(a[7])};
        NEED(tokens.scalar_type() == at::kLong && tokens.is_contiguous() && tokens.dim() == 2);
        const int64_t bs = tokens.size(0), S = tokens.size(1), vocab = logits.size(-1);
        NEED(logits.numel() == bs * S * vocab);
        Noise z = noise_of(a + 8, bs * S, vocab);
        Tensor x0 = make(tokens, at::kLong, bs, S), x0_p = make(tokens, at::kFloat, bs, S);
        Tensor transfer = make(tokens, at::kBool, bs, S), count = make(tokens, at::kInt, bs);
        step(logits, bs, S, static_cast<int64_t*>(ptr(tokens)), to_int(a[2]), (float)real(a[3]), (int32_t)to_int(a[4]), temps, f, z,
             static_cast<int64_t*>(ptr(x0)), static_cast<float*>(ptr(x0_p)), static_cast<uint8_t*>(ptr(transfer)), static_cast<int32_t*>(ptr(count)));
        return wrap_tuple(std::move(x0), std::move(x0_p), std::move(transfer), std::move(count));
    });
}

// The step of the runner's sampler, whose blocks live on the host and whose results are host values.  The selection kernel
// works on the blocks in pinned host memory (the GPU reads and writes a few hundred bytes of it per sequence), so that
// neither an upload nor a download is enqueued and the one wait of the call ends with the results in place.  (As copies, the
// blocks' upload, two downloads, a reduction and its download were six launches and three waits: 40 us of a call.)
//
// logits, temperatures | None, blocks (list), step maps (list), steps (list), mask_token_id, threshold, k, noise (5: see noise_of)
// -> (new blocks, number of committed positions); the step maps are written in place
PyObject* sampler_step(PyObject*, PyObject* const* a, Py_ssize_t n) {
    ARGS(13);
    return guarded([&]() -> PyObject* {
        const Tensor &logits = tensor(a[0]), &temps = optional_tensor(a[1]);
        need_gpu({&logits, &temps, &optional_tensor(a[8])});
        if (!PyList_Check(a[2]) || !PyList_Check(a[3]) || !PyList_Check(a[4])) throw PyRaise{PyExc_TypeError, "sampler_step: lists of blocks, step maps and steps"};
        const int64_t bs = PyList_GET_SIZE(a[2]);
        NEED(bs > 0 && PyList_GET_SIZE(a[3]) == bs && PyList_GET_SIZE(a[4]) == bs);
        const int64_t S = tensor(PyList_GET_ITEM(a[2], 0)).numel(), vocab = logits.size(-1);
        const int64_t flags_at = bs * S * 8, counts_at = flags_at + (bs * S + 3) / 4 * 4, bytes = counts_at + bs * 4;
        Tensor pinned = at::empty({bytes}, at::TensorOptions().dtype(at::kByte).pinned_memory(true));
        char* host = static_cast<char*>(ptr(pinned));
        for (int64_t i = 0; i < bs; ++i) {
            Tensor block = tensor(PyList_GET_ITEM(a[2], i));
            if (!block.is_cpu()) block = block.cpu();
            NEED(block.scalar_type() == at::kLong && block.numel() == S);
            if (!block.is_contiguous()) block = block.contiguous();
            std::memcpy(host + i * S * 8, ptr(block), S * 8);
        }
        const Noise z = noise_of(a + 8, bs * S, vocab);
        const Logits l = logits_of(logits);
        NEED(l.rows == bs * S);
        const Tensor t = temperatures_of(temps);
        if (t.defined()) NEED(t.numel() == bs);
        const int64_t ws_bytes = mdx_unmask_step_host_blocks_workspace_bytes(l.rows, l.vocab);
        const Tensor ws = make(logits, at::kByte, ws_bytes);
        const int64_t counter_bytes = mdx_unmask_step_host_blocks_counter_bytes((int32_t)bs, (int32_t)S);
        const Tensor counters = counter_bytes > 0 ? eager_counters(logits, counter_bytes) : Tensor();   // (the call waits: 0.15 us of three sequences' 40)
        check(mdx_unmask_step_host_blocks_single_launch(ptr(l.t), l.stride, dtype_of(logits), static_cast<const float*>(ptr_or_null(t)), z.data(), z.data() ? l.vocab : 0,
                                          z.seeded ? 1 : 0, z.seed, z.offset, static_cast<const int64_t*>(ptr_or_null(z.offset_dev)),
                                          reinterpret_cast<int64_t*>(host), to_int(a[5]), (float)real(a[6]), (int32_t)to_int(a[7]),
                                          reinterpret_cast<uint8_t*>(host + flags_at), reinterpret_cast<int32_t*>(host + counts_at), (int32_t)bs, (int32_t)S, l.vocab,
                                          ptr(ws), ws_bytes, ptr_or_null(counters), counters.defined() ? counters.nbytes() : 0, stream_of(logits)), "unmask_step");
        hipError_t rc;
        Py_BEGIN_ALLOW_THREADS
        rc = hipStreamSynchronize(static_cast<hipStream_t>(stream_of(logits)));
        Py_END_ALLOW_THREADS
        if (rc != hipSuccess) throw PyRaise{PyExc_RuntimeError, std::string("sampler step: HIP error: ") + hipGetErrorString(rc)};

        const uint8_t* flags = reinterpret_cast<const uint8_t*>(host + flags_at);
        int64_t total = 0;
        for (int64_t i = 0; i < bs; ++i) {
            int32_t c;
            std::memcpy(&c, host + counts_at + 4 * i, 4);
            total += c;
            const Tensor& map = tensor(PyList_GET_ITEM(a[3], i));
            const int64_t at_step = to_int(PyList_GET_ITEM(a[4], i));
            NEED(map.numel() == S);
            if (map.is_cpu() && map.scalar_type() == at::kInt && map.is_contiguous()) {
                int32_t* m = static_cast<int32_t*>(ptr(map));
                for (int64_t p = 0; p < S; ++p) if (flags[i * S + p]) m[p] = (int32_t)at_step;
            } else {
                Tensor mask = at::empty({S}, at::TensorOptions().dtype(at::kBool));
                std::memcpy(ptr(mask), flags + i * S, S);
                map.masked_fill_(mask.to(map.device()).view(map.sizes()), at_step);
            }
        }
        Tensor blocks = at::empty({bs, S}, at::TensorOptions().dtype(at::kLong));
        std::memcpy(ptr(blocks), host, bs * S * 8);
        PyObject* list = PyList_New(bs);
        for (int64_t i = 0; i < bs; ++i) PyList_SET_ITEM(list, i, wrap(blocks.select(0, i)));
        return Py_BuildValue("(NL)", list, (long long)total);
    });
}

#define ENTRY(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    ENTRY(store_kvcache), ENTRY(store_kvcache_maybe4d), ENTRY(qk_norm_rope_store), ENTRY(rms_norm), ENTRY(silu_and_mul), ENTRY(linear), ENTRY(linear_gated), ENTRY(linear_qk_norm_rope_store), ENTRY(linear_partials), ENTRY(linear_silu),
    ENTRY(rms_norm_partials), ENTRY(qk_norm_rope_store_partials), ENTRY(sparse_attn_varlen),
    ENTRY(flash_attn_with_kvcache), ENTRY(flash_attn_with_kvcache_read_ahead), ENTRY(kept_counters), ENTRY(attention_prefill), ENTRY(attention_decode), ENTRY(confidence_argmax), ENTRY(lm_head_confidence),
    ENTRY(filter_logits), ENTRY(select_transfer), ENTRY(unmask_step), ENTRY(sampler_step),
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "mdx._host", "Native host side of mdx.ops and mdx.layers.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
    PyObject* lib = PyImport_ImportModule("mdx._lib");
    if (!lib) return nullptr;
    g_mdx_error = PyObject_GetAttrString(lib, "MdxError");
    Py_DECREF(lib);
    if (!g_mdx_error) return nullptr;
    return PyModule_Create(&module);
}
