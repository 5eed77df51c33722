// Python bindings of the C ABI for torch tensors.
//
// One training iteration on a small batch is some fifteen entries of a few microseconds of GPU time each, and
// feeding them from Python through ctypes (argument objects, tensor checks and the stream looked up in Python)
// took longer than running them: 172 us per iteration against 96 us of kernels (50 graphs, hidden 64).  Here an
// argument is checked and unpacked in C++: a float* or int* parameter takes a contiguous float32 / int32 device
// tensor or None and nothing else, except for the few host pointers of the table below, which take an address as a
// plain integer or an int32 array; the last parameter, the stream, is the current one.  The functions carry the names of the C entries
// without `gnnhip_` and raise GnnHipError on a non-zero status.
//
// The entries are looked up in the library whose path bind() is given, so the module has no link to it.
#include <Python.h>

#include <dlfcn.h>
#include <limits.h>

#include <string>
#include <tuple>
#include <type_traits>
#include <utility>
#include <vector>

#include <ATen/core/Tensor.h>
#include <ATen/Context.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Device.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include "gnnhip.h"

namespace {

PyObject* g_error = nullptr;                 // graphnn_amd._lib.GnnHipError
const char* (*g_last_error)() = nullptr;

// ---------------------------------------------------------------- arguments
bool tensor_pointer(PyObject* o, at::ScalarType type, const char* type_name, const char* name, void** p)
{
    if (THPVariable_Check(o)) {
        const at::Tensor& t = THPVariable_Unpack(o);
        if (t.is_cuda() && t.scalar_type() == type && t.is_contiguous()) {
            *p = t.data_ptr();
            return true;
        }
    } else if (o == Py_None) {
        *p = nullptr;
        return true;
    }
    PyErr_Format(PyExc_ValueError, "%s must be a contiguous %s CUDA tensor", name, type_name);
    return false;
}

// one of the struct module's codes for a 32-bit integer in the host's byte order (no code means bytes)
bool is_int32(const Py_buffer& view)
{
    const char* f = view.format ? view.format : "B";
    const bool standard = *f == '=' || *f == '<';
    if (standard || *f == '@') ++f;
    return view.itemsize == 4 && (*f == 'i' || (standard && *f == 'l')) && !f[1];
}

// an address, or a contiguous int32 array of one dimension with the buffer protocol (a numpy array), which the caller keeps
// alive: of `need` elements at least, writable where the entry writes it
bool host_pointer(PyObject* o, const char* name, long long need, bool written, void** p)
{
    if (PyObject_CheckBuffer(o)) {
        Py_buffer view;
        if (PyObject_GetBuffer(o, &view, PyBUF_FORMAT | PyBUF_ND | (written ? PyBUF_WRITABLE : 0))) return false;
        const bool ok = view.ndim == 1 && is_int32(view) && view.shape[0] >= need;
        *p = view.buf;
        PyBuffer_Release(&view);
        if (!ok) PyErr_Format(PyExc_ValueError, "%s must be an address or an int32 array of %lld entries or more", name, need);
        return ok;
    }
    *p = o == Py_None ? nullptr : PyLong_AsVoidPtr(o);
    return !PyErr_Occurred();
}

template <class T> struct Arg;
template <> struct Arg<int> {
    int v = 0;
    bool take(PyObject* o, const char* name)
    {
        const long l = PyLong_AsLong(o);       // takes anything with __index__
        if (l == -1 && PyErr_Occurred()) return false;
        if (l < INT_MIN || l > INT_MAX) {
            PyErr_Format(PyExc_ValueError, "%s does not fit 32 bits", name);
            return false;
        }
        v = (int)l;
        return true;
    }
};
template <> struct Arg<size_t> {
    size_t v = 0;
    bool take(PyObject* o, const char*) { v = PyLong_AsSize_t(o); return !PyErr_Occurred(); }
};
template <> struct Arg<float> {
    float v = 0.f;
    bool take(PyObject* o, const char*)
    {
        const double d = PyFloat_AsDouble(o);
        v = (float)d;
        return !(d == -1.0 && PyErr_Occurred());
    }
};
template <> struct Arg<float*> {
    float* v = nullptr;
    bool take(PyObject* o, const char* name) { return tensor_pointer(o, at::kFloat, "float32", name, reinterpret_cast<void**>(&v)); }
};
template <> struct Arg<const float*> : Arg<float*> {};
template <> struct Arg<int*> {
    int* v = nullptr;
    bool take(PyObject* o, const char* name) { return tensor_pointer(o, at::kInt, "int32", name, reinterpret_cast<void**>(&v)); }
};
template <> struct Arg<const int*> : Arg<int*> {};
template <> struct Arg<void*> {               // a handle or an address
    void* v = nullptr;
    bool take(PyObject* o, const char*) { v = o == Py_None ? nullptr : PyLong_AsVoidPtr(o); return !PyErr_Occurred(); }
};

PyObject* finish(int rc)
{
    if (rc == GNNHIP_OK) Py_RETURN_NONE;
    if (PyObject* e = PyObject_CallFunction(g_error, "is", rc, g_last_error())) {
        PyErr_SetObject(g_error, e);
        Py_DECREF(e);
    }
    return nullptr;
}

bool current_stream(void** s)
{
    try {
        *s = c10::hip::getCurrentHIPStream().stream();
        return true;
    } catch (const std::exception& e) {      // no usable device
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return false;
    }
}

// ---------------------------------------------------------------- one function per entry
// An entry's parameter names as the C header spells them ("N, C, row_ptr, ..."), for error texts; '@' marks a pointer to
// host memory: a const one is read, one element more than the first parameter says; else one element is written.
std::string nth_name(const char* names, size_t i)
{
    for (; i > 0 && *names; ++names) i -= *names == ',';
    while (*names == ' ' || *names == '@') ++names;
    std::string s;
    for (; *names && *names != ','; ++names) s += *names;
    return s;
}

// index of the parameter marked '@', or past the last one
constexpr size_t host_argument(const char* names)
{
    size_t i = 0;
    for (; *names; ++names) {
        if (*names == '@') return i;
        i += *names == ',';
    }
    return i + 1;
}

template <class Fn, size_t HOST> struct Entry;
template <size_t HOST, class... P> struct Entry<int (*)(P...), HOST> {
    typedef int (*Fn)(P...);
    typedef std::tuple_element_t<0, std::tuple<P...>> First;
    static constexpr size_t kArgs = sizeof...(P) - 1;       // the stream comes last and is not passed

    template <size_t... I>
    static PyObject* call(Fn fn, const char* names, PyObject* const* args, std::index_sequence<I...>)
    {
        std::tuple<Arg<P>...> a;
        size_t failed = kArgs;
        auto one = [&](auto& arg, size_t i, const char* name) {
            if constexpr (HOST < kArgs && std::is_same_v<decltype(arg.v), int*>) {
                constexpr bool kRead = std::is_same_v<std::decay_t<decltype(arg)>, Arg<const int*>>;
                long long need = 1;
                if constexpr (kRead && std::is_same_v<First, int>) need += std::get<0>(a).v;
                if (i == HOST) return host_pointer(args[i], name, need, !kRead, (void**)&arg.v);
            }
            return arg.take(args[i], name);
        };
        auto take = [&](auto& arg, size_t i) {
            // the name is only worked out where an argument is refused
            if (one(arg, i, "argument")) return true;
            failed = i;
            return false;
        };
        if (!(take(std::get<I>(a), I) && ...)) {
            PyErr_Clear();
            auto again = [&](auto& arg, size_t i) { return i != failed || one(arg, i, nth_name(names, i).c_str()); };
            (void)(again(std::get<I>(a), I) && ...);
            return nullptr;
        }
        if (!current_stream(&std::get<kArgs>(a).v)) return nullptr;
        int rc;
        Py_BEGIN_ALLOW_THREADS
        rc = std::apply([fn](auto&... arg) { return fn(arg.v...); }, a);
        Py_END_ALLOW_THREADS
        return finish(rc);
    }

    static PyObject* checked(Fn fn, const char* entry, const char* names, PyObject* const* args, Py_ssize_t n)
    {
        if (!fn) return PyErr_Format(PyExc_RuntimeError, "bind() has not been called");
        if (n != (Py_ssize_t)kArgs) return PyErr_Format(PyExc_TypeError, "%s takes %zu arguments (%zd given)", entry, kArgs, n);
        return call(fn, names, args, std::make_index_sequence<kArgs>());
    }
};

#define GNNHIP_ENTRIES(X)                                                                                                               \
    X(spmm_csr_f32, "m, k, n, nnz, alpha, row_ptr, col_idx, val, B, ldb, beta, out, ldc")                                               \
    X(spmm_csr_planned_f32, "plan, n, alpha, B, ldb, beta, out, ldc")                                                                   \
    X(s2v_level_planned_f32, "plan, C, h_in, W, msg, bias, out")                                                                        \
    X(csr_group_i32, "rows, n, key, key_stride, payload, payload_stride, average, row_ptr, col_idx, val")                               \
    X(csr_group_both_i32, "rows, n, x, x_stride, y, y_stride, row_ptr, col_idx, val, t_row_ptr, t_col_idx, t_val")                      \
    X(csr_consecutive_rows_f32, "rows, row_ptr, average, col_idx, val")                                                                 \
    X(csr_consecutive_rows_host_f32, "rows, @offsets, average, row_ptr, col_idx, val")                                                   \
    X(csr_transpose_f32, "m, k, nnz, row_ptr, col_idx, val, t_row_ptr, t_col_idx, t_val")                                               \
    X(gemm_f32, "transA, transB, m, n, k, alpha, A, lda, B, ldb, beta, out, ldc")                                                       \
    X(s2v_level_f32, "N, C, nnz, row_ptr, col_idx, val, h_in, W, msg, bias, out")                                                       \
    X(s2v_input_f32, "N, K, C, X, W_n2l, msg, h0")                                                                                      \
    X(s2v_input_labels_f32, "N, K, C, label, W_n2l, msg, h0, status")                                                                   \
    X(s2v_readout_f32, "B, N, C, H, Q, s_row_ptr, s_col_idx, s_val, h, W_h1, W_h2, pool, hidden, logits, probs, pred")                  \
    X(s2v_forward_f32, "N, B, K, C, H, Q, L, nnz, a_row_ptr, a_col_idx, a_val, s_row_ptr, s_col_idx, s_val, X, W_n2l, W_conv, W_h1, "   \
                       "W_h2, msg, h_a, h_b, pool, hidden, logits, probs, pred, @which")                                                 \
    X(s2v_forward_planned_f32, "plan, B, K, C, H, Q, L, s_row_ptr, s_col_idx, s_val, X, W_n2l, W_conv, W_h1, W_h2, msg, h_a, h_b, "     \
                               "pool, hidden, logits, probs, pred, @which")                                                              \
    X(s2v_forward_batched_sized_f32, "N, B, K, C, H, Q, L, max_graph_nodes, a_nnz, a_row_ptr, a_col_idx, a_val, s_row_ptr, s_col_idx, "    \
                                     "s_val, X, W_n2l, W_conv, W_h1, W_h2, msg, h_final, pool, hidden, logits, probs, pred, status")    \
    X(s2v_forward_batched_train_sized_f32, "N, B, K, C, H, Q, L, max_graph_nodes, a_nnz, a_row_ptr, a_col_idx, a_val, s_row_ptr, "      \
                                           "s_col_idx, s_val, X, W_n2l, W_conv, W_h1, W_h2, msg, h_levels, pool, hidden, logits, "      \
                                           "probs, pred, status")                                                                       \
    X(s2v_forward_batched_labels_sized_f32, "N, B, K, C, H, Q, L, max_graph_nodes, a_nnz, a_row_ptr, a_col_idx, a_val, s_row_ptr, "     \
                                            "s_col_idx, s_val, label, W_n2l, W_conv, W_h1, W_h2, msg, h_final, pool, hidden, logits, "  \
                                            "probs, pred, status")                                                                      \
    X(unary_f32, "op, x, n, a0, a1")                                                                                                    \
    X(relu_f32, "x, out, n")                                                                                                            \
    X(axpy_f32, "n, a, x, y")                                                                                                           \
    X(axpby_f32, "n, a, x, b, y")                                                                                                       \
    X(add_f32, "n, a, b, out")                                                                                                          \
    X(row_softmax_f32, "x, rows, cols")                                                                                                 \
    X(jagged_softmax_f32, "x, lens, nseg")                                                                                              \
    X(jagged_softmax_static_f32, "x, lens, nseg")                                                                                       \
    X(reduce_f32, "op, x, n, out")                                                                                                      \
    X(row_argmax_f32, "x, rows, cols, out")                                                                                             \
    X(csr_row_argmax_f32, "row_ptr, col_idx, val, rows, out")                                                                           \
    X(cross_entropy_f32, "prob, rows, cols, l_row_ptr, l_col_idx, l_val, out")                                                          \
    X(in_top_k_f32, "pred, label, rows, cols, k, out")                                                                                  \
    X(cast_i32_f32, "src, dst, n")                                                                                                      \
    X(spmm_csr_t_f32, "m, k, n, alpha, row_ptr, col_idx, val, B, ldb, beta, out, ldc")                                                  \
    X(csr_axpy_f32, "rows, cols, a, row_ptr, col_idx, val, dense")                                                                      \
    X(relu_deriv_f32, "n, out, grad, dst")                                                                                              \
    X(jagged_softmax_deriv_f32, "dst, out, grad, lens, nseg")                                                                           \
    X(row_softmax_deriv_f32, "dst, out, grad, rows, cols")                                                                              \
    X(mul_f32, "n, x, y")                                                                                                               \
    X(row_scale_f32, "rows, cols, scale, y")                                                                                            \
    X(s2v_loss_acc_f32, "B, Q, logits, lrow_ptr, lcol, lval, probs, loss_rows, hit, loss, acc")                                         \
    X(s2v_readout_backward_f32, "B, N, C, H, Q, s_row_ptr, s_col_idx, s_val, probs, lrow_ptr, lcol, lval, scale, hidden, W_h1, W_h2, "  \
                                "dlogits, du, g_h")                                                                                     \
    X(s2v_level_backward_f32, "N, C, nnz, t_row_ptr, t_col_idx, t_val, dz, W, u, g_prev, gate_h, acc")                                  \
    X(s2v_grad_gate_f32, "n, h, g, dz, acc, accumulate")

#define GNNHIP_POINTER(name, names) decltype(&gnnhip_##name) p_##name = nullptr;
GNNHIP_ENTRIES(GNNHIP_POINTER)
decltype(&gnnhip_gemm_tn_batch_f32) p_gemm_tn_batch = nullptr;
decltype(&gnnhip_momentum_sgd_batch_f32) p_momentum_sgd_batch = nullptr;
decltype(&gnnhip_adam_batch_f32) p_adam_batch = nullptr;

#define GNNHIP_FUNCTION(name, names)                                                                        \
    PyObject* f_##name(PyObject*, PyObject* const* args, Py_ssize_t n)                                      \
    {                                                                                                       \
        return Entry<decltype(&gnnhip_##name), host_argument(names)>::checked(p_##name, #name, names, args, n);                   \
    }
GNNHIP_ENTRIES(GNNHIP_FUNCTION)

// ---------------------------------------------------------------- entries that take host arrays of device pointers
bool batch_tensor(PyObject* o, const char* name, const at::Tensor** t)
{
    void* p;
    if (!THPVariable_Check(o)) {
        PyErr_Format(PyExc_ValueError, "%s must be a contiguous float32 CUDA tensor", name);
        return false;
    }
    if (!tensor_pointer(o, at::kFloat, "float32", name, &p)) return false;
    *t = &THPVariable_Unpack(o);
    return true;
}

// gemm_tn_batch([(A, B, out), ...], alpha, beta)
PyObject* f_gemm_tn_batch(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    if (n != 3 || !PyList_Check(args[0])) return PyErr_Format(PyExc_TypeError, "gemm_tn_batch(list, alpha, beta)");
    if (!p_gemm_tn_batch) return PyErr_Format(PyExc_RuntimeError, "bind() has not been called");
    const Py_ssize_t count = PyList_GET_SIZE(args[0]);
    Arg<float> alpha, beta;
    if (!alpha.take(args[1], "alpha") || !beta.take(args[2], "beta")) return nullptr;
    std::vector<int> m(count), nn(count), k(count);
    std::vector<const float*> A(count), B(count);
    std::vector<float*> C(count);
    for (Py_ssize_t i = 0; i < count; ++i) {
        PyObject* t = PyList_GET_ITEM(args[0], i);
        if (!PyTuple_Check(t) || PyTuple_GET_SIZE(t) != 3) return PyErr_Format(PyExc_TypeError, "a product is a tuple (A, B, out)");
        const at::Tensor *a, *b, *c;
        if (!batch_tensor(PyTuple_GET_ITEM(t, 0), "A", &a) || !batch_tensor(PyTuple_GET_ITEM(t, 1), "B", &b) ||
            !batch_tensor(PyTuple_GET_ITEM(t, 2), "out", &c))
            return nullptr;
        if (a->dim() != 2 || b->dim() != 2 || c->dim() != 2 || a->size(0) != b->size(0) || c->size(0) != a->size(1) || c->size(1) != b->size(1))
            return PyErr_Format(PyExc_ValueError, "mat dim doesn't match");
        if (a->size(0) > INT_MAX || a->size(1) > INT_MAX || b->size(1) > INT_MAX) return PyErr_Format(PyExc_ValueError, "a product's sizes do not fit 32 bits");
        m[i] = (int)a->size(1), nn[i] = (int)b->size(1), k[i] = (int)a->size(0);
        A[i] = static_cast<const float*>(a->data_ptr()), B[i] = static_cast<const float*>(b->data_ptr()), C[i] = static_cast<float*>(c->data_ptr());
    }
    void* stream;
    if (!current_stream(&stream)) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = p_gemm_tn_batch((int)count, m.data(), nn.data(), k.data(), A.data(), m.data(), B.data(), nn.data(), alpha.v, beta.v, C.data(), nn.data(), stream);
    Py_END_ALLOW_THREADS
    return finish(rc);
}

// device pointers of the tensors of lists[0 .. tables-1] (a list may be None), element counts from the first list
bool pointer_tables(PyObject* const* lists, int tables, Py_ssize_t* count, std::vector<float*>* out, std::vector<size_t>& sizes)
{
    static const char* const names[] = {"w", "g", "m", "v"};
    *count = -1;
    for (int j = 0; j < tables; ++j) {
        if (lists[j] == Py_None) continue;
        if (!PyList_Check(lists[j])) return PyErr_Format(PyExc_TypeError, "lists of tensors are needed") != nullptr;
        const Py_ssize_t n = PyList_GET_SIZE(lists[j]);
        if (*count >= 0 && n != *count) return PyErr_Format(PyExc_ValueError, "the lists differ in length") != nullptr;
        *count = n;
        out[j].resize(n);
        sizes.resize(n);
        for (Py_ssize_t i = 0; i < n; ++i) {
            const at::Tensor* t;
            if (!batch_tensor(PyList_GET_ITEM(lists[j], i), names[j], &t)) return false;
            if (j == 0) sizes[i] = (size_t)t->numel();
            else if ((size_t)t->numel() != sizes[i]) return PyErr_Format(PyExc_ValueError, "the tensors of an update differ in size") != nullptr;
            out[j][i] = static_cast<float*>(t->data_ptr());
        }
    }
    return true;
}

// momentum_sgd_batch(ws, gs, vs or None, lr, momentum, l2)
PyObject* f_momentum_sgd_batch(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    if (n != 6) return PyErr_Format(PyExc_TypeError, "momentum_sgd_batch takes 6 arguments (%zd given)", n);
    if (!p_momentum_sgd_batch) return PyErr_Format(PyExc_RuntimeError, "bind() has not been called");
    Py_ssize_t count;
    std::vector<float*> p[3];
    std::vector<size_t> sizes;
    Arg<float> s[3];
    if (!pointer_tables(args, 3, &count, p, sizes)) return nullptr;
    for (int i = 0; i < 3; ++i)
        if (!s[i].take(args[3 + i], "lr")) return nullptr;
    void* stream;
    if (!current_stream(&stream)) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = p_momentum_sgd_batch((int)count, p[0].data(), p[1].data(), args[2] == Py_None ? nullptr : p[2].data(), sizes.data(), s[0].v, s[1].v, s[2].v, stream);
    Py_END_ALLOW_THREADS
    return finish(rc);
}

// adam_batch(ws, gs, ms, vs, lr, l2, clip_threshold, beta1, beta2, eps, s1, s2)
PyObject* f_adam_batch(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    if (n != 12) return PyErr_Format(PyExc_TypeError, "adam_batch takes 12 arguments (%zd given)", n);
    if (!p_adam_batch) return PyErr_Format(PyExc_RuntimeError, "bind() has not been called");
    Py_ssize_t count;
    std::vector<float*> p[4];
    std::vector<size_t> sizes;
    Arg<float> s[8];
    if (!pointer_tables(args, 4, &count, p, sizes)) return nullptr;
    for (int i = 0; i < 8; ++i)
        if (!s[i].take(args[4 + i], "lr")) return nullptr;
    void* stream;
    if (!current_stream(&stream)) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = p_adam_batch((int)count, p[0].data(), p[1].data(), p[2].data(), p[3].data(), sizes.data(), s[0].v, s[1].v, s[2].v, s[3].v, s[4].v, s[5].v, s[6].v, s[7].v, stream);
    Py_END_ALLOW_THREADS
    return finish(rc);
}

// ---------------------------------------------------------------- helpers
// An uninitialised tensor, as at::empty makes it.  A training iteration asks for seventeen of them, which took a quarter of the
// time that feeding it to the GPU takes; where nothing but the device's backend would see the call (default dispatch keys, no filling of
// fresh memory) the dispatcher is passed by, and several come from one call: 0.94 -> 0.77 us a tensor, 5.6 -> 3.5 six of them.
at::Tensor make_empty(at::Device device, at::ScalarType type, at::IntArrayRef sizes)
{
    const c10::impl::LocalDispatchKeySet keys = c10::impl::tls_local_dispatch_key_set();
    if (device.is_cuda() && keys.included_ == c10::default_included_set && keys.excluded_ == c10::default_excluded_set &&
        !at::globalContext().deterministicAlgorithms())
        return at::detail::empty_cuda(sizes, type, device, std::nullopt);
    return at::empty(sizes, at::TensorOptions().device(device).dtype(type));
}

// empty(where, types, *sizes): an uninitialised tensor, type 'f' (float32) or 'i' (int32) of one to three dimensions, or 'F' (a float32
// matrix); several letters: a tuple of tensors, 'f' and 'i' vectors, 'F' matrices, each taking as many of the sizes.  where: a
// torch.device, or a tensor on whose device they are made.
PyObject* f_empty(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    if (n < 3 || !(THPVariable_Check(args[0]) || THPDevice_Check(args[0])) || !PyUnicode_Check(args[1]))
        return PyErr_Format(PyExc_TypeError, "empty(tensor or device, types, *sizes)");
    Py_ssize_t count;
    const char* types = PyUnicode_AsUTF8AndSize(args[1], &count);
    if (!types) return nullptr;
    auto dims_of = [&](Py_ssize_t k) { return types[k] == 'F' ? 2 : count == 1 ? n - 2 : 1; };
    Py_ssize_t needed = 0;
    for (Py_ssize_t k = 0; k < count; ++k) {
        if (types[k] != 'f' && types[k] != 'i' && types[k] != 'F') return PyErr_Format(PyExc_TypeError, "empty(): types are 'f', 'i' and 'F'");
        needed += dims_of(k);
    }
    if (count == 0 || needed != n - 2 || (count == 1 && needed > 3))
        return PyErr_Format(PyExc_TypeError, "empty(): %zd sizes do not make the tensors of '%s'", n - 2, types);
    HANDLE_TH_ERRORS                          // an allocation that fails raises what torch.empty raises
    const at::Device device = THPVariable_Check(args[0]) ? THPVariable_Unpack(args[0]).device() : reinterpret_cast<THPDevice*>(args[0])->device;
    PyObject* all = count > 1 ? PyTuple_New(count) : nullptr;
    if (count > 1 && !all) return nullptr;
    THPObjectPtr owner(all);
    Py_ssize_t next = 2;
    for (Py_ssize_t k = 0; k < count; ++k) {
        const int dims = (int)dims_of(k);
        int64_t sizes[3];
        for (int d = 0; d < dims; ++d) {
            sizes[d] = PyLong_AsLongLong(args[next++]);
            if (sizes[d] == -1 && PyErr_Occurred()) return nullptr;
        }
        PyObject* t = THPVariable_Wrap(make_empty(device, types[k] == 'i' ? at::kInt : at::kFloat, at::IntArrayRef(sizes, dims)));
        if (!t) return nullptr;
        if (count == 1) return t;
        PyTuple_SET_ITEM(all, k, t);
    }
    return owner.release();
    END_HANDLE_TH_ERRORS
}

// bind(path of libgnnhip.so, GnnHipError)
PyObject* f_bind(PyObject*, PyObject* args)
{
    const char* path;
    PyObject* error;
    if (!PyArg_ParseTuple(args, "sO", &path, &error)) return nullptr;
    void* lib = dlopen(path, RTLD_NOW);
    if (!lib) return PyErr_Format(PyExc_RuntimeError, "%s", dlerror());
    const char* missing = nullptr;
    auto look_up = [&](auto& fn, const char* name) {
        fn = reinterpret_cast<std::remove_reference_t<decltype(fn)>>(dlsym(lib, name));
        if (!fn) missing = name;
    };
#define GNNHIP_LOOK_UP(name, names) look_up(p_##name, "gnnhip_" #name);
    GNNHIP_ENTRIES(GNNHIP_LOOK_UP)
    look_up(p_gemm_tn_batch, "gnnhip_gemm_tn_batch_f32");
    look_up(p_momentum_sgd_batch, "gnnhip_momentum_sgd_batch_f32");
    look_up(p_adam_batch, "gnnhip_adam_batch_f32");
    look_up(g_last_error, "gnnhip_last_error");
    if (missing) return PyErr_Format(PyExc_RuntimeError, "%s exports no %s", path, missing);
    Py_INCREF(error);
    Py_XDECREF(g_error);
    g_error = error;
    Py_RETURN_NONE;
}

template <class F> PyCFunction as_method(F f) { return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)); }
#define GNNHIP_METHOD(name, names) {#name, as_method(f_##name), METH_FASTCALL, names},
PyMethodDef methods[] = {
    GNNHIP_ENTRIES(GNNHIP_METHOD)
    {"gemm_tn_batch", as_method(f_gemm_tn_batch), METH_FASTCALL, nullptr},
    {"momentum_sgd_batch", as_method(f_momentum_sgd_batch), METH_FASTCALL, nullptr},
    {"adam_batch", as_method(f_adam_batch), METH_FASTCALL, nullptr},
    {"empty", as_method(f_empty), METH_FASTCALL, nullptr},
    {"bind", f_bind, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_gnnhip_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__gnnhip_torch() { return PyModule_Create(&module); }
