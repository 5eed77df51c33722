"""Thin torch-pointer helpers over the C ABI (used by the tests, the smoke check and the bench).

torch supplies device memory and the stream; all arithmetic happens in libgnnhip.so.
Every helper validates dtype / device / contiguity on the host before a pointer
reaches a kernel, and raises GnnHipError on a non-zero status.
"""
import ctypes
import numpy as np

import torch

from ._lib import check, load_bindings, load_library

UNARY = {
    "set": 0, "truncate": 1, "scale": 2, "add": 3, "abs": 4, "inv": 5, "relu": 6, "sigmoid": 7,
    "tanh": 8, "log": 9, "invsqrt": 10, "exp": 11, "square": 12, "sqrt": 13,
}
REDUCE = {"sum": 0, "mean": 1, "max": 2, "sumsq": 3}

_initialised = False


def init(device_id=0):
    global _initialised
    lib = load_library()
    check(lib.gnnhip_init(int(device_id)))
    _initialised = True
    return lib


def _lib():
    if not _initialised:
        init(torch.cuda.current_device())
    return load_library()


_bindings = None


def _bound():
    """the compiled bindings: each C entry under its name without gnnhip_, taking torch tensors (checked there for type,
    device and contiguity) and the current stream, raising GnnHipError"""
    global _bindings
    if _bindings is None or not _initialised:
        _lib()
        _bindings = load_bindings()
    return _bindings


def _empty(where, kind, *sizes):
    """uninitialised tensor of float32 ('f') or int32 ('i') on the device of a tensor, or on a torch.device; several letters: a
    tuple of vectors ('f', 'i') and float32 matrices ('F'), each taking its sizes in turn"""
    return _bound().empty(where, kind, *sizes)


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _f32(t, name):
    if t is None:
        return None
    if not (t.is_cuda and t.dtype == torch.float32 and t.is_contiguous()):
        raise ValueError("%s must be a contiguous float32 CUDA tensor" % name)
    return ctypes.c_void_p(t.data_ptr())


def _i32(t, name):
    if t is None:
        return None
    if not (t.is_cuda and t.dtype == torch.int32 and t.is_contiguous()):
        raise ValueError("%s must be a contiguous int32 CUDA tensor" % name)
    return ctypes.c_void_p(t.data_ptr())


def _check_csr(row_ptr, col_idx, val, rows, name):
    if row_ptr.numel() != rows + 1:
        raise ValueError("%s.row_ptr must have rows+1 = %d entries" % (name, rows + 1))
    if col_idx.numel() != val.numel():
        raise ValueError("%s: col_idx and val differ in length" % name)


def spmm(row_ptr, col_idx, val, B, m, alpha=1.0, beta=0.0, out=None, nnz_hint=None):
    """out[m,n] = alpha * A * B + beta * out, A CSR with m rows and B.shape[0] columns.
    nnz_hint: the host-side entry count handed to the library (default: the arrays' length); it only sizes
    scratch, so any value from 0 up must give the same values."""
    k, n = B.shape
    _check_csr(row_ptr, col_idx, val, m, "A")
    if out is None:
        out = _empty(B, "f", m, n)
    elif tuple(out.shape) != (m, n):
        raise ValueError("out has the wrong shape")
    nnz = int(col_idx.numel()) if nnz_hint is None else int(nnz_hint)
    _bound().spmm_csr_f32(m, k, n, nnz, alpha, row_ptr, col_idx,
                                     val, B, n, beta, out, n)
    return out


class CsrPlan:
    """gnnhip_csr_plan_create for a CSR matrix [m, k] held in torch tensors, which the plan keeps alive; close() (or
    the end of a `with` block) destroys it.  spmm / level run the planned entry points."""

    def __init__(self, row_ptr, col_idx, val, m, k):
        _check_csr(row_ptr, col_idx, val, m, "A")
        self.m, self.k = int(m), int(k)
        self._keep = (row_ptr, col_idx, val)
        h = ctypes.c_void_p()
        check(_lib().gnnhip_csr_plan_create(self.m, self.k, _i32(row_ptr, "row_ptr"), _i32(col_idx, "col_idx"), _f32(val, "val"),
                                            _stream(), ctypes.byref(h)))
        self.handle = h

    def bytes(self):
        n = ctypes.c_size_t()
        check(_lib().gnnhip_csr_plan_bytes(self.handle, ctypes.byref(n)))
        return int(n.value)

    def spmm(self, B, alpha=1.0, beta=0.0, out=None):
        k, n = B.shape
        if k != self.k:
            raise ValueError("B must have %d rows" % self.k)
        if out is None:
            out = _empty(B, "f", self.m, n)
        elif tuple(out.shape) != (self.m, n):
            raise ValueError("out has the wrong shape")
        _bound().spmm_csr_planned_f32(self.handle.value, n, alpha, B, n, beta, out, n)
        return out

    def level(self, h_in, W, msg=None, bias=None, out=None):
        N, C = h_in.shape
        if N != self.m or tuple(W.shape) != (C, C):
            raise ValueError("h_in must be [m,C] and W [C,C]")
        if out is None:
            out = _empty(h_in, "f", N, C)
        _bound().s2v_level_planned_f32(self.handle.value, C, h_in, W, msg,
                                                  bias, out)
        return out

    def close(self):
        if self.handle is not None:
            check(_lib().gnnhip_csr_plan_destroy(self.handle))
            self.handle = None
            self._keep = None

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        self.close()


def release_scratch():
    """gives the current stream's library scratch back to the driver"""
    check(_lib().gnnhip_release_scratch(_stream()))


def gemm(A, B, transA=False, transB=False, alpha=1.0, beta=0.0, out=None, cols_a=None, cols_b=None):
    """cols_a / cols_b: use only the first so many columns of the stored A / B (the row stride stays the tensor's)"""
    ca = A.shape[1] if cols_a is None else int(cols_a)
    cb = B.shape[1] if cols_b is None else int(cols_b)
    if not (0 <= ca <= A.shape[1] and 0 <= cb <= B.shape[1]):
        raise ValueError("cols_a / cols_b out of range")
    m = ca if transA else A.shape[0]
    k = A.shape[0] if transA else ca
    kb = cb if transB else B.shape[0]
    n = B.shape[0] if transB else cb
    if k != kb:
        raise ValueError("mat dim doesn't match")
    if out is None:
        out = _empty(A, "f", m, n)
    elif tuple(out.shape) != (m, n):
        raise ValueError("out has the wrong shape")
    _bound().gemm_f32(int(transA), int(transB), m, n, k, alpha, A, A.shape[1],
                                 B, B.shape[1], beta, out, n)
    return out


def read_scalars(tensors):
    """the first element of each device tensor, all behind one wait for the stream"""
    n = len(tensors)
    outs = [np.zeros(1, np.float32 if t.dtype == torch.float32 else np.int32) for t in tensors]
    P = ctypes.c_void_p * n
    check(_lib().gnnhip_memcpy_d2h_batch(n, P(*[o.ctypes.data for o in outs]), P(*[t.data_ptr() for t in tensors]),
                                         (ctypes.c_size_t * n)(*[4] * n), _stream()))
    return [o[0] for o in outs]


def row_softmax_deriv(dst, out, grad):
    """dst += out * (grad - <grad, out> per row), in place on dst"""
    rows, cols = out.shape
    _bound().row_softmax_deriv_f32(dst, out, grad, rows, cols)
    return dst


def gemm_tn_batch(products, alpha=1.0, beta=0.0):
    """products: list of (A [k,m], B [k,n], out [m,n]); out = alpha * A^T B + beta * out for all of them in two launches"""
    products = [tuple(p) for p in products]
    _bound().gemm_tn_batch(products, alpha, beta)
    return [out for _, _, out in products]


def s2v_input(X, W_n2l):
    N, K = X.shape
    if W_n2l.shape[0] != K:
        raise ValueError("X and W_n2l disagree on the label width")
    C = W_n2l.shape[1]
    msg = _empty(X, "f", N, C)
    h0 = _empty(msg, "f", N, C)
    _bound().s2v_input_f32(N, K, C, X, W_n2l, msg,
                                      h0)
    return msg, h0


def s2v_input_labels(label, W_n2l, status=None):
    """msg = W_n2l[label], h0 = ReLU(msg): the input stage from one int label per node."""
    N = label.numel()
    K, C = W_n2l.shape
    msg = _empty(W_n2l, "f", N, C)
    h0 = _empty(msg, "f", N, C)
    _bound().s2v_input_labels_f32(N, K, C, label, W_n2l, msg,
                                             h0, status)
    return msg, h0


def s2v_level(row_ptr, col_idx, val, h_in, W, msg=None, bias=None, out=None, nnz_hint=None):
    """nnz_hint: the host-side entry count handed to the library (default: the arrays' length); it only
    sizes scratch, so any value from 0 up must give the same result."""
    N, C = h_in.shape
    _check_csr(row_ptr, col_idx, val, N, "A")
    if tuple(W.shape) != (C, C):
        raise ValueError("W must be [C,C]")
    if msg is not None and tuple(msg.shape) != (N, C):
        raise ValueError("msg must be [N,C]")
    if bias is not None and bias.numel() != C:
        raise ValueError("bias must have C entries")
    if out is None:
        out = _empty(h_in, "f", N, C)
    nnz = int(col_idx.numel()) if nnz_hint is None else int(nnz_hint)
    _bound().s2v_level_f32(N, C, nnz, row_ptr, col_idx, val,
                                      h_in, W, msg, bias,
                                      out)
    return out


def s2v_readout(s_row_ptr, s_col_idx, s_val, h, W_h1, W_h2, B):
    N, C = h.shape
    H, Q = W_h1.shape[1], W_h2.shape[1]
    _check_csr(s_row_ptr, s_col_idx, s_val, B, "S")
    if W_h1.shape[0] != C or W_h2.shape[0] != H:
        raise ValueError("readout weight shapes do not chain")
    dev = h.device
    pool = _empty(dev, "f", B, C)
    hidden = _empty(dev, "f", B, H)
    logits = _empty(dev, "f", B, Q)
    probs = _empty(dev, "f", B, Q)
    pred = _empty(dev, "i", B)
    _bound().s2v_readout_f32(B, N, C, H, Q, s_row_ptr, s_col_idx,
                                        s_val, h, W_h1, W_h2,
                                        pool, hidden, logits,
                                        probs, pred)
    return pool, hidden, logits, probs, pred


class ForwardBuffers:
    """Caller-owned activations of one forward; allocated once and reused across calls."""

    def __init__(self, N, B, C, H, Q, device):
        f = dict(dtype=torch.float32, device=device)
        self.msg = torch.empty((N, C), **f)
        self.h_a = torch.empty((N, C), **f)
        self.h_b = torch.empty((N, C), **f)
        self.pool = torch.empty((B, C), **f)
        self.hidden = torch.empty((B, H), **f)
        self.logits = torch.empty((B, Q), **f)
        self.probs = torch.empty((B, Q), **f)
        self.pred = torch.empty((B,), dtype=torch.int32, device=device)
        self.which = ctypes.c_int(0)

    @property
    def h_final(self):
        return self.h_a if self.which.value == 0 else self.h_b


def s2v_forward(a_csr, s_csr, X, W_n2l, W_conv, W_h1, W_h2, L, bufs=None):
    """Whole forward.  a_csr / s_csr are (row_ptr, col_idx, val) triples of int32/int32/float32 device tensors."""
    N, K = X.shape
    C, H, Q = W_n2l.shape[1], W_h1.shape[1], W_h2.shape[1]
    B = s_csr[0].numel() - 1
    _check_csr(a_csr[0], a_csr[1], a_csr[2], N, "A")
    _check_csr(s_csr[0], s_csr[1], s_csr[2], B, "S")
    if W_n2l.shape[0] != K or tuple(W_conv.shape) != (C, C) or W_h1.shape[0] != C or W_h2.shape[0] != H:
        raise ValueError("weight shapes do not chain")
    if bufs is None:
        bufs = ForwardBuffers(N, B, C, H, Q, X.device)
    _bound().s2v_forward_f32(
        N, B, K, C, H, Q, L, int(a_csr[1].numel()),
        a_csr[0], a_csr[1], a_csr[2],
        s_csr[0], s_csr[1], s_csr[2],
        X, W_n2l, W_conv, W_h1, W_h2,
        bufs.msg, bufs.h_a, bufs.h_b, bufs.pool,
        bufs.hidden, bufs.logits, bufs.probs,
        bufs.pred, ctypes.addressof(bufs.which))
    return bufs


def s2v_forward_planned(plan, s_csr, X, W_n2l, W_conv, W_h1, W_h2, L, bufs=None):
    """Whole forward with a CsrPlan of A (gnnhip_s2v_forward_planned_f32)."""
    N, K = X.shape
    C, H, Q = W_n2l.shape[1], W_h1.shape[1], W_h2.shape[1]
    B = s_csr[0].numel() - 1
    if N != plan.m or plan.m != plan.k:
        raise ValueError("the plan must be of the [N,N] adjacency")
    _check_csr(s_csr[0], s_csr[1], s_csr[2], B, "S")
    if W_n2l.shape[0] != K or tuple(W_conv.shape) != (C, C) or W_h1.shape[0] != C or W_h2.shape[0] != H:
        raise ValueError("weight shapes do not chain")
    if bufs is None:
        bufs = ForwardBuffers(N, B, C, H, Q, X.device)
    _bound().s2v_forward_planned_f32(
        plan.handle.value, B, K, C, H, Q, L,
        s_csr[0], s_csr[1], s_csr[2],
        X, W_n2l, W_conv, W_h1, W_h2,
        bufs.msg, bufs.h_a, bufs.h_b, bufs.pool,
        bufs.hidden, bufs.logits, bufs.probs,
        bufs.pred, ctypes.addressof(bufs.which))
    return bufs


class BatchedBuffers:
    """Caller-owned outputs of the graph-resident forward."""

    def __init__(self, N, B, C, H, Q, device):
        f = dict(dtype=torch.float32, device=device)
        self.msg = torch.empty((N, C), **f)
        self.h_final = torch.empty((N, C), **f)
        self.pool = torch.empty((B, C), **f)
        self.hidden = torch.empty((B, H), **f)
        self.logits = torch.empty((B, Q), **f)
        self.probs = torch.empty((B, Q), **f)
        self.pred = torch.empty((B,), dtype=torch.int32, device=device)
        self.status = torch.zeros((1,), dtype=torch.int32, device=device)


def s2v_forward_batched(a_csr, s_csr, X, W_n2l, W_conv, W_h1, W_h2, L, max_graph_nodes, bufs=None):
    """One-launch forward for block-diagonal batches (see gnnhip_s2v_forward_batched_sized_f32)."""
    N, K = X.shape
    C, H, Q = W_n2l.shape[1], W_h1.shape[1], W_h2.shape[1]
    B = s_csr[0].numel() - 1
    _check_csr(a_csr[0], a_csr[1], a_csr[2], N, "A")
    _check_csr(s_csr[0], s_csr[1], s_csr[2], B, "S")
    if s_csr[1].numel() != N:
        raise ValueError("S must list every node exactly once")
    if W_n2l.shape[0] != K or tuple(W_conv.shape) != (C, C) or W_h1.shape[0] != C or W_h2.shape[0] != H:
        raise ValueError("weight shapes do not chain")
    if bufs is None:
        bufs = BatchedBuffers(N, B, C, H, Q, X.device)
    _bound().s2v_forward_batched_sized_f32(
        N, B, K, C, H, Q, L, int(max_graph_nodes), int(a_csr[1].numel()),
        a_csr[0], a_csr[1], a_csr[2],
        s_csr[0], s_csr[1], s_csr[2],
        X, W_n2l, W_conv, W_h1, W_h2,
        bufs.msg, bufs.h_final, bufs.pool,
        bufs.hidden, bufs.logits, bufs.probs,
        bufs.pred, bufs.status)
    return bufs


def s2v_forward_batched_train(a_csr, s_csr, X, W_n2l, W_conv, W_h1, W_h2, L, max_graph_nodes, bufs=None):
    """The one-launch forward that keeps every level: returns (bufs, h_levels [(L + 1), N, C]); bufs.h_final is
    not written (h_levels[L] is that embedding)."""
    N, K = X.shape
    C, H, Q = W_n2l.shape[1], W_h1.shape[1], W_h2.shape[1]
    B = s_csr[0].numel() - 1
    _check_csr(a_csr[0], a_csr[1], a_csr[2], N, "A")
    _check_csr(s_csr[0], s_csr[1], s_csr[2], B, "S")
    if s_csr[1].numel() != N:
        raise ValueError("S must list every node exactly once")
    if W_n2l.shape[0] != K or tuple(W_conv.shape) != (C, C) or W_h1.shape[0] != C or W_h2.shape[0] != H:
        raise ValueError("weight shapes do not chain")
    if bufs is None:
        bufs = BatchedBuffers(N, B, C, H, Q, X.device)
    h_levels = _empty(X, "f", L + 1, N, C)
    _bound().s2v_forward_batched_train_sized_f32(
        N, B, K, C, H, Q, L, int(max_graph_nodes), int(a_csr[1].numel()),
        a_csr[0], a_csr[1], a_csr[2],
        s_csr[0], s_csr[1], s_csr[2],
        X, W_n2l, W_conv, W_h1, W_h2,
        bufs.msg, h_levels, bufs.pool,
        bufs.hidden, bufs.logits, bufs.probs,
        bufs.pred, bufs.status)
    return bufs, h_levels


def bind_s2v_forward_batched(a_csr, s_csr, X, W_n2l, W_conv, W_h1, W_h2, L, max_graph_nodes, bufs, stream):
    """The call of s2v_forward_batched with every argument converted once: returns a function that queues one
    forward on `stream` (a torch.cuda.Stream) and raises on a non-zero status code.  For callers that keep several
    batches in flight on several streams, where the per-call argument checks of the helper above would be the
    bottleneck."""
    N, K = X.shape
    C, H, Q = W_n2l.shape[1], W_h1.shape[1], W_h2.shape[1]
    B = s_csr[0].numel() - 1
    _check_csr(a_csr[0], a_csr[1], a_csr[2], N, "A")
    _check_csr(s_csr[0], s_csr[1], s_csr[2], B, "S")
    if s_csr[1].numel() != N:
        raise ValueError("S must list every node exactly once")
    if W_n2l.shape[0] != K or tuple(W_conv.shape) != (C, C) or W_h1.shape[0] != C or W_h2.shape[0] != H:
        raise ValueError("weight shapes do not chain")
    fn = _lib().gnnhip_s2v_forward_batched_sized_f32
    args = (N, B, K, C, H, Q, L, int(max_graph_nodes), int(a_csr[1].numel()),
            _i32(a_csr[0], "a_row_ptr"), _i32(a_csr[1], "a_col_idx"), _f32(a_csr[2], "a_val"),
            _i32(s_csr[0], "s_row_ptr"), _i32(s_csr[1], "s_col_idx"), _f32(s_csr[2], "s_val"),
            _f32(X, "X"), _f32(W_n2l, "W_n2l"), _f32(W_conv, "W_conv"), _f32(W_h1, "W_h1"), _f32(W_h2, "W_h2"),
            _f32(bufs.msg, "msg"), _f32(bufs.h_final, "h_final"), _f32(bufs.pool, "pool"),
            _f32(bufs.hidden, "hidden"), _f32(bufs.logits, "logits"), _f32(bufs.probs, "probs"),
            _i32(bufs.pred, "pred"), _i32(bufs.status, "status"), ctypes.c_void_p(stream.cuda_stream))

    def queue():
        rc = fn(*args)
        if rc:
            check(rc)
    return queue


def s2v_forward_batched_labels(a_csr, s_csr, label, W_n2l, W_conv, W_h1, W_h2, L, max_graph_nodes, bufs=None):
    """One-launch forward from one int label per node (see gnnhip_s2v_forward_batched_labels_sized_f32)."""
    N = label.numel()
    K, C = W_n2l.shape
    H, Q = W_h1.shape[1], W_h2.shape[1]
    B = s_csr[0].numel() - 1
    _check_csr(a_csr[0], a_csr[1], a_csr[2], N, "A")
    _check_csr(s_csr[0], s_csr[1], s_csr[2], B, "S")
    if s_csr[1].numel() != N:
        raise ValueError("S must list every node exactly once")
    if tuple(W_conv.shape) != (C, C) or W_h1.shape[0] != C or W_h2.shape[0] != H:
        raise ValueError("weight shapes do not chain")
    if bufs is None:
        bufs = BatchedBuffers(N, B, C, H, Q, W_n2l.device)
    _bound().s2v_forward_batched_labels_sized_f32(
        N, B, K, C, H, Q, L, int(max_graph_nodes), int(a_csr[1].numel()),
        a_csr[0], a_csr[1], a_csr[2],
        s_csr[0], s_csr[1], s_csr[2],
        label, W_n2l, W_conv, W_h1, W_h2,
        bufs.msg, bufs.h_final, bufs.pool,
        bufs.hidden, bufs.logits, bufs.probs,
        bufs.pred, bufs.status)
    return bufs


def unary(op, x, a0=0.0, a1=0.0):
    _bound().unary_f32(UNARY[op], x, x.numel(), a0, a1)
    return x


def relu(x, out=None):
    if out is None:
        out = torch.empty_like(x)
    _bound().relu_f32(x, out, x.numel())
    return out


def axpy(a, x, y):
    if x.numel() != y.numel():
        raise ValueError("shape doesn't match in Axpy")
    _bound().axpy_f32(x.numel(), a, x, y)
    return y


def axpby(a, x, b, y):
    if x.numel() != y.numel():
        raise ValueError("shape doesn't match in Axpby")
    _bound().axpby_f32(x.numel(), a, x, b, y)
    return y


def add(a, b, out=None):
    if a.numel() != b.numel():
        raise ValueError("no broadcasting is supported")
    if out is None:
        out = torch.empty_like(a)
    _bound().add_f32(a.numel(), a, b, out)
    return out


def row_softmax(x):
    rows, cols = x.shape
    _bound().row_softmax_f32(x, rows, cols)
    return x


def jagged_softmax(x, lens):
    _bound().jagged_softmax_f32(x, lens, lens.numel())
    return x


def jagged_softmax_deriv(dst, out, grad, lens):
    """dst += (grad - <grad, out> per segment) * out"""
    _bound().jagged_softmax_deriv_f32(dst, out, grad, lens,
                                                 lens.numel())
    return dst


def jagged_softmax_static(x, lens):
    """gnnhip_jagged_softmax_static_f32: the same result, segment offsets in the library's static array."""
    _bound().jagged_softmax_static_f32(x, lens, lens.numel())
    return x


def reduce(op, x):
    out = _empty(x, "f", 1)
    _bound().reduce_f32(REDUCE[op], x, x.numel(), out)
    return out


def row_argmax(x):
    rows, cols = x.shape
    out = _empty(x, "i", rows)
    _bound().row_argmax_f32(x, rows, cols, out)
    return out


def csr_row_argmax(row_ptr, col_idx, val):
    rows = row_ptr.numel() - 1
    out = _empty(row_ptr, "i", rows)
    _bound().csr_row_argmax_f32(row_ptr, col_idx, val,
                                           rows, out)
    return out


def cross_entropy(prob, l_row_ptr, l_col_idx, l_val):
    rows, cols = prob.shape
    _check_csr(l_row_ptr, l_col_idx, l_val, rows, "label")
    out = _empty(prob, "f", rows, 1)
    _bound().cross_entropy_f32(prob, rows, cols, l_row_ptr,
                                          l_col_idx, l_val, out)
    return out


def in_top_k(pred, label, k=1):
    rows, cols = pred.shape
    if label.numel() != rows:
        raise ValueError("# instances doesn't match")
    out = _empty(pred, "i", rows)
    _bound().in_top_k_f32(pred, label, rows, cols, k, out)
    return out


def cast_i32_f32(src):
    dst = torch.empty(src.shape, dtype=torch.float32, device=src.device)
    _bound().cast_i32_f32(src, dst, src.numel())
    return dst


def memset0(t):
    check(_lib().gnnhip_memset0(ctypes.c_void_p(t.data_ptr()), t.numel() * t.element_size(), _stream()))
    return t


def memset0_batch(tensors):
    """zero-fill several device buffers in one launch"""
    n = len(tensors)
    ptrs = (ctypes.c_void_p * n)(*[t.data_ptr() for t in tensors])
    sizes = (ctypes.c_size_t * n)(*[t.numel() * t.element_size() for t in tensors])
    check(_lib().gnnhip_memset0_batch(n, ptrs, sizes, _stream()))
    return tensors


# ---- backward-pass entry points
def spmm_t(row_ptr, col_idx, val, B, m, k, alpha=1.0, beta=0.0, out=None):
    """out[k,n] = alpha * A^T * B + beta * out, A CSR [m,k], B [m,n]"""
    n = B.shape[1]
    _check_csr(row_ptr, col_idx, val, m, "A")
    if B.shape[0] != m:
        raise ValueError("mat dim doesn't match")
    if out is None:
        out = torch.zeros((k, n), dtype=torch.float32, device=B.device)
    _bound().spmm_csr_t_f32(m, k, n, alpha, row_ptr, col_idx,
                                       val, B, n, beta, out, n)
    return out


def csr_axpy(a, row_ptr, col_idx, val, dense):
    rows, cols = dense.shape
    _check_csr(row_ptr, col_idx, val, rows, "x")
    _bound().csr_axpy_f32(rows, cols, a, row_ptr, col_idx, val,
                                     dense)
    return dense


def relu_deriv(dst, out, grad):
    if not (dst.numel() == out.numel() == grad.numel()):
        raise ValueError("shape mismatch in ReLUDeriv")
    _bound().relu_deriv_f32(dst.numel(), out, grad, dst)
    return dst


def mul(x, y):
    if x.numel() != y.numel():
        raise ValueError("shape mismatch in ElewiseMul")
    _bound().mul_f32(x.numel(), x, y)
    return y


def row_scale(scale, y):
    rows, cols = y.shape
    if scale.numel() != rows:
        raise ValueError("one factor per row is needed")
    _bound().row_scale_f32(rows, cols, scale, y)
    return y


# ---- device-side CSR construction
def csr_group(rows, key, payload, average=False, key_stride=1, payload_stride=1, n=None):
    """row i lists payload[e] of the pairs with key[e] == i in input order (device arrays, int32)"""
    if n is None:
        n = key.numel() // key_stride
    row_ptr, col_idx, val = _empty(key, "iif", rows + 1, n, n)
    _bound().csr_group_i32(rows, n, key, key_stride, payload, payload_stride,
                                      int(average), row_ptr, col_idx, val)
    return row_ptr, col_idx, val


def csr_group_both(rows, x, y, x_stride=1, y_stride=1, n=None):
    """the pairs (x, y) grouped by y (row i lists x) and by x (row i lists y): a matrix and its transpose, values 1"""
    if n is None:
        n = x.numel() // x_stride
    out = _empty(x, "iifiif", rows + 1, n, n, rows + 1, n, n)
    _bound().csr_group_both_i32(rows, n, x, x_stride, y, y_stride,
                                           out[0], out[1], out[2],
                                           out[3], out[4], out[5])
    return out[:3], out[3:]


def csr_consecutive_rows(row_ptr, average=False):
    """col_idx, val of the CSR matrix whose row i lists the columns row_ptr[i] .. row_ptr[i+1]-1 (row_ptr on the device)"""
    rows = row_ptr.numel() - 1
    n = int(row_ptr[-1].item())
    col_idx = _empty(row_ptr, "i", n)
    val = _empty(row_ptr, "f", n)
    _bound().csr_consecutive_rows_f32(rows, row_ptr, int(average), col_idx,
                                                 val)
    return col_idx, val


def csr_consecutive_rows_host(offsets, device, average=False):
    """(row_ptr, col_idx, val) on the device from the row offsets in a host int32 array"""
    offsets = np.ascontiguousarray(offsets, np.int32)
    rows, n = offsets.size - 1, int(offsets[-1])
    device = torch.device(device)
    row_ptr, col_idx, val = _empty(device, "iif", rows + 1, n, n)
    _bound().csr_consecutive_rows_host_f32(rows, offsets, int(average), row_ptr, col_idx if n else None, val if n else None)
    return row_ptr, col_idx, val


def csr_transpose(row_ptr, col_idx, val, m, k):
    nnz = col_idx.numel()
    dev = row_ptr.device
    t_rp = _empty(dev, "i", k + 1)
    t_ci = _empty(dev, "i", nnz)
    t_v = _empty(dev, "f", nnz)
    _bound().csr_transpose_f32(m, k, nnz, row_ptr, col_idx, val,
                                          t_rp, t_ci, t_v)
    return t_rp, t_ci, t_v


# ---------------------------------------------------------------- training iteration
def loss_acc(logits, lrow_ptr, lcol, lval, want_rows=False):
    """mean cross-entropy (softmax inside) and mean top-1 accuracy of a batch in one pass over the logits"""
    B, Q = logits.shape
    probs, loss, acc = _empty(logits, "Fff", B, Q, 1, 1)
    loss_rows, hit = _empty(logits, "fi", B, B) if want_rows else (None, None)
    _bound().s2v_loss_acc_f32(B, Q, logits, lrow_ptr, lcol,
                                         lval, probs, loss_rows,
                                         hit, loss, acc)
    return loss, acc, probs, loss_rows, hit


def readout_backward(s_csr, probs, label_csr, scale, hidden, W_h1, W_h2, N):
    B, Q = probs.shape
    C, H = W_h1.shape
    dlogits, du, g_h = _empty(probs, "FFF", B, Q, B, H, N, C)
    _bound().s2v_readout_backward_f32(
        B, N, C, H, Q, s_csr[0], s_csr[1], s_csr[2],
        probs, label_csr[0], label_csr[1], label_csr[2],
        float(scale), hidden, W_h1, W_h2,
        dlogits, du, g_h)
    return dlogits, du, g_h


def s2v_level_backward(t_row_ptr, t_col_idx, t_val, dz, W, u=None, g_prev=None, gate_h=None, acc=None):
    """u = A^T dz, g_prev = u W^T (zeroed where gate_h <= 0 when gate_h is given), acc += g_prev when acc is given;
    the CSR arrays are those of A^T"""
    N, C = dz.shape
    _check_csr(t_row_ptr, t_col_idx, t_val, N, "A^T")
    if u is None:
        u = _empty(dz, "f", N, C)
    if g_prev is None:
        g_prev = _empty(dz, "f", N, C)
    _bound().s2v_level_backward_f32(N, C, int(t_col_idx.numel()), t_row_ptr, t_col_idx,
                                               t_val, dz, W, u, g_prev,
                                               gate_h, acc)
    return u, g_prev


def grad_gate(h, g, dz=None, acc=None, accumulate=False):
    _bound().s2v_grad_gate_f32(h.numel(), h, g, dz, acc,
                                          1 if accumulate else 0)


def momentum_sgd_batch(ws, gs, vs, lr, momentum, l2):
    _bound().momentum_sgd_batch(list(ws), list(gs), list(vs) if vs is not None else None, float(lr), float(momentum), float(l2))


def adam_batch(ws, gs, ms, vs, lr, l2, clip_threshold, beta1, beta2, eps, t):
    """one AdamOptimizer::Update over the tensors, t = the iteration count after the increment (1 for the first)"""
    s1 = np.float32(1.0 / (1 - float(np.float32(beta1)) ** t))
    s2 = np.float32(1.0 / (1 - float(np.float32(beta2)) ** t))
    _bound().adam_batch(list(ws), list(gs), list(ms), list(vs), float(lr), float(l2), float(clip_threshold), float(beta1), float(beta2),
                        float(eps), float(s1), float(s2))


def upload_sparse32(host_array, out=None):
    """Host numpy array of 32-bit elements -> device tensor through gnnhip_memcpy_h2d_sparse32 (non-zero words only
    when they are few); the device tensor has the bits of the host array."""
    import numpy as np
    a = np.ascontiguousarray(host_array)
    if a.dtype.itemsize != 4:
        raise ValueError("upload_sparse32 takes 32-bit elements")
    tdt = {"float32": torch.float32, "int32": torch.int32}[a.dtype.name]
    if out is None:
        out = torch.empty(a.shape, dtype=tdt, device="cuda")
    check(_lib().gnnhip_memcpy_h2d_sparse32(ctypes.c_void_p(out.data_ptr()), a.ctypes.data_as(ctypes.c_void_p), a.size, _stream()))
    return out
