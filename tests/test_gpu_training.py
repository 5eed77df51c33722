"""The kernels that carry one training iteration of the structure2vec path (loss/accuracy tail, readout
backward, gradient gate, batched momentum-SGD update) against the oracle, and the whole iteration composed
from C-ABI calls the way the host layer's fused training plan composes it, against float64 autograd."""
import numpy as np
import pytest

from conftest import PARITY_TOL, assert_parity, max_rel
from graphnn_amd import batching, synth

pytestmark = pytest.mark.gpu


def _t(a, dev):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def _n(t):
    return t.detach().cpu().numpy()


@pytest.mark.parametrize("B,Q", [(256, 2), (1, 3), (5000, 7), (1025, 2), (300, 70)])
def test_loss_and_accuracy_tail(gpu, oracle, B, Q):
    from graphnn_amd import ops
    rng = np.random.default_rng(B + Q)
    logits = (rng.standard_normal((B, Q)) * 3).astype(np.float32)
    logits[::7] = np.round(logits[::7])                            # ties between logits
    if B > 10:
        logits[3] = [200.0] + [-200.0] * (Q - 1)                   # a probability that underflows: the 1e-8 clamp
    y = rng.integers(0, Q, B).astype(np.int32)
    if B > 10:
        y[3] = Q - 1
    lab = (np.arange(B + 1, dtype=np.int32), y, np.ones(B, np.float32))
    loss, acc, probs, loss_rows, hit = ops.loss_acc(_t(logits, gpu), *[_t(a, gpu) for a in lab], want_rows=True)
    w_probs = oracle.row_softmax(logits)
    w_rows = oracle.cross_entropy(w_probs, *lab)
    w_hit = oracle.in_top_k(logits, oracle.csr_row_argmax(*lab), 1)
    assert max_rel(_n(probs), w_probs, floor=1e-6) < PARITY_TOL
    assert np.allclose(_n(loss_rows), w_rows, rtol=1e-4, atol=1e-6)
    assert np.array_equal(_n(hit), w_hit)
    assert abs(float(_n(loss)[0]) - oracle.mean(w_rows)) <= 1e-4 * abs(oracle.mean(w_rows))
    assert abs(float(_n(acc)[0]) - oracle.mean(oracle.cast(w_hit))) <= 1e-6


def test_loss_tail_with_weighted_and_empty_label_rows(gpu, oracle):
    from graphnn_amd import ops
    rng = np.random.default_rng(9)
    B, Q = 40, 5
    logits = rng.standard_normal((B, Q)).astype(np.float32)
    lens = rng.integers(0, 4, B); lens[0] = 0
    rp = np.zeros(B + 1, np.int32); np.cumsum(lens, out=rp[1:])
    ci = rng.integers(0, Q, rp[-1]).astype(np.int32)
    v = rng.random(rp[-1]).astype(np.float32)
    lab = (rp, ci, v)
    loss, acc, probs, loss_rows, hit = ops.loss_acc(_t(logits, gpu), *[_t(a, gpu) for a in lab], want_rows=True)
    w_probs = oracle.row_softmax(logits)
    assert np.allclose(_n(loss_rows), oracle.cross_entropy(w_probs, *lab), rtol=1e-4, atol=1e-6)
    assert np.array_equal(_n(hit), oracle.in_top_k(logits, oracle.csr_row_argmax(*lab), 1))


@pytest.mark.parametrize("C,H,Q,B", [(64, 32, 2, 256), (16, 8, 3, 5), (256, 128, 2, 700), (48, 100, 70, 33),
                                     # from 1,024 graphs: du W_h1^T as one product over all graphs, node rows by a kernel of their own
                                     (256, 128, 2, 1024), (64, 32, 2, 3000), (130, 20, 3, 1100), (600, 16, 2, 1030)])
def test_readout_backward(gpu, oracle, C, H, Q, B):
    from graphnn_amd import ops
    rng = np.random.default_rng(C + H + B)
    batch = synth.molecule_batch(C + B, B, 5, Q, size_mode="uniform", size_lo=1, size_hi=40)
    N = batch.num_nodes
    s = batching.subgraph_csr(B, batch.subg_id, batch.node_idx)
    s = (s[0], s[1], (0.5 + rng.random(N)).astype(np.float32))
    lab = batch.label_csr()
    probs = oracle.row_softmax(rng.standard_normal((B, Q)).astype(np.float32))
    hidden = np.maximum(rng.standard_normal((B, H)), 0).astype(np.float32)
    W1 = (rng.standard_normal((C, H)) * 0.2).astype(np.float32)
    W2 = (rng.standard_normal((H, Q)) * 0.2).astype(np.float32)
    scale = 1.0 / B
    dl, du, gh = ops.readout_backward([_t(a, gpu) for a in s], _t(probs, gpu), [_t(a, gpu) for a in lab], scale,
                                      _t(hidden, gpu), _t(W1, gpu), _t(W2, gpu), N)
    Y = np.zeros((B, Q), np.float32); Y[np.arange(B), batch.graph_label] = 1.0
    w_dl = ((probs - Y) * np.float32(scale)).astype(np.float32)
    w_du = (oracle.gemm(w_dl, W2, transB=True) * (hidden > 0)).astype(np.float32)
    w_dpool = oracle.gemm(w_du, W1, transB=True)
    w_gh = oracle.spmm_T(*s, w_dpool, B, N)
    assert np.array_equal(_n(dl), w_dl)
    f8 = np.float64
    du64 = (w_dl.astype(f8) @ W2.astype(f8).T) * (hidden > 0)
    assert_parity("du", _n(du), w_du, du64)
    gh64 = np.repeat(du64 @ W1.astype(f8).T, batch.graph_sizes, axis=0) * s[2][:, None].astype(f8)
    assert_parity("g_h", _n(gh), w_gh, gh64)


@pytest.mark.parametrize("C", [1, 4, 6, 100, 500, 1024, 1028])
def test_readout_backward_rows_whatever_the_width(gpu, oracle, C):
    """the node rows written as 128-bit words (a width that is a multiple of four, at most 1,024, into a buffer that starts on
    one) and element by element, graphs of more rows than the lanes hold list entries of: the same bits, and the oracle's"""
    import torch
    from graphnn_amd import ops
    rng = np.random.default_rng(C)
    sizes = np.array([1, 7, 8, 9, 64, 65, 300, 2])
    B, H, Q, N = sizes.size, 9, 3, int(sizes.sum())
    s = (np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32), rng.permutation(N).astype(np.int32), rng.random(N).astype(np.float32))
    lab = (np.arange(B + 1, dtype=np.int32), rng.integers(0, Q, B).astype(np.int32), np.ones(B, np.float32))
    probs = oracle.row_softmax(rng.standard_normal((B, Q)).astype(np.float32))
    hidden = np.maximum(rng.standard_normal((B, H)), 0).astype(np.float32)
    W1 = (rng.standard_normal((C, H)) * 0.2).astype(np.float32)
    W2 = (rng.standard_normal((H, Q)) * 0.2).astype(np.float32)
    dev = [_t(a, gpu) for a in (*s, probs, *lab)]
    hid, w1, w2 = _t(hidden, gpu), _t(W1, gpu), _t(W2, gpu)
    got = []
    for shift in (0, 1):
        dl, du = torch.empty(B, Q, device=gpu), torch.empty(B, H, device=gpu)
        gh = torch.zeros(N * C + shift, device=gpu)[shift:].view(N, C)
        ops._bound().s2v_readout_backward_f32(B, N, C, H, Q, *dev, 0.25, hid, w1, w2, dl, du, gh)
        got.append(_n(gh))
    assert np.array_equal(got[0], got[1])
    du64 = _n(du).astype(np.float64)
    w_gh = oracle.spmm_T(*s, oracle.gemm(_n(du), W1, transB=True), B, N)
    gh64 = np.zeros((N, C))
    gh64[s[1]] = np.repeat(du64 @ W1.astype(np.float64).T, sizes, axis=0) * s[2][:, None]
    assert_parity("g_h", got[0], w_gh, gh64)


@pytest.mark.parametrize("C,nodes", [(4, 3), (64, 7), (64, 8), (128, 3), (128, 4), (100, 5), (100, 6)])
def test_readout_backward_of_small_graphs(gpu, C, nodes):
    """from 512 elements per graph on the node rows are written as 128-bit words, below element by element: the same bits as in
    a buffer that starts between two words, where they always are"""
    import torch
    from graphnn_amd import ops
    B, H, Q = 37, 9, 3
    N = B * nodes
    gen = torch.Generator(device=gpu).manual_seed(C + nodes)
    s = (torch.arange(B + 1, device=gpu).int() * nodes, torch.randperm(N, generator=gen, device=gpu).int(), torch.rand(N, generator=gen, device=gpu))
    lab = (torch.arange(B + 1, device=gpu).int(), torch.randint(0, Q, (B,), generator=gen, device=gpu).int(), torch.ones(B, device=gpu))
    probs, hidden = torch.rand(B, Q, generator=gen, device=gpu), torch.rand(B, H, generator=gen, device=gpu)
    W1, W2 = torch.randn(C, H, generator=gen, device=gpu), torch.randn(H, Q, generator=gen, device=gpu)
    dl, du, gh = ops.readout_backward(s, probs, lab, 0.25, hidden, W1, W2, N)
    between = torch.zeros(N * C + 1, device=gpu)[1:].view(N, C)
    ops._bound().s2v_readout_backward_f32(B, N, C, H, Q, *s, probs, *lab, 0.25, hidden, W1, W2, torch.empty_like(dl), torch.empty_like(du), between)
    assert torch.equal(gh, between)
    want = torch.zeros(N, C, dtype=torch.float64, device=gpu)
    want[s[1].long()] = (du.double() @ W1.double().T).repeat_interleave(nodes, 0) * s[2].double()[:, None]
    terms = torch.zeros_like(want)
    terms[s[1].long()] = (du.double().abs() @ W1.double().abs().T).repeat_interleave(nodes, 0) * s[2].double()[:, None]
    assert bool(((gh.double() - want).abs() <= (H + 2) * 2.0 ** -24 * terms).all())      # a rounding per product and sum, and the weight's


@pytest.mark.parametrize("N,C", [(N, C) for C in (16, 32, 64, 128, 256) for N in (77, 7450, 40_000)] + [(70_001, 128), (70_001, 256), (16_400, 256)])
def test_level_backward(gpu, oracle, C, N):
    """u = A^T dz and g_prev = u W^T in one pass (hidden 16/32/64: the streaming kernel; hidden 128/256: the wide kernel's
    backward variant in passes of 16, 32 and 64 rows, which the row counts select): ragged rows, two long rows (the larger
    matrices send them through the balanced pass at the narrow sizes), signed dz"""
    from graphnn_amd import ops
    rng = np.random.default_rng(C + N)
    lens = rng.integers(0, 7, N); lens[N // 3] = min(N, 3000); lens[N - 1] = 70
    rp = np.zeros(N + 1, np.int32); np.cumsum(lens, out=rp[1:])
    nnz = int(rp[-1])
    ci = rng.integers(0, N, nnz).astype(np.int32)
    v = (rng.random(nnz) * 0.5).astype(np.float32)
    dz = (rng.standard_normal((N, C)) * (rng.random((N, C)) < 0.5)).astype(np.float32)      # about half the gates closed
    W = (rng.standard_normal((C, C)) * 0.1).astype(np.float32)
    u, g = ops.s2v_level_backward(_t(rp, gpu), _t(ci, gpu), _t(v, gpu), _t(dz, gpu), _t(W, gpu))
    w_u = oracle.spmm(rp, ci, v, dz, N)
    w_g = oracle.gemm(w_u, W, transB=True)
    import scipy.sparse as sp
    u64 = sp.csr_matrix((v.astype(np.float64), ci, rp), shape=(N, N)) @ dz.astype(np.float64)
    assert_parity("u", _n(u), w_u, u64)
    assert_parity("g_prev", _n(g), w_g, u64 @ W.astype(np.float64).T)
    # with the ReLU gate of the level below and the running sum of the msg gradient: the stored g_prev is the
    # ungated one with the closed gates zeroed (same bits), and acc grows by exactly what was stored
    h_prev = rng.standard_normal((N, C)).astype(np.float32)
    h_prev[rng.random((N, C)) < 0.1] = 0.0                       # zeros close the gate, like negative values
    acc0 = rng.standard_normal((N, C)).astype(np.float32)
    acc = _t(acc0, gpu)
    u2, g2 = ops.s2v_level_backward(_t(rp, gpu), _t(ci, gpu), _t(v, gpu), _t(dz, gpu), _t(W, gpu), gate_h=_t(h_prev, gpu), acc=acc)
    gated = np.where(h_prev > 0, _n(g), np.float32(0))
    assert np.array_equal(_n(u2), _n(u))
    assert np.array_equal(_n(g2), gated)
    assert np.array_equal(_n(acc), acc0 + gated)
    # the sum alone, without a gate
    acc = _t(acc0, gpu)
    _, g3 = ops.s2v_level_backward(_t(rp, gpu), _t(ci, gpu), _t(v, gpu), _t(dz, gpu), _t(W, gpu), acc=acc)
    assert np.array_equal(_n(g3), _n(g)) and np.array_equal(_n(acc), acc0 + _n(g))


@pytest.mark.parametrize("C", [4, 7, 48, 63, 65, 100, 129, 255])
@pytest.mark.parametrize("N", [1, 17, 1_500, 16_421, 32_770])
def test_level_of_any_hidden_size_both_directions(gpu, oracle, C, N):
    """hidden sizes without a kernel of their own, forward and backward in one launch each: column counts around the blocks of
    16 and the shares of the wavefronts, row counts around the tiles of 16, 32 and 64 rows, tiles whose entries do not fit
    LDS, rows longer than 64 (the balanced pass from 32,768 rows on) and 2,048 entries, empty rows, the input stage"""
    from graphnn_amd import ops
    if N * C > 2_200_000:
        pytest.skip("the float64 model of the larger sizes adds nothing")
    rng = np.random.default_rng(C + N)
    lens = rng.integers(0, 6, N)
    if N > 100:
        lens[10:40] = 60; lens[41] = 0; lens[N // 2] = 3000; lens[N - 1] = 70
    rp = np.zeros(N + 1, np.int32); np.cumsum(lens, out=rp[1:])
    nnz = int(rp[-1])
    ci = rng.integers(0, N, nnz).astype(np.int32)
    v = (rng.random(nnz) * 0.5).astype(np.float32)
    x = rng.random((N, C)).astype(np.float32)           # sums of 3,000 signed terms would cancel
    W = (rng.standard_normal((C, C)) * 0.1).astype(np.float32)
    msg = rng.standard_normal((N, C)).astype(np.float32)
    bias = rng.standard_normal(C).astype(np.float32)
    pad = lambda a, dt: _t(np.concatenate([a, np.zeros(1, dt)]), gpu)[:a.size]      # never a null pointer for an empty array
    A = (_t(rp, gpu), pad(ci, np.int32), pad(v, np.float32))
    import scipy.sparse as sp
    u64 = sp.csr_matrix((v.astype(np.float64), ci, rp), shape=(N, N)) @ x.astype(np.float64)
    got = ops.s2v_level(*A, _t(x, gpu), _t(W, gpu), _t(msg, gpu), _t(bias, gpu))
    assert_parity("level", _n(got), oracle.level(rp, ci, v, x, W, msg, bias), np.maximum(u64 @ W.astype(np.float64) + bias + msg, 0))
    h_prev = rng.standard_normal((N, C)).astype(np.float32)
    acc = _t(msg, gpu)
    u, g = ops.s2v_level_backward(*A, _t(x, gpu), _t(W, gpu), gate_h=_t(h_prev, gpu), acc=acc)
    w_u = oracle.spmm(rp, ci, v, x, N)
    assert_parity("u", _n(u), w_u, u64)
    assert_parity("g_prev", _n(g), (oracle.gemm(w_u, W, transB=True) * (h_prev > 0)).astype(np.float32), (u64 @ W.astype(np.float64).T) * (h_prev > 0))
    assert np.array_equal(_n(acc), msg + _n(g))
    X = rng.standard_normal((N, 19)).astype(np.float32)
    Wn = rng.standard_normal((19, C)).astype(np.float32)
    m, h0 = ops.s2v_input(_t(X, gpu), _t(Wn, gpu))
    assert_parity("msg", _n(m), oracle.gemm(X, Wn), X.astype(np.float64) @ Wn.astype(np.float64))
    assert np.array_equal(_n(h0), np.maximum(_n(m), 0))


@pytest.mark.parametrize("C", [66, 100, 129, 150, 255])
def test_level_of_wide_odd_hidden_sizes_with_long_rows(gpu, C):
    """hidden sizes without a kernel of their own past 64 columns, from the row count on at which the balanced pass sums the rows
    of more than 64 entries (one chunk, several chunks, the first and the last row of a tile and of the matrix): forward,
    backward, with a plan, and reading its input through ReLU as a forward's first level does"""
    import torch
    from graphnn_amd import ops
    rng = np.random.default_rng(C)
    N = 32_768 + 37
    lens = rng.integers(0, 6, N)
    for r, n in ((0, 65), (63, 64), (64, 2048), (700, 2049), (701, 9000), (N // 2, 300), (N - 1, 4500)):
        lens[r] = n
    rp = np.zeros(N + 1, np.int32); np.cumsum(lens, out=rp[1:])
    ci = rng.integers(0, N, rp[-1]).astype(np.int32)
    v = (rng.random(rp[-1]) * 0.5).astype(np.float32)
    gen = torch.Generator(device=gpu).manual_seed(C)
    x = torch.rand(N, C, generator=gen, device=gpu) - 0.25
    W = torch.randn(C, C, generator=gen, device=gpu) * 0.1
    msg = torch.randn(N, C, generator=gen, device=gpu)
    A = [_t(a, gpu) for a in (rp, ci, v)]
    A64 = torch.sparse_csr_tensor(A[0].long(), A[1].long(), A[2].double(), (N, N))
    # a chunk of 2,048 entries is summed in order and the chunks after it, then C products: an fp32 sum of t terms is within t 2^-24 of
    # the sum of their magnitudes, and nothing near that far
    bound = (2048 + 5 + C) * 2.0 ** -24

    def close(got, left, right, extra=None, mask=None):
        want, terms = left[0] @ right, left[1] @ right.abs()
        if extra is not None:
            want, terms = (want + extra).clamp(min=0), terms + extra.abs()
        if mask is not None:
            want = want * mask
        assert bool(((got.double() - want).abs() <= bound * terms).all())

    agg = (A64 @ x.double(), A64 @ x.double().abs())
    got = ops.s2v_level(*A, x, W, msg)
    close(got, agg, W.double(), msg.double())
    with ops.CsrPlan(*A, N, N) as plan:
        assert torch.equal(plan.level(x, W, msg), got)
    acc = msg.clone()
    u, g = ops.s2v_level_backward(*A, x, W, gate_h=msg, acc=acc)
    assert bool(((u.double() - agg[0]).abs() <= bound * agg[1]).all())
    close(g, agg, W.double().T.contiguous(), mask=(msg > 0).double())
    assert torch.equal(acc, msg + g)
    Wn = torch.randn(5, C, generator=gen, device=gpu)
    X = torch.rand(N, 5, generator=gen, device=gpu)
    S = (torch.tensor([0, N], device=gpu).int(), torch.arange(N, device=gpu).int(), torch.ones(N, device=gpu))
    bufs = ops.s2v_forward(A, S, X, Wn, W, torch.zeros(C, 4, device=gpu), torch.zeros(4, 2, device=gpu), 1)
    h0 = A64 @ bufs.msg.clamp(min=0).double()
    close(bufs.h_final, (h0, h0), W.double(), bufs.msg.double())


@pytest.mark.parametrize("C", [128, 256])
@pytest.mark.parametrize("nnz", [0, 3, 6])
def test_level_backward_wide_with_hardly_any_entries(gpu, oracle, C, nnz):
    """the wide kernel's backward variant on a transposed adjacency with fewer entries than one index batch (and none)"""
    from graphnn_amd import ops
    rng = np.random.default_rng(C + nnz)
    N = 40
    rows = np.sort(rng.integers(0, N, nnz))
    rp = np.zeros(N + 1, np.int32); np.cumsum(np.bincount(rows, minlength=N), out=rp[1:])
    ci = rng.integers(0, N, nnz).astype(np.int32)
    v = (0.5 + rng.random(nnz)).astype(np.float32)
    dz = rng.standard_normal((N, C)).astype(np.float32)
    W = (rng.standard_normal((C, C)) * 0.1).astype(np.float32)
    h_prev = rng.standard_normal((N, C)).astype(np.float32)
    acc0 = rng.standard_normal((N, C)).astype(np.float32)
    acc = _t(acc0, gpu)
    pad = lambda a, dt: _t(np.concatenate([a, np.zeros(1, dt)]), gpu)[:a.size]      # never a null pointer for an empty array
    u, g = ops.s2v_level_backward(_t(rp, gpu), pad(ci, np.int32), pad(v, np.float32), _t(dz, gpu), _t(W, gpu), gate_h=_t(h_prev, gpu), acc=acc)
    import scipy.sparse as sp
    u64 = sp.csr_matrix((v.astype(np.float64), ci, rp), shape=(N, N)) @ dz.astype(np.float64)
    g64 = (u64 @ W.astype(np.float64).T) * (h_prev > 0)
    w_u = oracle.spmm(rp, ci, v, dz, N)
    w_g = (oracle.gemm(w_u, W, transB=True) * (h_prev > 0)).astype(np.float32)
    assert_parity("u", _n(u), w_u, u64)
    assert_parity("g_prev", _n(g), w_g, g64)
    assert np.array_equal(_n(acc), acc0 + _n(g))


def test_grad_gate_is_exact(gpu):
    import torch
    from graphnn_amd import ops
    rng = np.random.default_rng(3)
    n = 100003
    h = np.maximum(rng.standard_normal(n), 0).astype(np.float32); h[5] = -0.0; h[6] = np.nan
    g = rng.standard_normal(n).astype(np.float32)
    acc0 = rng.standard_normal(n).astype(np.float32)
    dz = torch.empty(n, device=gpu); acc = _t(acc0, gpu)
    ops.grad_gate(_t(h, gpu), _t(g, gpu), dz, acc, accumulate=True)
    want = np.where(h > 0, g, 0).astype(np.float32)
    assert np.array_equal(_n(dz), want) and np.array_equal(_n(acc), acc0 + want)
    gd = _t(g, gpu)
    ops.grad_gate(_t(h, gpu), gd, gd, acc, accumulate=False)            # in place, acc overwritten
    assert np.array_equal(_n(gd), want) and np.array_equal(_n(acc), want)


@pytest.mark.parametrize("momentum", [0.9, 0.0])
def test_momentum_sgd_batch_two_steps(gpu, oracle, momentum):
    from graphnn_amd import ops
    rng = np.random.default_rng(17)
    shapes = [(38, 64), (64, 64), (64, 32), (32, 2), (1,), (100003,)]
    lr, l2 = 0.05, 0.01
    w = [rng.standard_normal(s).astype(np.float32) for s in shapes]
    v = [np.zeros(s, np.float32) for s in shapes]
    wd, vd = [_t(a, gpu) for a in w], [_t(a, gpu) for a in v]
    for step in range(2):
        g = [rng.standard_normal(s).astype(np.float32) for s in shapes]
        gd = [_t(a, gpu) for a in g]
        ops.momentum_sgd_batch(wd, gd, vd if momentum > 0 else None, lr, momentum, l2)
        for i in range(len(shapes)):
            w[i], g0, v[i] = oracle.momentum_sgd(w[i], g[i], v[i], lr, momentum, l2)
            assert not _n(gd[i]).any()
            assert np.allclose(_n(wd[i]), w[i], rtol=1e-6, atol=1e-7), (step, i)
            if momentum > 0:
                assert np.allclose(_n(vd[i]), v[i], rtol=1e-6, atol=1e-7), (step, i)


@pytest.mark.parametrize("clip,l2", [(5.0, 0.01), (0.0, 0.0), (1e6, 0.3)])
def test_adam_batch_three_steps(gpu, oracle, clip, l2):
    """AdamOptimizer::Update over a parameter set in two launches (the norm of all gradients, then the update with
    the clipping factor formed on the device), three consecutive steps: gradients that are clipped (their norm is
    far above 5), not clipped (threshold off or out of reach), 18 tensors (more than one table), one of them large"""
    from graphnn_amd import ops
    rng = np.random.default_rng(23)
    shapes = [(38, 64), (64, 64), (64, 32), (32, 2), (1,), (300007,)] + [(5, 3)] * 12
    lr, b1, b2, eps = 0.01, 0.9, 0.999, 1e-8
    w = [rng.standard_normal(s).astype(np.float32) for s in shapes]
    m = [np.zeros(s, np.float32) for s in shapes]
    v = [np.zeros(s, np.float32) for s in shapes]
    wd, md, vd = [_t(a, gpu) for a in w], [_t(a, gpu) for a in m], [_t(a, gpu) for a in v]
    for step in range(1, 4):
        g = [(rng.standard_normal(s) * (0.02 if step == 3 else 1.0)).astype(np.float32) for s in shapes]
        gd = [_t(a, gpu) for a in g]
        ops.adam_batch(wd, gd, md, vd, lr, l2, clip, b1, b2, eps, step)
        scale = oracle.clip_factor(g, clip) if clip > 0 else 1.0
        if clip == 5.0:
            assert (scale < 0.05) == (step < 3)
        for i in range(len(shapes)):
            # where weight decay and the scaled gradient cancel (l2 w = -scale g to four digits) the sum carries the
            # last bits of the clipping factor, which the device forms in double: those elements are left out
            parts = np.abs(l2 * w[i]) + np.abs(scale * g[i])
            steady = np.abs(l2 * w[i] + scale * g[i]) > 1e-3 * parts
            w[i], g0, m[i], v[i] = oracle.adam(w[i], g[i], m[i], v[i], lr, l2, scale, b1, b2, eps, step)
            assert not _n(gd[i]).any()
            assert steady.size < 1000 or steady.mean() > 0.99
            # both sides round b m + (1 - b) g term by term, the device with one fused step: an ulp of the larger term
            assert np.allclose(_n(md[i]), m[i], rtol=2e-6, atol=1e-6), (step, i)
            assert np.allclose(_n(vd[i]), v[i], rtol=4e-6, atol=1e-6), (step, i)
            assert np.allclose(_n(wd[i])[steady], w[i][steady], rtol=1e-6, atol=2e-7), (step, i)
            assert np.allclose(_n(wd[i]), w[i], rtol=0, atol=2.1 * lr), (step, i)
            # the device's own values go on, so that a left-out element does not carry into the next step
            w[i], m[i], v[i] = _n(wd[i]).copy(), _n(md[i]).copy(), _n(vd[i]).copy()


def _dense(csr, rows, cols):
    import scipy.sparse as sp
    return sp.csr_matrix((csr[2].astype(np.float64), csr[1], csr[0]), shape=(rows, cols)).toarray()


@pytest.mark.parametrize("config_id,C", [(1, 64), (2, 64), (1, 128)])
def test_training_iteration_composed_from_the_c_abi(gpu, oracle, config_id, C):
    """forward with every level kept, loss tail, backward (readout backward; per level gate, A^T dz, (.) W^T;
    the weight gradients as four products) and one momentum-SGD update: gradients against float64 autograd
    of the same network at 1e-4, updated weights against the oracle's update of those gradients"""
    import torch
    from graphnn_amd import ops
    batch, w, cfg = synth.make_config(config_id)
    K, H, Q, L = cfg["K"], cfg["H"], cfg["Q"], cfg["L"]
    if C != cfg["C"]:
        w = synth.make_weights(synth.Stream(900 + C), K, C, H, Q)
    a = batching.node2node_csr(batch.num_nodes, batch.edge_x, batch.edge_y)
    s = batching.subgraph_csr(batch.num_graphs, batch.subg_id, batch.node_idx)
    lab = batch.label_csr()
    X = batch.one_hot()
    N, B = batch.num_nodes, batch.num_graphs
    a_d, s_d, lab_d = ([_t(x, gpu) for x in m] for m in (a, s, lab))
    Wn, Wc, W1, W2 = (_t(m, gpu) for m in (w.W_n2l, w.W_conv, w.W_h1, w.W_h2))
    X_d = _t(X, gpu)
    # ---- forward, embeddings of all levels stacked
    hs = torch.empty((L + 1, N, C), device=gpu)
    msg, h0 = ops.s2v_input(X_d, Wn)
    hs[0] = h0
    for l in range(L):
        ops.s2v_level(*a_d, hs[l], Wc, msg, out=hs[l + 1])
    pool, hidden, logits, probs, pred = ops.s2v_readout(*s_d, hs[L], W1, W2, B)
    loss, acc, probs2, _, _ = ops.loss_acc(logits, *lab_d)
    # ---- backward
    dl, du, g = ops.readout_backward(s_d, probs2, lab_d, 1.0 / B, hidden, W1, W2, N)
    at = ops.csr_transpose(*a_d, N, N)
    us = torch.empty((L, N, C), device=gpu)
    dmsg = torch.empty((N, C), device=gpu)
    g2 = torch.empty_like(g)
    ops.grad_gate(hs[L], g, g, dmsg, accumulate=False)
    for l in range(L, 0, -1):
        # the gradient comes out past the gate of the level below and is added to the msg gradient on the way
        ops.s2v_level_backward(*at, g, Wc, u=us[l - 1], g_prev=g2, gate_h=hs[l - 1], acc=dmsg)
        g, g2 = g2, g
    gWc = ops.gemm(hs[:L].reshape(L * N, C), us.reshape(L * N, C), transA=True)
    gWn = ops.gemm(X_d, dmsg, transA=True)
    gW1 = ops.gemm(pool, du, transA=True)
    gW2 = ops.gemm(hidden, dl, transA=True)
    # ---- float64 autograd of the same network
    t64 = lambda m: torch.tensor(np.asarray(m, np.float64), requires_grad=True)
    P = [t64(m) for m in (w.W_n2l, w.W_conv, w.W_h1, w.W_h2)]
    A = torch.tensor(_dense(a, N, N)); S = torch.tensor(_dense(s, B, N)); X64 = torch.tensor(X.astype(np.float64))
    m64 = X64 @ P[0]
    h64 = torch.relu(m64)
    for _ in range(L):
        h64 = torch.relu((A @ h64) @ P[1] + m64)
    lg64 = torch.relu((S @ h64) @ P[2]) @ P[3]
    loss64 = torch.nn.functional.cross_entropy(lg64, torch.tensor(batch.graph_label.astype(np.int64)))
    loss64.backward()
    assert abs(float(_n(loss)[0]) - float(loss64)) <= 1e-5 * abs(float(loss64))
    for name, got, p in (("w_n2l", gWn, P[0]), ("w_conv", gWc, P[1]), ("w_h1", gW1, P[2]), ("w_h2", gW2, P[3])):
        err = max_rel(_n(got), p.grad.numpy())
        print("gradient %s: max_rel %.2e against float64" % (name, err))
        assert err < PARITY_TOL, name
    # ---- one update of all four tensors in one launch
    ws = [Wn.clone(), Wc.clone(), W1.clone(), W2.clone()]
    gs = [gWn.clone(), gWc.clone(), gW1.clone(), gW2.clone()]
    vs = [torch.zeros_like(t) for t in ws]
    ops.momentum_sgd_batch(ws, gs, vs, 0.01, 0.9, 1e-4)
    for t, w0, g0 in zip(ws, (w.W_n2l, w.W_conv, w.W_h1, w.W_h2), (gWn, gWc, gW1, gW2)):
        want_w, _, _ = oracle.momentum_sgd(w0, _n(g0), np.zeros_like(w0), 0.01, 0.9, 1e-4)
        assert np.allclose(_n(t), want_w, rtol=1e-6, atol=1e-8)


def _relative_errors(got, want, terms):
    """rms and mean of the errors, each against the sum of its terms' magnitudes (float64 tensors)"""
    e = (got.double() - want) / terms
    return float(e.square().mean().sqrt()), float(e.mean())


@pytest.mark.parametrize("C", [16, 32, 64])
@pytest.mark.parametrize("N", [1, 15, 16, 17, 31, 1000, 24_561, 24_576])
def test_level_of_a_small_batch_has_the_bits_of_a_large_one(gpu, C, N):
    """up to 24,576 rows a level runs a workgroup per 16-row tile, beyond that the streaming kernel: the same rows followed by
    empty ones until the other kernel takes over give the same bits, forward and backward, with and without msg, bias, gate
    and gradient sum; rows of 0, 4, 5, 8, 9, 16, 17, 48, 49 and 200 entries (taken at once, in a loop, by the whole wavefront)"""
    import torch
    from graphnn_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(C + N)
    normal = lambda *shape: torch.randn(*shape, generator=gen, device=gpu)
    lens = torch.tensor([0, 4, 5, 2, 8, 9, 1, 16, 17, 3, 48, 49, 0, 200, 2, 2, 1], device=gpu).repeat(N // 17 + 1)[:N]
    if N > 2000:
        lens = torch.where(torch.arange(N, device=gpu) % 1700 < 1600, lens.clamp(max=3), lens)
    more = 24_577 + 13 - N                                  # empty rows behind them
    grow = lambda x: torch.cat([x, normal(more, x.shape[1])])
    rp = torch.zeros(N + 1, dtype=torch.int32, device=gpu)
    rp[1:] = torch.cumsum(lens, 0)
    nnz = int(rp[-1])
    ci = torch.randint(0, N, (nnz,), generator=gen, device=gpu).int()
    v = normal(nnz)
    rp_more = torch.cat([rp, rp[-1:].expand(more)])
    h, W, msg, bias, gate, acc0 = normal(N, C), normal(C, C) * 0.2, normal(N, C), normal(C), normal(N, C), normal(N, C)
    h_more, msg_more, gate_more, acc_more0 = grow(h), grow(msg), grow(gate), grow(acc0)
    for m, b in ((None, None), (msg, None), (msg, bias)):
        got = ops.s2v_level(rp, ci, v, h, W, m, b)
        want = ops.s2v_level(rp_more, ci, v, h_more, W, None if m is None else msg_more, b)
        assert torch.equal(got, want[:N])
    for g, a in ((None, None), (gate, None), (gate, acc0), (None, acc0)):
        acc = None if a is None else acc0.clone()
        acc_more = None if a is None else acc_more0.clone()
        u, out = ops.s2v_level_backward(rp, ci, v, h, W, gate_h=g, acc=acc)
        u_more, out_more = ops.s2v_level_backward(rp_more, ci, v, h_more, W, gate_h=None if g is None else gate_more, acc=acc_more)
        assert torch.equal(u, u_more[:N]) and torch.equal(out, out_more[:N])
        assert a is None or torch.equal(acc, acc_more[:N])


@pytest.mark.parametrize("N", [12_288, 12_289, 24_576])
def test_level_of_long_rows_at_hidden_16_has_the_same_bits_either_way(gpu, N):
    """from 12,289 rows on the entry count decides whether a level at hidden 16 runs a workgroup per tile or the streaming kernel: a
    count of zero takes the former; rows of 0 to 60 entries, 24 on average, and a few of 200"""
    import torch
    from graphnn_amd import ops
    C = 16
    gen = torch.Generator(device=gpu).manual_seed(N)
    normal = lambda *shape: torch.randn(*shape, generator=gen, device=gpu)
    lens = torch.tensor([0, 60, 5, 24, 48, 49, 17, 16, 3, 15, 23, 31], device=gpu).repeat(N // 12 + 1)[:N]
    lens[N // 3:N // 3 + 5] = 200
    rp = torch.zeros(N + 1, dtype=torch.int32, device=gpu)
    rp[1:] = torch.cumsum(lens, 0)
    nnz = int(rp[-1])
    assert 20 * N < nnz < 25 * N
    ci, v = torch.randint(0, N, (nnz,), generator=gen, device=gpu).int(), normal(nnz)
    h, W, msg, gate, acc0 = normal(N, C), normal(C, C) * 0.2, normal(N, C), normal(N, C), normal(N, C)
    assert torch.equal(ops.s2v_level(rp, ci, v, h, W, msg), ops.s2v_level(rp, ci, v, h, W, msg, nnz_hint=0))
    got = []
    for count in (nnz, 0):
        u, out, acc = torch.empty_like(h), torch.empty_like(h), acc0.clone()
        ops._bound().s2v_level_backward_f32(N, C, count, rp, ci, v, h, W, u, out, gate, acc)
        got.append((u, out, acc))
    assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("C", [5, 36, 100, 127])
def test_level_of_any_hidden_size_has_the_same_bits_whatever_the_tile(gpu, C):
    """levels of hidden sizes without a kernel of their own take 16, 32 or 64 rows per workgroup by the number of rows: the same rows
    followed by empty ones, up to and past each of the turns, give the same bits forward, backward and in the input stage"""
    import torch
    from graphnn_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(C)
    normal = lambda *shape: torch.randn(*shape, generator=gen, device=gpu)
    most, N = 49_153, 1003
    # (rows of more than 64 entries change their order with the balanced pass, from 32,768 rows on)
    lens = torch.tensor([0, 4, 5, 2, 8, 9, 1, 16, 17, 3, 48, 49, 0, 64, 2, 2, 1], device=gpu).repeat(N // 17 + 1)[:N]
    rp = torch.zeros(N + 1, dtype=torch.int32, device=gpu)
    rp[1:] = torch.cumsum(lens, 0)
    nnz = int(rp[-1])
    ci, v = torch.randint(0, N, (nnz,), generator=gen, device=gpu).int(), normal(nnz)
    h, W, msg, gate, acc0, X, Wn = normal(most, C), normal(C, C) * 0.2, normal(most, C), normal(most, C), normal(most, C), normal(most, 9), normal(9, C)
    want = None
    for n in (N, 16_383, 16_384, 20_001, 40_959, 40_960, 49_152, 49_153):
        rows = torch.cat([rp, rp[-1:].expand(n - N)])
        acc = acc0[:n].clone()
        u, g = ops.s2v_level_backward(rows, ci, v, h[:n], W, gate_h=gate[:n], acc=acc)
        got = [ops.s2v_level(rows, ci, v, h[:n], W, msg[:n]), u, g, acc, *ops.s2v_input(X[:n], Wn)]
        # rows behind the matrix's own: no entries (ReLU(msg), nothing, zero, the old sum), and the last row of every size
        assert torch.equal(got[0][N:], msg[N:n].clamp(min=0)) and not bool(u[N:].any()) and not bool(g[N:].any()) and torch.equal(acc[N:], acc0[N:n])
        assert torch.equal(got[5], got[4].clamp(min=0))
        if want is None:
            want = got
        assert all(torch.equal(x[:N], y[:N]) for x, y in zip(got, want)), n


@pytest.mark.parametrize("C", [128, 256])
@pytest.mark.parametrize("N", [5003, 40_009])
@pytest.mark.parametrize("kind", ["zero_mean", "relu", "one_sign"])
def test_wide_products_in_pieces_are_no_less_exact_than_fp32_ones(gpu, C, N, kind):
    """the contraction of the wide inference level and of the wide level backward (bf16 pieces) against float64, next to the FP32
    matrix cores' (the level of a training forward, a GEMM) on the same operands: the rms of its errors is no larger"""
    import torch
    from graphnn_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(C + N)
    normal = lambda *shape: torch.randn(*shape, generator=gen, device=gpu)
    A = (torch.arange(N + 1, device=gpu).int(), torch.arange(N, device=gpu).int(), torch.ones(N, device=gpu))     # the identity
    W = normal(C, C) * (0.8 / C ** 0.5)
    x = normal(N, C)
    if kind == "relu":
        x = x.clamp(min=0)
    if kind == "one_sign":
        x, W = x.abs(), W.abs()
    fp32 = _relative_errors(ops.gemm(x, W, transB=True), x.double() @ W.double().T.contiguous(), x.double().abs() @ W.double().abs().T.contiguous())
    _, g = ops.s2v_level_backward(*A, x, W)
    pieces = _relative_errors(g, x.double() @ W.double().T.contiguous(), x.double().abs() @ W.double().abs().T.contiguous())
    print("backward: pieces rms %.2e mean %.1e, fp32 rms %.2e mean %.1e" % (pieces + fp32))
    assert pieces[0] <= fp32[0] and abs(pieces[1]) < 0.1 * fp32[0]
    # forward: msg = x W_n2l, h = ReLU(ReLU(msg) W + msg); the outputs that are not cut off
    Wn = normal(64, C) * (0.1 if kind != "one_sign" else 0.0) + (0.1 if kind == "one_sign" else 0.0)
    X = normal(N, 64)
    S = (torch.tensor([0, N], device=gpu).int(), A[1], A[2])
    bufs = ops.s2v_forward(A, S, X, Wn, W, normal(C, 4), normal(4, 2), 1)
    h, msg = bufs.msg.clamp(min=0), bufs.msg
    want = h.double() @ W.double() + msg.double()
    terms = h.double() @ W.double().abs() + msg.double().abs()
    on = want > 0
    fp32 = _relative_errors(ops.s2v_level(*A, h, W, msg)[on], want[on], terms[on])
    pieces = _relative_errors(bufs.h_final[on], want[on], terms[on])
    print("forward: pieces rms %.2e mean %.1e, fp32 rms %.2e mean %.1e" % (pieces + fp32))
    assert pieces[0] <= fp32[0] and abs(pieces[1]) < 0.1 * fp32[0]


@pytest.mark.parametrize("m,n,k", [(256, 256, 8192), (256, 256, 20_011), (255, 33, 40_007), (129, 256, 9_001), (64, 256, 16_385),
                                   (1, 256, 1_048_577), (128, 128, 16_384), (100, 127, 23_456), (65, 64, 65_600), (64, 64, 65_543)])
def test_weight_gradient_over_a_long_k(gpu, m, n, k):
    """A^T B with an output of up to 256 x 256 over a long k (operands in bf16 pieces on the matrix cores, the whole output in
    one workgroup): every tile shape and its transposed form, columns short of a tile, k short of a stage, against float64;
    the error stays within what an fp32 sum of this length has, and the batch call gives the same bits"""
    import torch
    from graphnn_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(m * 1000 + n)
    A = torch.randn(k, m, generator=gen, device=gpu)
    B = torch.randn(k, n, generator=gen, device=gpu) + 0.5
    out0 = torch.randn(m, n, generator=gen, device=gpu)
    got = ops.gemm(A, B, transA=True, alpha=0.5, beta=2.0, out=out0.clone())
    want = 0.5 * (A.double().T.contiguous() @ B.double()) + 2.0 * out0.double()
    terms = 0.5 * (A.double().abs().T.contiguous() @ B.double().abs()) + 2.0 * out0.double().abs()
    assert float(((got.double() - want).abs() / terms).max()) < 1e-6
    assert float((got.double() - want).norm() / want.norm()) < 2e-6
    batched = out0.clone()
    ops.gemm_tn_batch([(A, B, batched)], alpha=0.5, beta=2.0)
    assert torch.equal(batched, got)


@pytest.mark.parametrize("m,n,k", [(64, 64, 70_000), (64, 64, 400_003), (64, 128, 40_000), (128, 128, 20_000), (64, 256, 20_000), (128, 256, 20_011),
                                   (256, 256, 8192), (256, 256, 300_007)])
@pytest.mark.parametrize("kind", ["zero_mean", "relu", "one_sign"])
def test_weight_gradient_in_pieces_is_no_less_exact_than_an_fp32_one(gpu, m, n, k, kind):
    """A^T B over a long k from bf16 pieces against float64, next to the FP32 matrix cores' sum of the same terms (A stored
    transposed takes the general kernel): the rms of its errors is no larger"""
    import torch
    from graphnn_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(m + n + k)
    A, B = torch.randn(k, m, generator=gen, device=gpu), torch.randn(k, n, generator=gen, device=gpu)
    if kind == "relu":
        A = A.clamp(min=0)
    if kind == "one_sign":
        A, B = A.abs(), B.abs()
    At = A.T.contiguous()
    want, terms = At.double() @ B.double(), At.double().abs() @ B.double().abs()
    pieces = _relative_errors(ops.gemm(A, B, transA=True), want, terms)
    fp32 = _relative_errors(ops.gemm(At, B), want, terms)
    print("%s %dx%d k %d: pieces rms %.2e mean %.1e, fp32 rms %.2e mean %.1e" % ((kind, m, n, k) + pieces + fp32))
    assert pieces[0] <= fp32[0] and abs(pieces[1]) < 0.1 * fp32[0]


def _in_pieces(route, gpu, x, W):
    """(x W from bf16 pieces, the same product on the FP32 matrix cores); the wide forward's with negatives cut off in both"""
    import torch
    from graphnn_amd import ops
    N, C = x.shape
    if route == "gradient":
        return ops.gemm(x.T.contiguous(), W, transA=True), ops.gemm(x, W)
    A = (torch.arange(N + 1, device=gpu).int(), torch.arange(N, device=gpu).int(), torch.ones(N, device=gpu))     # the identity
    if route == "backward":
        _, g = ops.s2v_level_backward(*A, x, W.T.contiguous())
        return g, ops.gemm(x, W)
    # msg = the first 64 rows of x in turn; h1 = ReLU(ReLU(msg) W + msg), and the same level by itself
    S = (torch.tensor([0, N], device=gpu).int(), A[1], A[2])
    bufs = ops.ForwardBuffers(N, 1, C, 4, 2, gpu)
    labels = torch.eye(64, device=gpu)[torch.arange(N, device=gpu) % 64].contiguous()
    ops.s2v_forward(A, S, labels, x[:64].contiguous(), W, torch.zeros(C, 4, device=gpu), torch.zeros(4, 2, device=gpu), 1, bufs=bufs)
    return bufs.h_final, ops.s2v_level(*A, bufs.msg.clamp(min=0), W, bufs.msg)


@pytest.mark.parametrize("C", [128, 256])
@pytest.mark.parametrize("route", ["backward", "forward", "gradient"])
@pytest.mark.parametrize("x_size,w_size", [(1e-33, 1.0), (1e-36, 1.0), (3e-38, 8.0), (1e-41, 1e3), (1e-36, 1e36), (1e36, 1e-36), (3e11, 1.0), (1.0, 3e11),
                                           (1e30, 1e-4), (1e18, 1e18), (1e37, 1e-20), (1e-20, 1e37)])
def test_products_in_pieces_over_the_whole_range(gpu, C, route, x_size, w_size):
    """operands anywhere between the smallest floats and the largest: no further from float64 than the FP32 matrix cores"""
    import torch
    N = 20_000 if route == "gradient" else 640
    gen = torch.Generator(device=gpu).manual_seed(C)
    x = torch.randn(N if route != "gradient" else C, C if route != "gradient" else N, generator=gen, device=gpu) * x_size
    W = torch.randn(x.shape[1], C, generator=gen, device=gpu) * w_size
    got, fp32 = _in_pieces(route, gpu, x, W)
    if route == "forward":
        x = x[torch.arange(N, device=gpu) % 64]
        h = x.clamp(min=0).double()
        want, terms = h @ W.double() + x.double(), h @ W.double().abs() + x.double().abs()
    else:
        want, terms = x.double() @ W.double(), x.double().abs() @ W.double().abs()
    on = want > 0 if route == "forward" else torch.ones_like(want, dtype=torch.bool)
    # where the result itself lies at the lower end of the range its own spacing (2^-149) comes on top
    ours, theirs = (float(((t.double() - want).abs() / (terms + 2.0 ** -125))[on].square().mean().sqrt()) for t in (got, fp32))
    print("%s %d, %g * %g: pieces rms %.2e, fp32 rms %.2e" % (route, C, x_size, w_size, ours, theirs))
    assert ours <= 1.05 * theirs


@pytest.mark.parametrize("C", [128, 256])
@pytest.mark.parametrize("route,side", [("backward", "x"), ("backward", "W"), ("forward", "W"), ("gradient", "x"), ("gradient", "W")])
def test_products_in_pieces_carry_infinities_and_nan(gpu, C, route, side):
    """an infinity, a NaN or a product past the largest float on either side, against factors of three pieces whose corrections
    have either sign: the classes (finite, infinite, NaN) and signs of the FP32 matrix cores in every output"""
    import torch
    gen = torch.Generator(device=gpu).manual_seed(7)
    shape = (64, C) if route != "gradient" else (C, 20_000)
    x = 1 + torch.rand(*shape, generator=gen, device=gpu)
    W = 1000 + 1000 * torch.rand(shape[1], C, generator=gen, device=gpu)
    t, at = (x, lambda i: (5 + i, 17 + 3 * i)) if side == "x" else (W, lambda i: (17 + 3 * i, 5 + i))
    for i, v in enumerate([float("inf"), float("-inf"), float("nan"), 3.4e38, -3.4e38, 0.0]):
        t[at(i)] = v
    if side == "x":
        x[30, 4] = x[31, 9] = float("inf")
        W[4, 40], W[9, 41], W[9, 42] = float("inf"), float("-inf"), 0.0        # inf inf, inf -inf, inf 0
    got, fp32 = _in_pieces(route, gpu, x, W)
    assert torch.equal(torch.isnan(got), torch.isnan(fp32))
    assert torch.equal(got == float("inf"), fp32 == float("inf")) and torch.equal(got == float("-inf"), fp32 == float("-inf"))
    finite = torch.isfinite(fp32)
    assert bool(finite.any()) and bool(((got - fp32)[finite].abs() <= 1e-5 * fp32[finite].abs()).all())


def test_weight_gradient_carries_infinities_and_nan(gpu):
    """an infinite or NaN term reaches the outputs it is part of and no others, next to values whose bf16 rounding would overflow"""
    import torch
    from graphnn_amd import ops
    k, m, n = 20_000, 64, 256
    A = torch.zeros(k, m, device=gpu)
    B = torch.ones(k, n, device=gpu)
    A[5, 1], A[6, 2], A[7, 3], A[8, 4] = float("inf"), float("-inf"), float("nan"), 3.4028e38
    got = ops.gemm(A, B, transA=True)
    assert bool((got[1] == float("inf")).all()) and bool((got[2] == float("-inf")).all()) and bool(torch.isnan(got[3]).all())
    assert bool(torch.isfinite(got[4]).all()) and bool((got[0] == 0).all()) and bool((got[5:] == 0).all())
