"""Parity of the HIP path (through the C ABI) with the CPU oracle on identical seeded inputs.

Bit-exact for integer / index outputs and for single-rounding element-wise ops;
PARITY_TOL = 1e-4 under conftest.max_rel (floors measured per tensor kind) for fp32 sums; where two
fp32 summation orders legitimately differ by more, a float64 model of the same computation decides
(conftest.assert_parity).
"""
import ctypes
import json
import os

import numpy as np
import pytest

from conftest import FLOOR_POOL, FLOOR_PROBS_ABS, PARITY_TOL, Lazy, assert_condition, assert_parity, assert_stages, forward_float64, max_rel
from graphnn_amd import batching, synth

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(__file__), "golden")


def _t(a, dev):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def _n(t):
    return t.detach().cpu().numpy()


def _csr_t(csr, dev):
    return tuple(_t(a, dev) for a in csr)


def _random_csr(rng, m, k, nnz, unit=False, sort_cols=False):
    rows = np.sort(rng.integers(0, m, nnz))
    rp = np.zeros(m + 1, np.int32)
    np.cumsum(np.bincount(rows, minlength=m), out=rp[1:])
    ci = rng.integers(0, max(k, 1), nnz).astype(np.int32)
    if sort_cols:
        order = np.lexsort((ci, rows))
        ci = ci[order]
    v = np.ones(nnz, np.float32) if unit else rng.standard_normal(nnz).astype(np.float32)
    return rp, ci, v


# float64 models of the kernels: assert_parity consults them only when a device result misses the oracle
# (both are then fp32 evaluations in different summation orders, and float64 tells which one is off)
def _csr64(rp, v, m, k, ci):
    import scipy.sparse as sp
    return sp.csr_matrix((np.asarray(v, np.float64), ci, rp), shape=(m, k))


def _spmm_want(oracle, rp, ci, v, B, m, alpha=1.0, beta=0.0, C=None):
    want = oracle.spmm(rp, ci, v, B, m, alpha=alpha, beta=beta, C=C)
    def model(mag=lambda x: x):
        y = mag(alpha) * (_csr64(rp, mag(np.asarray(v, np.float64)), m, B.shape[0], ci) @ mag(B.astype(np.float64)))
        return y if C is None else y + mag(beta) * mag(C.astype(np.float64))
    return want, Lazy(model, Lazy(lambda: model(np.abs)))


def _gemm_want(oracle, A, B, ta=False, tb=False, alpha=1.0, beta=0.0, C=None):
    want = oracle.gemm(A, B, ta, tb, alpha=alpha, beta=beta, C=C)
    def model(mag=lambda x: x):
        a64, b64 = mag(A.astype(np.float64)), mag(B.astype(np.float64))
        y = mag(alpha) * ((a64.T if ta else a64) @ (b64.T if tb else b64))
        return y if C is None else y + mag(beta) * mag(C.astype(np.float64))
    return want, Lazy(model, Lazy(lambda: model(np.abs)))


def _level_want(oracle, rp, ci, v, h_in, W, msg=None, bias=None):
    want = oracle.level(rp, ci, v, h_in, W, msg, bias)
    def model(mag=None):
        N = h_in.shape[0]
        f = mag or (lambda x: x)
        z = (_csr64(rp, f(np.asarray(v, np.float64)), N, N, ci) @ f(h_in.astype(np.float64))) @ f(W.astype(np.float64))
        if bias is not None:
            z = z + f(bias.astype(np.float64))
        if msg is not None:
            z = z + f(msg.astype(np.float64))
        return z if mag else np.maximum(z, 0)
    return want, Lazy(model, Lazy(lambda: model(np.abs)))


def _forward_want(oracle, a, s, X, w, L, lab=None):
    """the oracle's forward; want["_f64"] is the lazily computed float64 model of the same network, and carries the
    same network on absolute values as its condition tensors"""
    want = oracle.forward(a, s, X, w, L, lab)
    want["_f64"] = Lazy(lambda: forward_float64(a, s, X, w, L), Lazy(lambda: forward_float64(a, s, X, w, L, magnitudes=True)))
    return want


def _assert_forward_parity(got, want, L, tag="", keys=("msg", "h_final", "pool", "hidden", "logits", "probs")):
    """got: name -> device array.  Floors as measured for each tensor (conftest): pooled features at 1e-4 of
    their scale, probabilities at the fixed 1e-6, the rest at the default; a miss is settled by float64."""
    f64 = want.get("_f64")
    for key in keys:
        ref = want["h"][L] if key == "h_final" else want[key]
        ref64 = None if f64 is None else (f64["h"][L] if key == "h_final" else f64[key])
        kw = {}
        if key == "pool":
            kw["floor_frac"] = FLOOR_POOL
        elif key == "probs":
            kw["floor"] = FLOOR_PROBS_ABS
        assert_parity("%s%s" % (key, tag), got[key], ref, ref64, **kw)


# ------------------------------------------------------------------ SpMM
def test_spmm_known_answer(gpu, oracle):
    from graphnn_amd import ops
    g = json.load(open(os.path.join(GOLDEN, "sparse_mm_known_answer.json")))
    csr = (np.array(g["row_ptr"], np.int32), np.array(g["col_idx"], np.int32), np.array(g["val"], np.float32))
    B = np.array(g["b_for_normal"], np.float32)
    got = _n(ops.spmm(*_csr_t(csr, gpu), _t(B, gpu), g["a_rows"]))
    assert np.array_equal(got, np.array(g["expected_A_b"], np.float32))


@pytest.mark.parametrize("n", [1, 2, 3, 4, 7, 16, 32, 64, 100, 128, 256, 300, 512, 1100])
def test_spmm_widths_random_values(gpu, oracle, n):
    from graphnn_amd import ops
    rng = np.random.default_rng(100 + n)
    m, k = 517, 389                        # not multiples of any group count
    csr = _random_csr(rng, m, k, 4000)
    B = rng.standard_normal((k, n)).astype(np.float32)
    C0 = rng.standard_normal((m, n)).astype(np.float32)
    want, w64 = _spmm_want(oracle, *csr, B, m)
    got = _n(ops.spmm(*_csr_t(csr, gpu), _t(B, gpu), m))
    assert_parity("spmm", got, want, w64)
    want2, w64b = _spmm_want(oracle, *csr, B, m, alpha=0.5, beta=-2.0, C=C0)
    got2 = _n(ops.spmm(*_csr_t(csr, gpu), _t(B, gpu), m, alpha=0.5, beta=-2.0, out=_t(C0, gpu)))
    assert_parity("spmm", got2, want2, w64b)


@pytest.mark.parametrize("n", [2, 64, 128, 256])
def test_spmm_unit_weights_bit_exact(gpu, oracle, n):
    """unit edge weights and row-order accumulation: same additions in the same order as the oracle"""
    from graphnn_amd import ops
    rng = np.random.default_rng(200 + n)
    m = 3001
    csr = _random_csr(rng, m, m, 30000, unit=True, sort_cols=True)
    B = rng.standard_normal((m, n)).astype(np.float32)
    got = _n(ops.spmm(*_csr_t(csr, gpu), _t(B, gpu), m))
    assert np.array_equal(got, oracle.spmm(*csr, B, m))


def test_spmm_edge_cases(gpu, oracle):
    from graphnn_amd import ops
    import torch
    rng = np.random.default_rng(3)
    n = 64
    # all rows empty; beta = 0 must overwrite NaN garbage
    rp = np.zeros(11, np.int32)
    ci = np.zeros(0, np.int32); v = np.zeros(0, np.float32)
    B = rng.standard_normal((5, n)).astype(np.float32)
    out = torch.full((10, n), float("nan"), device=gpu)
    got = _n(ops.spmm(_t(rp, gpu), _t(ci, gpu), _t(v, gpu), _t(B, gpu), 10, out=out))
    assert np.array_equal(got, np.zeros((10, n), np.float32))
    # identity
    m = 300
    eye = (np.arange(m + 1, dtype=np.int32), np.arange(m, dtype=np.int32), np.ones(m, np.float32))
    X = rng.standard_normal((m, n)).astype(np.float32)
    assert np.array_equal(_n(ops.spmm(*_csr_t(eye, gpu), _t(X, gpu), m)), X)
    # single row, single column
    one = (np.array([0, 3], np.int32), np.array([0, 0, 0], np.int32), np.array([1, 2, 3], np.float32))
    X1 = rng.standard_normal((1, 4)).astype(np.float32)
    assert max_rel(_n(ops.spmm(*_csr_t(one, gpu), _t(X1, gpu), 1)), oracle.spmm(*one, X1, 1)) < PARITY_TOL
    # operand validation happens on the host
    with pytest.raises(ValueError):
        ops.spmm(_t(rp, gpu), _t(ci, gpu), _t(v, gpu), _t(B, gpu), 12)


@pytest.mark.parametrize("n", [64, 128, 6])
def test_spmm_long_rows(gpu, oracle, n):
    """rows far longer than the per-group limit take the whole-workgroup path (hub vertices)"""
    from graphnn_amd import ops
    rng = np.random.default_rng(4)
    m, k = 70, 5000
    lens = rng.integers(0, 12, m)
    lens[3] = 5000; lens[4] = 2049; lens[40] = 9000; lens[69] = 2048
    rp = np.zeros(m + 1, np.int32); np.cumsum(lens, out=rp[1:])
    nnz = int(rp[-1])
    ci = rng.integers(0, k, nnz).astype(np.int32)
    v = rng.standard_normal(nnz).astype(np.float32)
    B = rng.standard_normal((k, n)).astype(np.float32)
    want, w64 = _spmm_want(oracle, rp, ci, v, B, m)
    got = _n(ops.spmm(_t(rp, gpu), _t(ci, gpu), _t(v, gpu), _t(B, gpu), m))
    assert_parity("spmm", got, want, w64)
    # twice the same input: identical bits (no atomics, fixed combination order)
    got_again = _n(ops.spmm(_t(rp, gpu), _t(ci, gpu), _t(v, gpu), _t(B, gpu), m))
    assert np.array_equal(got, got_again)


# ------------------------------------------------------------------ GEMM
@pytest.mark.parametrize("shape", [(1, 1, 1), (7, 5, 3), (64, 64, 16), (65, 63, 17), (300, 2, 32), (1000, 64, 38), (33, 130, 70),
                                   (5000, 1, 64), (4097, 2, 32), (6000, 3, 8), (5001, 4, 260), (5000, 1, 4), (5003, 3, 256),
                                   (600_001, 2, 64),           # more rows than the row-strided kernel has lane groups
                                  
                                   # few output tiles, long k (weight gradients): the product is split along k
                                   (64, 64, 7450), (38, 64, 7450), (70, 130, 3000), (64, 32, 1024), (2, 64, 4099)])
def test_gemm_all_transposes(gpu, oracle, shape):
    from graphnn_amd import ops
    m, n, k = shape
    rng = np.random.default_rng(sum(shape))
    for ta in (False, True):
        for tb in (False, True):
            A = rng.standard_normal((k, m) if ta else (m, k)).astype(np.float32)
            B = rng.standard_normal((n, k) if tb else (k, n)).astype(np.float32)
            C0 = rng.standard_normal((m, n)).astype(np.float32)
            got = _n(ops.gemm(_t(A, gpu), _t(B, gpu), ta, tb))
            assert_parity("gemm %d%d" % (ta, tb), got, *_gemm_want(oracle, A, B, ta, tb))
            got2 = _n(ops.gemm(_t(A, gpu), _t(B, gpu), ta, tb, alpha=1.5, beta=-0.5, out=_t(C0, gpu)))
            assert_parity("gemm %d%d" % (ta, tb), got2, *_gemm_want(oracle, A, B, ta, tb, alpha=1.5, beta=-0.5, C=C0))


@pytest.mark.parametrize("k,c", [(8192, 128), (20_003, 128), (8191, 256), (8192, 256), (40_001, 256), (300_007, 256)])
def test_gemm_wide_weight_gradient_over_a_long_k(gpu, oracle, k, c):
    """h^T u with a 128 x 128 or 256 x 256 output and k in the thousands to hundreds of thousands (the level weight gradient
    at hidden 128 / 256): from k = 8,192 the whole output lives in one workgroup's registers, each workgroup a range of k
    (ranges that end inside a step of 16 rows, one row short of the threshold, a last range shorter than the others);
    alone and inside a batch: same bits"""
    from graphnn_amd import ops
    rng = np.random.default_rng(k + c)
    A = (rng.standard_normal((k, c)) * (rng.random((k, c)) < 0.6)).astype(np.float32)      # embeddings past a ReLU: many zeros
    B = rng.standard_normal((k, c)).astype(np.float32)
    C0 = rng.standard_normal((c, c)).astype(np.float32)
    got = _n(ops.gemm(_t(A, gpu), _t(B, gpu), True, False))
    assert_parity("gemm 10", got, *_gemm_want(oracle, A, B, True, False))
    assert np.array_equal(got, _n(ops.gemm(_t(A, gpu), _t(B, gpu), True, False)))           # fixed order of the ranges
    got2 = _n(ops.gemm(_t(A, gpu), _t(B, gpu), True, False, alpha=0.5, beta=1.0, out=_t(C0, gpu)))
    assert_parity("gemm 10", got2, *_gemm_want(oracle, A, B, True, False, alpha=0.5, beta=1.0, C=C0))
    if k == 20_003 or k == 40_001:
        # the operands as the leading columns of wider matrices (row strides of c + 64 and c + 4 floats)
        Aw = np.concatenate([A, rng.standard_normal((k, 64)).astype(np.float32)], axis=1)
        Bw = np.concatenate([B, rng.standard_normal((k, 4)).astype(np.float32)], axis=1)
        assert np.array_equal(_n(ops.gemm(_t(Aw, gpu), _t(Bw, gpu), True, False, cols_a=c, cols_b=c)), got)
    small = lambda: (_t(A[:300, :64].copy(), gpu), _t(B[:300, :32].copy(), gpu), _t(C0[:64, :32].copy(), gpu))
    outs = ops.gemm_tn_batch([small(), (_t(A, gpu), _t(B, gpu), _t(C0, gpu)), small()], alpha=0.5, beta=1.0)
    assert np.array_equal(_n(outs[1]), got2)
    assert np.array_equal(_n(outs[0]), _n(outs[2]))
    assert_parity("gemm batch", _n(outs[0]), *_gemm_want(oracle, A[:300, :64], B[:300, :32], True, False, alpha=0.5, beta=1.0, C=C0[:64, :32]))


@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (1.0, 1.0), (-0.75, 0.5)])
def test_gemm_batch_of_weight_gradient_products(gpu, oracle, alpha, beta):
    """the four x^T dy products at the end of a configuration-2 backward pass, a product too short to split, one that
    covers several output tiles, an empty one and a single element, in two launches: each against the oracle, and
    bit-identical to the same product through gnnhip_gemm_f32 where that call splits k too"""
    from graphnn_amd import ops
    rng = np.random.default_rng(77)
    shapes = [(29800, 64, 64), (7450, 38, 64), (256, 64, 32), (256, 32, 2), (100, 20, 30), (3000, 150, 70), (40, 0, 5),
              (1, 1, 1), (513, 64, 64)]                       # (k, m, n); nine products: more than one table
    host = []
    products = []
    for k, m, n in shapes:
        A = rng.standard_normal((k, m)).astype(np.float32); B = rng.standard_normal((k, n)).astype(np.float32)
        C0 = rng.standard_normal((m, n)).astype(np.float32)
        host.append((A, B, C0))
        products.append((_t(A, gpu), _t(B, gpu), _t(C0, gpu)))
    outs = ops.gemm_tn_batch(products, alpha=alpha, beta=beta)
    for (k, m, n), (A, B, C0), got in zip(shapes, host, outs):
        if m == 0:
            continue
        assert_parity("gemm batch k=%d m=%d n=%d" % (k, m, n), _n(got), *_gemm_want(oracle, A, B, True, False, alpha=alpha, beta=beta, C=C0))
        alone = _n(ops.gemm(_t(A, gpu), _t(B, gpu), True, False, alpha=alpha, beta=beta, out=_t(C0, gpu)))
        if k >= 256 and m <= 512 and n <= 512:
            assert np.array_equal(_n(got), alone), (k, m, n)


@pytest.mark.parametrize("m,n", [(1, 1), (2, 64), (3, 5), (4, 4), (5, 63), (38, 64), (64, 3), (63, 65), (67, 66), (66, 130), (577, 520)])
@pytest.mark.parametrize("k", [1, 3, 15, 16, 17, 33, 63, 64, 255, 256, 257, 545, 4099])
def test_transposed_product_at_the_edges_of_its_tiles(gpu, m, n, k):
    """A^T B around the sizes where its kernel turns: fewer than four columns, units of four that are moved back, one and several
    64 x 64 tiles, k short of a step of 16 rows, of a wavefront's four rows of it and of the four steps under way, one and
    several ranges; the operands are the leading columns of wider rows that start at any float, with NaN behind the columns
    and infinities behind the rows.  Every element within k + 8 roundings of the sum of its terms' magnitudes of float64
    (one per product and sum, and those of alpha and beta), and the same bits from the batch call"""
    import torch
    from graphnn_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(1000 * m + n + k)
    def operand(cols, pad):
        rows = torch.full((k + 3, cols + pad), float("nan"), device=gpu)
        rows[k:] = float("inf")
        rows[:k, :cols] = torch.randn(k, cols, generator=gen, device=gpu)
        return rows
    for pad_a, pad_b, alpha, beta in ((0, 0, 1.0, 0.0), (3, 1, -0.75, 0.5)):
        A, B = operand(m, pad_a), operand(n, pad_b)
        if pad_a:                                       # rows that start at odd floats
            A = torch.cat([torch.full((1,), float("nan"), device=gpu), A.reshape(-1)])[1:].view(k + 3, m + pad_a)
        out0 = torch.randn(m, n, generator=gen, device=gpu)
        a64, b64 = A[:k, :m].double(), B[:k, :n].double()
        want = alpha * (a64.T.contiguous() @ b64) + beta * out0.double()
        terms = abs(alpha) * (a64.abs().T.contiguous() @ b64.abs()) + abs(beta) * out0.double().abs()
        got = ops.gemm(A[:k], B[:k], transA=True, alpha=alpha, beta=beta, out=out0.clone(), cols_a=m, cols_b=n)
        assert bool(((got.double() - want).abs() <= (k + 8) * 2.0 ** -24 * terms).all())
        if pad_a == 0:
            batched = out0.clone()
            ops.gemm_tn_batch([(A[:k], B[:k], batched), (A[:k], B[:k], torch.empty_like(out0))], alpha=alpha, beta=beta)
            assert torch.equal(batched, got)


@pytest.mark.parametrize("m,n", [(1, 1), (16, 16), (17, 33), (32, 32), (25, 41), (16, 65), (64, 2), (7, 256), (65, 64), (130, 66)])
@pytest.mark.parametrize("k", [0, 1, 2, 4, 5, 31, 32, 33, 47, 48, 49])
def test_transposed_product_over_few_rows(gpu, m, n, k):
    """A^T B over up to 32 rows, and up to 48 where the output has at most 1,024 elements, without sharing the rows between wavefronts:
    NaN behind the columns and infinities behind the rows are not read into the result.  Every element within k + 8 roundings of
    the sum of its terms' magnitudes of float64 (one per product and sum, and those of alpha and beta); the same bits from a batch
    of products, short and long ones"""
    import torch
    from graphnn_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(1000 * m + n + k)
    def operand(rows, cols, pad):
        held = torch.full((rows + 3, cols + pad), float("nan"), device=gpu)
        held[rows:] = float("inf")
        held[:rows, :cols] = torch.randn(rows, cols, generator=gen, device=gpu)
        return held
    for pad, alpha, beta in ((0, 1.0, 0.0), (3, -0.75, 0.5)):
        A, B = operand(k, m, pad), operand(k, n, pad)
        out0 = torch.randn(m, n, generator=gen, device=gpu)
        a64, b64 = A[:k, :m].double(), B[:k, :n].double()
        want = alpha * (a64.T.contiguous() @ b64) + beta * out0.double()
        terms = abs(alpha) * (a64.abs().T.contiguous() @ b64.abs()) + abs(beta) * out0.double().abs()
        got = ops.gemm(A[:k], B[:k], transA=True, alpha=alpha, beta=beta, out=out0.clone(), cols_a=m, cols_b=n)
        assert bool(((got.double() - want).abs() <= (k + 8) * 2.0 ** -24 * terms).all())
        if pad == 0:
            long_a, long_b = operand(400, 20, 0)[:400], operand(400, 30, 0)[:400]
            batched = [out0.clone() for _ in range(2)]
            ops.gemm_tn_batch([(A[:k], B[:k], batched[0]), (long_a, long_b, torch.zeros(20, 30, device=gpu)), (A[:k], B[:k], batched[1])],
                              alpha=alpha, beta=beta)
            assert torch.equal(batched[0], got) and torch.equal(batched[1], got)


@pytest.mark.parametrize("m,n,k", [(1409, 1473, 127), (1409, 1473, 128), (1409, 1473, 131), (33, 32_705, 141), (1409, 1472, 33)])
def test_transposed_product_of_many_tiles(gpu, m, n, k):
    """A^T B of more than 512 tiles over 128 rows and more, one row less, and few rows: every element within k + 8 roundings of the sum of its
    terms' magnitudes of float64, and the bits that the same columns have as an output of a few tiles"""
    import torch
    from graphnn_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(m + k)
    A, B = torch.randn(k, m, generator=gen, device=gpu), torch.randn(k, n, generator=gen, device=gpu)
    got = ops.gemm(A, B, transA=True)
    want, terms = A.double().T.contiguous() @ B.double(), A.double().abs().T.contiguous() @ B.double().abs()
    assert bool(((got.double() - want).abs() <= (k + 8) * 2.0 ** -24 * terms).all())
    few = ops.gemm(A, B, transA=True, cols_a=min(m, 128), cols_b=128)
    assert torch.equal(few[:, :128], got[:few.shape[0], :128])


def test_gemm_reference_test_shape(gpu, oracle):
    """10x20 . (30x20)^T with |delta ASum| <= 1e-4 (test/gpu_tensor_test.cpp:131-149)"""
    from graphnn_amd import ops
    rng = np.random.default_rng(5)
    A = rng.standard_normal((10, 20)).astype(np.float32); B = rng.standard_normal((30, 20)).astype(np.float32)
    got = _n(ops.gemm(_t(A, gpu), _t(B, gpu), False, True))
    want = oracle.gemm(A, B, False, True)
    assert abs(float(np.abs(got).sum()) - float(np.abs(want).sum())) <= 1e-4 * 30
    with pytest.raises(ValueError):
        ops.gemm(_t(A, gpu), _t(B, gpu), False, False)


@pytest.mark.parametrize("k", [5, 6, 7, 8, 53, 255, 260])
@pytest.mark.parametrize("n", [1, 4])
@pytest.mark.parametrize("side", ["A", "B"])
def test_gemm_of_few_columns_carries_infinities(gpu, n, k, side):
    """an infinity in any of the last columns of A, or rows of B, reaches the sums it is a term of, with its sign, and no
    others: where k is no multiple of four a lane group's last lane reads columns of the lane before it a second time"""
    from graphnn_amd import ops
    rng = np.random.default_rng(7 * k + n)
    m = 4133
    for tb in (False, True):
        for at in range(max(0, k - 6), k):
            A = (0.5 + rng.random((m, k))).astype(np.float32)
            B = (0.5 + rng.random((k, n))).astype(np.float32)
            want = A.astype(np.float64) @ B
            if side == "A":
                A[17, at], want[17] = -np.inf, -np.inf
            else:
                B[at, n - 1], want[:, n - 1] = np.inf, np.inf
            got = _n(ops.gemm(_t(A, gpu), _t(np.ascontiguousarray(B.T) if tb else B, gpu), False, tb))
            finite = np.isfinite(want)
            assert np.array_equal(got[~finite], want[~finite]), (tb, at)
            assert np.allclose(got[finite], want[finite], rtol=1e-5, atol=0), (tb, at)     # k <= 260 positive terms: 2^-24 k


# ------------------------------------------------------------------ element-wise engine
EXACT_UNARY = [("set", 0, 3.5, 0.0), ("truncate", 1, -0.5, 0.75), ("scale", 2, -1.75, 0.0), ("add", 3, 0.125, 0.0),
               ("abs", 4, 0, 0), ("relu", 6, 0, 0), ("square", 12, 0, 0)]
CLOSE_UNARY = [("inv", 5), ("sigmoid", 7), ("tanh", 8), ("exp", 11)]
POS_UNARY = [("log", 9), ("invsqrt", 10), ("sqrt", 13)]


@pytest.mark.parametrize("n,offset", [(1, 0), (3, 0), (1024, 0), (100003, 0), (4099, 1), (4099, 3)])
def test_unary_engine(gpu, oracle, n, offset):
    """offset > 0 gives a pointer that is not 16-byte aligned (a row view), exercising the scalar path"""
    from graphnn_amd import ops
    rng = np.random.default_rng(n + offset)
    base = (rng.standard_normal(n + offset) * 2).astype(np.float32)
    base[offset::7] = -0.0
    x = base[offset:]
    for name, code, a0, a1 in EXACT_UNARY:
        buf = _t(base, gpu)
        ops.unary(name, buf[offset:], a0, a1)
        got = _n(buf)
        assert np.array_equal(got[offset:].view(np.uint32), oracle.unary(code, x, a0, a1).view(np.uint32)), name
        assert np.array_equal(got[:offset], base[:offset])
    for name, code in CLOSE_UNARY:
        buf = _t(base, gpu)
        ops.unary(name, buf[offset:])
        assert np.allclose(_n(buf)[offset:], oracle.unary(code, x), rtol=2e-6, atol=1e-7), name
    pos = np.abs(base) + np.float32(0.01)
    for name, code in POS_UNARY:
        buf = _t(pos, gpu)
        ops.unary(name, buf[offset:])
        assert np.allclose(_n(buf)[offset:], oracle.unary(code, pos[offset:]), rtol=2e-6, atol=1e-7), name


def test_relu_keeps_negative_zero_and_nan(gpu):
    from graphnn_amd import ops
    x = np.array([-1.0, -0.0, 0.0, 2.0, np.nan, -np.inf, np.inf, -1e-45], np.float32)
    got = _n(ops.relu(_t(x, gpu)))
    assert np.array_equal(got[[0, 2, 3, 5, 6, 7]], np.array([0, 0, 2, 0, np.inf, 0], np.float32))
    assert got[1] == 0 and np.signbit(got[1]) and np.isnan(got[4])


@pytest.mark.parametrize("n", [1, 5, 4096, 250001])
def test_axpy_add_cast(gpu, oracle, n):
    from graphnn_amd import ops
    rng = np.random.default_rng(n)
    x = rng.standard_normal(n).astype(np.float32); y = rng.standard_normal(n).astype(np.float32)
    assert np.array_equal(_n(ops.axpy(1.0, _t(x, gpu), _t(y, gpu))), oracle.axpy(1.0, x, y))      # one rounded add
    assert np.array_equal(_n(ops.add(_t(x, gpu), _t(y, gpu))), x + y)
    assert np.allclose(_n(ops.axpy(0.3, _t(x, gpu), _t(y, gpu))), oracle.axpy(0.3, x, y), rtol=1e-6, atol=1e-7)
    assert np.allclose(_n(ops.axpby(0.3, _t(x, gpu), -1.5, _t(y, gpu))), oracle.axpby(0.3, x, -1.5, y), rtol=1e-6, atol=1e-7)
    ints = rng.integers(-2**30, 2**30, n).astype(np.int32)
    assert np.array_equal(_n(ops.cast_i32_f32(_t(ints, gpu))), oracle.cast(ints))
    with pytest.raises(ValueError):
        ops.axpy(1.0, _t(x, gpu), _t(np.zeros(n + 1, np.float32), gpu))


@pytest.mark.parametrize("n,offset", [(1, 0), (15, 1), (16, 0), (1000, 3), (1 << 20, 5)])
def test_memset0(gpu, n, offset):
    import torch
    from graphnn_amd import ops
    buf = torch.full((n + offset + 7,), 7, dtype=torch.uint8, device=gpu)
    ops.memset0(buf[offset:offset + n])
    got = _n(buf)
    assert np.all(got[offset:offset + n] == 0) and np.all(got[:offset] == 7) and np.all(got[offset + n:] == 7)


def test_memset0_batch(gpu):
    """many buffers in one launch: ragged starts and lengths, an empty one, more buffers than one launch takes"""
    import torch
    from graphnn_amd import ops
    rng = np.random.default_rng(3)
    sizes = [0, 1, 15, 16, 17, 1000, 4097, 1 << 20] + [int(x) for x in rng.integers(1, 5000, 100)]
    offs = [int(x) for x in rng.integers(0, 16, len(sizes))]
    bufs = [torch.full((n + o + 9,), 7, dtype=torch.uint8, device=gpu) for n, o in zip(sizes, offs)]
    ops.memset0_batch([b[o:o + n] for b, n, o in zip(bufs, sizes, offs)])
    for b, n, o in zip(bufs, sizes, offs):
        got = _n(b)
        assert np.all(got[o:o + n] == 0) and np.all(got[:o] == 7) and np.all(got[o + n:] == 7), (n, o)


# ------------------------------------------------------------------ softmax family
@pytest.mark.parametrize("rows,cols", [(20, 200), (256, 2), (7, 1), (3, 64), (5, 65), (2, 5000), (3, 1023), (3, 1024), (3, 1025)])
def test_row_softmax(gpu, oracle, rows, cols):
    from graphnn_amd import ops
    rng = np.random.default_rng(rows * cols)
    x = (rng.standard_normal((rows, cols)) * 3).astype(np.float32)
    got = _n(ops.row_softmax(_t(x, gpu)))
    want = oracle.row_softmax(x)
    assert float(np.abs(got - want).sum()) <= 1e-4              # the reference's own bound (gpu_tensor_test.cpp:151-166)
    assert max_rel(got, want) < PARITY_TOL
    assert np.allclose(got.sum(axis=1), 1.0, atol=1e-5)


def test_jagged_softmax(gpu, oracle):
    from graphnn_amd import ops
    rng = np.random.default_rng(6)
    x = (1.0 + rng.random(10)).astype(np.float32)
    lens = np.array([2, 3, 5], np.int32)                        # gpu_tensor_test.cpp:182-209, bound 1e-5
    got = _n(ops.jagged_softmax(_t(x, gpu), _t(lens, gpu)))
    assert float(np.abs(got - oracle.jagged_softmax(x, lens)).sum()) <= 1e-5
    # ragged: empty segments, length-1 segments, one long segment, > 1024 segments (several scan chunks)
    lens2 = rng.integers(0, 40, 3000).astype(np.int32)
    lens2[[0, 17, 2999]] = 0
    lens2[5] = 1
    lens2[1234] = 20000
    total = int(lens2.sum())
    x2 = (rng.standard_normal(total) * 2).astype(np.float32)
    got2 = _n(ops.jagged_softmax(_t(x2, gpu), _t(lens2, gpu)))
    want2 = oracle.jagged_softmax(x2, lens2)
    assert max_rel(got2, want2) < PARITY_TOL
    sums = np.add.reduceat(got2.astype(np.float64), np.concatenate([[0], np.cumsum(lens2)[:-1]])[lens2 > 0])
    assert np.allclose(sums, 1.0, atol=1e-4)
    # segment counts on both sides of the limit up to which one launch does it all (each workgroup adds up the
    # lengths ahead of its segments) and beyond which a scan launch comes first; the last workgroup is not full
    for nseg in (8191, 8192, 8193, 20001):
        lens3 = rng.integers(0, 9, nseg).astype(np.int32)
        lens3[nseg // 2] = 3000
        x3 = (rng.standard_normal(int(lens3.sum())) * 2).astype(np.float32)
        got3 = _n(ops.jagged_softmax(_t(x3, gpu), _t(lens3, gpu)))
        assert max_rel(got3, oracle.jagged_softmax(x3, lens3)) < PARITY_TOL, nseg


@pytest.mark.parametrize("nseg", [1, 7, 1024, 1025])
def test_jagged_softmax_of_segments_of_any_length(gpu, nseg):
    """a workgroup per segment (up to 1,024 segments) and a wavefront per segment: lengths around what a lane holds, empty segments,
    the lowest value everywhere, infinities and NaN (only one that comes first survives the scan for the maximum); against
    float64, each probability within the 2^-24 roundings of the exponent's argument, exponential, sum and division"""
    from graphnn_amd import ops
    rng = np.random.default_rng(nseg)
    edge = [0, 1, 63, 64, 65, 255, 256, 257, 1023, 1024, 1025, 4095, 4096, 4097, 8193, 20_000]
    lens = np.array([edge[i % len(edge)] if i < 2 * len(edge) else i % 5 for i in range(nseg)], np.int32)
    if nseg == 1:
        lens[0] = 70_001
    x = (rng.standard_normal(int(lens.sum())) * 4).astype(np.float32)
    off = np.concatenate([[0], np.cumsum(lens)])
    special = {}
    if nseg > 1:
        for i, kind in ((5, "lowest"), (4, "inf"), (6, "nan later"), (3, "nan first")):
            seg = x[off[i]:off[i + 1]]
            special[i] = kind
            if kind == "lowest": seg[:] = np.finfo(np.float32).min
            elif kind == "inf": seg[7] = np.inf
            elif kind == "nan later": seg[9] = np.nan
            else: seg[0] = np.nan
    got = _n(ops.jagged_softmax(_t(x, gpu), _t(lens, gpu)))
    for i in range(nseg):
        seg, out = x[off[i]:off[i + 1]], got[off[i]:off[i + 1]]
        if seg.size == 0: continue
        kind = special.get(i)
        if kind == "lowest":
            assert np.allclose(out, 1.0 / seg.size, rtol=4 * 2.0 ** -24, atol=0), i
        elif kind is not None:
            # inf - inf and NaN make the sum, and with it every quotient but 0 / NaN, NaN
            assert np.isnan(out).all(), (i, kind)
        else:
            e = np.exp(seg.astype(np.float64) - float(seg.max()))
            # argument up to 2^5 in magnitude (half an ulp of it, 2^-20), exponential 2 ulp, the sum as a tree over lanes of runs of
            # len / 64 terms of one sign at most, division
            bound = 2.0 ** -20 + (2 + max(1, seg.size / 64) + 16 + 1) * 2.0 ** -24
            assert np.all(np.abs(out - e / e.sum()) <= bound * (e / e.sum()) + 2.0 ** -126), (i, seg.size)


def test_jagged_softmax_gradient(gpu, oracle):
    """dst += (grad - <grad, out>) * out per segment (src/nn/jagged_softmax.cpp:8-31), ragged segments"""
    from graphnn_amd import ops
    rng = np.random.default_rng(61)
    lens = rng.integers(0, 50, 2500).astype(np.int32)
    lens[[0, 9]] = 0; lens[4] = 1; lens[700] = 9000
    n = int(lens.sum())
    p = oracle.jagged_softmax((rng.standard_normal(n) * 2).astype(np.float32), lens)
    g = rng.standard_normal(n).astype(np.float32)
    d0 = rng.standard_normal(n).astype(np.float32)
    want = oracle.jagged_softmax_deriv(d0, p, g, lens)
    got = _n(ops.jagged_softmax_deriv(_t(d0, gpu), _t(p, gpu), _t(g, gpu), _t(lens, gpu)))
    off = np.concatenate([[0], np.cumsum(lens)])
    seg = np.repeat(np.arange(lens.size), lens)
    z = np.bincount(seg, weights=g.astype(np.float64) * p, minlength=lens.size)
    want64 = d0 + (g - z[seg]) * p.astype(np.float64)
    assert_parity("jagged softmax gradient", got, want, want64)


@pytest.mark.parametrize("rows,cols", [(100, 10), (1, 1), (37, 300), (5000, 2), (3, 1025)])
def test_row_softmax_gradient(gpu, oracle, rows, cols):
    """dst += (grad - <grad, out>) * out per row (SoftmaxDeriv, src/nn/softmax.cpp:8-29): the segment rule of the
    jagged softmax with equal segments, which is how the oracle states it; float64 settles a miss; and the
    textbook property that a constant gradient passes nothing on (the probabilities of a row add up to 1)"""
    from graphnn_amd import ops
    rng = np.random.default_rng(rows + cols)
    p = oracle.row_softmax((rng.standard_normal((rows, cols)) * 2).astype(np.float32))
    g = rng.standard_normal((rows, cols)).astype(np.float32)
    d0 = rng.standard_normal((rows, cols)).astype(np.float32)
    lens = np.full(rows, cols, np.int32)
    want = oracle.jagged_softmax_deriv(d0.reshape(-1), p.reshape(-1), g.reshape(-1), lens).reshape(rows, cols)
    got = _n(ops.row_softmax_deriv(_t(d0, gpu), _t(p, gpu), _t(g, gpu)))
    z = (g.astype(np.float64) * p).sum(axis=1, keepdims=True)
    assert_parity("row softmax gradient", got, want, d0 + (g - z) * p.astype(np.float64))
    flat = _n(ops.row_softmax_deriv(_t(np.zeros_like(d0), gpu), _t(p, gpu), _t(np.full_like(g, 3.5), gpu)))
    assert np.abs(flat).max() < 1e-5


# ------------------------------------------------------------------ reductions and index ops
@pytest.mark.parametrize("n", [1, 63, 256, 4000, 16385, 3_000_001])
def test_reduce(gpu, oracle, n):
    from graphnn_amd import ops
    rng = np.random.default_rng(n)
    x = (1.0 + rng.random(n)).astype(np.float32)                # U(1,2): the reference's Mean test distribution
    xd = _t(x, gpu)
    ref64 = x.astype(np.float64)
    assert abs(float(_n(ops.reduce("sum", xd))[0]) - ref64.sum()) <= 1e-5 * ref64.sum()
    assert abs(float(_n(ops.reduce("mean", xd))[0]) - ref64.mean()) <= 1e-5     # gpu_tensor_test.cpp:168-180
    assert float(_n(ops.reduce("max", xd))[0]) == oracle.max(x)
    ints = rng.integers(-50, 50, min(n, 100000)).astype(np.float32)
    assert float(_n(ops.reduce("sum", _t(ints, gpu)))[0]) == float(ints.astype(np.float64).sum())   # exact in fp32
    # views that start 4, 8 and 12 bytes past a 16-byte boundary (the kernel reads 128-bit words from the first aligned one)
    for off in (1, 2, 3):
        if n > off:
            v = xd[off:]
            assert v.data_ptr() % 16 == 4 * off
            assert abs(float(_n(ops.reduce("sum", v))[0]) - ref64[off:].sum()) <= 1e-5 * ref64[off:].sum()
            assert float(_n(ops.reduce("max", v))[0]) == oracle.max(x[off:])
            assert float(_n(ops.reduce("sum", _t(ints, gpu)[min(off, ints.size - 1):]))[0]) == float(ints[min(off, ints.size - 1):].astype(np.float64).sum())
    sq = float(_n(ops.reduce("sumsq", xd))[0])
    assert abs(sq - (ref64 ** 2).sum()) <= 1e-5 * (ref64 ** 2).sum()
    # max keeps the reference's rule for NaN: one in the first place is the result, one anywhere else is never selected
    if n > 1:
        y = x.copy(); y[n // 2] = np.nan
        assert float(_n(ops.reduce("max", _t(y, gpu)))[0]) == oracle.max(y) == np.nanmax(y)
    y = x.copy(); y[0] = np.nan
    assert np.isnan(float(_n(ops.reduce("max", _t(y, gpu)))[0])) and np.isnan(oracle.max(y))


def test_row_argmax(gpu, oracle):
    from graphnn_amd import ops
    rng = np.random.default_rng(7)
    big = rng.standard_normal((10, 1023)).astype(np.float32)     # gpu_tensor_test.cpp:111-129
    assert np.array_equal(_n(ops.row_argmax(_t(big, gpu))), oracle.row_argmax(big))
    ties = np.array([[1, 3, 3, 2], [5, 5, 5, 5], [-1, -2, -0.5, -0.5], [0.0, -0.0, 0.0, 0.0]], np.float32)
    assert list(_n(ops.row_argmax(_t(ties, gpu)))) == [1, 0, 2, 0]
    withnan = np.array([[np.nan, 9, 1], [1, np.nan, 3], [2, 5, np.nan], [-np.inf, np.nan, -np.inf]], np.float32)
    assert np.array_equal(_n(ops.row_argmax(_t(withnan, gpu))), oracle.row_argmax(withnan))
    # many rows with heavy ties: small integer values
    tied = rng.integers(0, 3, (5000, 130)).astype(np.float32)
    assert np.array_equal(_n(ops.row_argmax(_t(tied, gpu))), oracle.row_argmax(tied))
    two = rng.standard_normal((256, 2)).astype(np.float32)
    assert np.array_equal(_n(ops.row_argmax(_t(two, gpu))), oracle.row_argmax(two))


def test_label_ops(gpu, oracle):
    from graphnn_amd import ops
    rng = np.random.default_rng(8)
    B, Q = 1000, 6
    # general CSR label rows: 0..3 entries per row
    lens = rng.integers(0, 4, B)
    rp = np.zeros(B + 1, np.int32); np.cumsum(lens, out=rp[1:])
    nnz = int(rp[-1])
    ci = rng.integers(0, Q, nnz).astype(np.int32)
    v = rng.integers(0, 3, nnz).astype(np.float32)              # ties between stored values
    assert np.array_equal(_n(ops.csr_row_argmax(_t(rp, gpu), _t(ci, gpu), _t(v, gpu))), oracle.csr_row_argmax(rp, ci, v))
    prob = oracle.row_softmax(rng.standard_normal((B, Q)).astype(np.float32) * 4)
    prob[3, :] = 0.0                                             # exercises the 1e-8 clamp
    got = _n(ops.cross_entropy(_t(prob, gpu), _t(rp, gpu), _t(ci, gpu), _t(v, gpu)))[:, 0]
    assert np.allclose(got, oracle.cross_entropy(prob, rp, ci, v), rtol=1e-6, atol=1e-7)
    label = rng.integers(0, Q, B).astype(np.int32)
    pred = rng.integers(0, 4, (B, Q)).astype(np.float32)         # ties
    for k in (1, 2, 3):
        assert np.array_equal(_n(ops.in_top_k(_t(pred, gpu), _t(label, gpu), k)), oracle.in_top_k(pred, label, k))
    wide = rng.standard_normal((50, 300)).astype(np.float32)
    wl = rng.integers(0, 300, 50).astype(np.int32)
    assert np.array_equal(_n(ops.in_top_k(_t(wide, gpu), _t(wl, gpu), 5)), oracle.in_top_k(wide, wl, 5))


# ------------------------------------------------------------------ fused stages
def _small_problem(seed, B, K, C, H, Q, lo=3, hi=40):
    batch = synth.molecule_batch(seed, B, K, Q, size_mode="uniform", size_lo=lo, size_hi=hi)
    w = synth.make_weights(synth.Stream(seed), K, C, H, Q)
    a = batching.node2node_csr(batch.num_nodes, batch.edge_x, batch.edge_y)
    s = batching.subgraph_csr(batch.num_graphs, batch.subg_id, batch.node_idx)
    return batch, w, a, s


@pytest.mark.parametrize("C", [16, 32, 64, 48, 128, 256])
@pytest.mark.parametrize("K", [7, 17, 38, 64, 70])
def test_input_stage(gpu, oracle, C, K):
    from graphnn_amd import ops
    batch, w, a, s = _small_problem(10 + C + K, 9, K, C, 8, 2)
    X = batch.one_hot()
    X += (np.random.default_rng(C).standard_normal(X.shape) * 0.01).astype(np.float32)    # dense, not just one-hot
    msg, h0 = ops.s2v_input(_t(X, gpu), _t(w.W_n2l, gpu))
    want = oracle.gemm(X, w.W_n2l)
    assert max_rel(_n(msg), want) < PARITY_TOL
    assert np.array_equal(_n(h0), np.maximum(_n(msg), 0))       # ReLU of what was stored, exactly


@pytest.mark.parametrize("C", [16, 32, 64, 128])
@pytest.mark.parametrize("K", [5, 38])
def test_input_stage_many_rows(gpu, oracle, C, K):
    """40,003 rows: past 32,768 rows the narrow hidden sizes take four row tiles per workgroup, and every
    kernel gives a workgroup more than one tile; msg and h0 both stored, real-valued X"""
    from graphnn_amd import ops
    rng = np.random.default_rng(7 * C + K)
    N = 40_003
    X = rng.standard_normal((N, K)).astype(np.float32)
    Wn = (rng.standard_normal((K, C)) * 0.3).astype(np.float32)
    msg, h0 = ops.s2v_input(_t(X, gpu), _t(Wn, gpu))
    assert max_rel(_n(msg), oracle.gemm(X, Wn)) < PARITY_TOL
    assert np.array_equal(_n(h0), np.maximum(_n(msg), 0))


@pytest.mark.parametrize("C", [16, 32, 64, 48, 128, 256])
@pytest.mark.parametrize("with_msg,with_bias", [(True, False), (True, True), (False, False)])
def test_level_stage(gpu, oracle, C, with_msg, with_bias):
    from graphnn_amd import ops
    batch, w, a, s = _small_problem(20 + C, 40, 5, C, 8, 2)
    rng = np.random.default_rng(C)
    N = batch.num_nodes
    h_in = np.maximum(rng.standard_normal((N, C)), 0).astype(np.float32)
    msg = rng.standard_normal((N, C)).astype(np.float32) if with_msg else None
    bias = rng.standard_normal(C).astype(np.float32) if with_bias else None
    want, w64 = _level_want(oracle, *a, h_in, w.W_conv, msg, bias)
    got = _n(ops.s2v_level(*_csr_t(a, gpu), _t(h_in, gpu), _t(w.W_conv, gpu),
                           _t(msg, gpu) if with_msg else None, _t(bias, gpu) if with_bias else None))
    assert_parity("level", got, want, w64)
    assert np.all(got >= 0)


@pytest.mark.parametrize("C", [16, 32, 64, 128, 256])
def test_level_stage_row_counts_around_every_threshold(gpu, oracle, C):
    """row counts on both sides of the tile sizes (16, 64), of the sizes at which the kernels change their
    rows per pass or start asking for gathers a tile early (16,384, 32,768, 65,536) and of one, two and more
    tiles per wavefront; ragged rows of 0..5 entries, weights, msg and bias"""
    from graphnn_amd import ops
    for N in (1, 15, 16, 17, 63, 64, 65, 1023, 1025, 4097, 12289, 16383, 16385, 32767, 32769, 49153, 65535, 65537):
        rng = np.random.default_rng(1000 * C + N)
        lens = rng.integers(0, 6, N)
        rp = np.zeros(N + 1, np.int32); np.cumsum(lens, out=rp[1:])
        nnz = int(rp[-1])
        ci = rng.integers(0, N, nnz).astype(np.int32)
        v = (rng.random(nnz) * 0.5).astype(np.float32)
        h_in = np.maximum(rng.standard_normal((N, C)), 0).astype(np.float32)
        W = (rng.standard_normal((C, C)) * 0.1).astype(np.float32)
        msg = rng.standard_normal((N, C)).astype(np.float32)
        bias = rng.standard_normal(C).astype(np.float32)
        want, w64 = _level_want(oracle, rp, ci, v, h_in, W, msg, bias)
        if nnz:
            ci_d, v_d = _t(ci, gpu), _t(v, gpu)
        else:
            import torch
            ci_d = torch.zeros(1, dtype=torch.int32, device=gpu)[:0]; v_d = torch.zeros(1, dtype=torch.float32, device=gpu)[:0]
        got = _n(ops.s2v_level(_t(rp, gpu), ci_d, v_d, _t(h_in, gpu), _t(W, gpu), _t(msg, gpu), _t(bias, gpu)))
        assert_parity("level", got, want, w64)


def test_level_stage_hub_rows_and_weights(gpu, oracle):
    """one vertex with thousands of in-neighbours (whole-workgroup gather) and non-unit edge weights"""
    from graphnn_amd import ops
    rng = np.random.default_rng(9)
    N, C = 5000, 64
    lens = rng.integers(0, 6, N); lens[17] = 4000; lens[4999] = 1500; lens[2048] = 1025
    rp = np.zeros(N + 1, np.int32); np.cumsum(lens, out=rp[1:])
    nnz = int(rp[-1])
    ci = rng.integers(0, N, nnz).astype(np.int32)
    v = (rng.random(nnz) * 0.1).astype(np.float32)
    h_in = np.maximum(rng.standard_normal((N, C)), 0).astype(np.float32)
    W = (rng.standard_normal((C, C)) * 0.1).astype(np.float32)
    msg = rng.standard_normal((N, C)).astype(np.float32)
    want, w64 = _level_want(oracle, rp, ci, v, h_in, W, msg, None)
    got = _n(ops.s2v_level(_t(rp, gpu), _t(ci, gpu), _t(v, gpu), _t(h_in, gpu), _t(W, gpu), _t(msg, gpu)))
    assert_parity("level", got, want, w64)


@pytest.mark.parametrize("C", [16, 32, 64])
@pytest.mark.parametrize("N", [20_011, 160_007])
def test_level_every_row_length_up_to_70(gpu, oracle, C, N):
    """row lengths 0..70 in turn: the boundaries of the streaming level kernel (4 entries fetched at once, 8
    with the second go, 16 per batch at hidden 64, 48 for one lane group, 64 for the balanced pass, which only
    the larger matrix gets); the larger matrix also gives every wavefront several tiles, so the look-ahead of
    row pointers and first batches runs in its steady state; N is not a multiple of the tile"""
    from graphnn_amd import ops
    rng = np.random.default_rng(C + N)
    lens = (np.arange(N) * 7) % 71
    rp = np.zeros(N + 1, np.int32); np.cumsum(lens, out=rp[1:])
    nnz = int(rp[-1])
    ci = rng.integers(0, N, nnz).astype(np.int32)
    v = (rng.random(nnz) * 0.2).astype(np.float32)
    h_in = np.maximum(rng.standard_normal((N, C)), 0).astype(np.float32)
    W = (rng.standard_normal((C, C)) * 0.1).astype(np.float32)
    msg = rng.standard_normal((N, C)).astype(np.float32)
    bias = rng.standard_normal(C).astype(np.float32)
    want, w64 = _level_want(oracle, rp, ci, v, h_in, W, msg, bias)
    got = _n(ops.s2v_level(_t(rp, gpu), _t(ci, gpu), _t(v, gpu), _t(h_in, gpu), _t(W, gpu), _t(msg, gpu), _t(bias, gpu)))
    assert_parity("level", got, want, w64)


@pytest.mark.parametrize("C", [128, 256])
def test_wide_level_on_a_large_dense_skewed_graph(gpu, oracle, C):
    """hidden 128 / 256 on a graph of 40,000 rows with 14 entries per row on average and two rows of 5,000 and
    3,000 entries: the level leaves the one-launch wide kernel (one wavefront per row, whatever its length) for
    SpMM with the balanced pass, then the wide kernel's contraction and epilogue over the summed rows (read
    through the identity matrix).  The result carries the bits of those two steps made by hand, which is how
    the route shows; the forward entry must not hand it ReLU-through-msg"""
    from graphnn_amd import ops
    rng = np.random.default_rng(77)
    N = 40_000
    lens = rng.integers(10, 17, N); lens[123] = 5_000; lens[39_999] = 3_000
    rp = np.zeros(N + 1, np.int32); np.cumsum(lens, out=rp[1:])
    nnz = int(rp[-1])
    assert nnz >= 12 * N
    ci = rng.integers(0, N, nnz).astype(np.int32)
    v = (rng.random(nnz) * 0.05).astype(np.float32)
    h_in = np.maximum(rng.standard_normal((N, C)), 0).astype(np.float32)
    W = (rng.standard_normal((C, C)) * 0.1).astype(np.float32)
    msg = rng.standard_normal((N, C)).astype(np.float32)
    want, w64 = _level_want(oracle, rp, ci, v, h_in, W, msg, None)
    got = _n(ops.s2v_level(_t(rp, gpu), _t(ci, gpu), _t(v, gpu), _t(h_in, gpu), _t(W, gpu), _t(msg, gpu)))
    assert_parity("level", got, want, w64)
    import torch
    agg = ops.spmm(_t(rp, gpu), _t(ci, gpu), _t(v, gpu), _t(h_in, gpu), N)
    eye = (torch.arange(N + 1, dtype=torch.int32, device=gpu), torch.arange(N, dtype=torch.int32, device=gpu),
           torch.ones(N, dtype=torch.float32, device=gpu))
    by_hand = _n(ops.s2v_level(*eye, agg, _t(W, gpu), _t(msg, gpu)))
    assert np.array_equal(got, by_hand)
    # with a bias row, and the same bits on a second run
    bias = rng.standard_normal(C).astype(np.float32)
    want_b, w64_b = _level_want(oracle, rp, ci, v, h_in, W, msg, bias)
    got_b = _n(ops.s2v_level(_t(rp, gpu), _t(ci, gpu), _t(v, gpu), _t(h_in, gpu), _t(W, gpu), _t(msg, gpu), bias=_t(bias, gpu)))
    assert_parity("level", got_b, want_b, w64_b)
    assert np.array_equal(got_b, _n(ops.s2v_level(_t(rp, gpu), _t(ci, gpu), _t(v, gpu), _t(h_in, gpu), _t(W, gpu), _t(msg, gpu),
                                                 bias=_t(bias, gpu))))


@pytest.mark.parametrize("C", [128, 256])
@pytest.mark.parametrize("nnz", [0, 1, 5, 6, 7])
def test_wide_level_fewer_entries_than_one_index_batch(gpu, oracle, C, nnz):
    """the wide kernel reads column indices and weights six at a time: matrices with fewer entries than that,
    exactly that many, and one more; the entries sit in the last rows, so the last batch ends at the end of
    the arrays"""
    import torch
    from graphnn_amd import ops
    rng = np.random.default_rng(300 + C + nnz)
    N = 77
    lens = np.zeros(N, np.int64)
    for i in range(nnz): lens[N - 1 - (i % 3)] += 1
    rp = np.zeros(N + 1, np.int32); np.cumsum(lens, out=rp[1:])
    ci = rng.integers(0, N, nnz).astype(np.int32)
    v = (rng.random(nnz) + 0.5).astype(np.float32)
    h_in = np.maximum(rng.standard_normal((N, C)), 0).astype(np.float32)
    W = (rng.standard_normal((C, C)) * 0.1).astype(np.float32)
    msg = rng.standard_normal((N, C)).astype(np.float32)
    want, w64 = _level_want(oracle, rp, ci, v, h_in, W, msg, None)
    ci_d = _t(ci, gpu) if nnz else torch.zeros(1, dtype=torch.int32, device=gpu)[:0]
    v_d = _t(v, gpu) if nnz else torch.zeros(1, dtype=torch.float32, device=gpu)[:0]
    got = _n(ops.s2v_level(_t(rp, gpu), ci_d, v_d, _t(h_in, gpu), _t(W, gpu), _t(msg, gpu)))
    assert_parity("level", got, want, w64)


@pytest.mark.parametrize("C", [64, 128, 256])
@pytest.mark.parametrize("hint", [0, 5, 6, 1000])
def test_level_entry_count_hint_does_not_bound_the_reads(gpu, oracle, C, hint):
    """the nnz argument only sizes scratch: a 77-row matrix with 10 entries gives the same bits whether the
    host states 0, 5, 6 or 1,000 entries (the kernels bound their index reads with row_ptr[N] on the device;
    the hidden-128/256 kernel reads indices six at a time and once took the host's count for it)"""
    from graphnn_amd import ops
    rng = np.random.default_rng(900 + C)
    N, nnz = 77, 10
    lens = np.zeros(N, np.int64)
    for i in range(nnz): lens[[3, 40, 76][i % 3]] += 1
    rp = np.zeros(N + 1, np.int32); np.cumsum(lens, out=rp[1:])
    ci = rng.integers(0, N, nnz).astype(np.int32)
    v = (rng.random(nnz) + 0.5).astype(np.float32)
    h_in = np.maximum(rng.standard_normal((N, C)), 0).astype(np.float32)
    W = (rng.standard_normal((C, C)) * 0.1).astype(np.float32)
    msg = rng.standard_normal((N, C)).astype(np.float32)
    want, w64 = _level_want(oracle, rp, ci, v, h_in, W, msg, None)
    args = (_t(rp, gpu), _t(ci, gpu), _t(v, gpu), _t(h_in, gpu), _t(W, gpu), _t(msg, gpu))
    exact = _n(ops.s2v_level(*args))
    got = _n(ops.s2v_level(*args, nnz_hint=hint))
    assert np.array_equal(got, exact)
    assert_parity("level", got, want, w64)


@pytest.mark.parametrize("C", [128, 256])
@pytest.mark.parametrize("N", [5_003, 10_007, 15_991, 64 * 300 + 37, 40_037, 70_001])
def test_wide_level_ragged_rows_and_weights(gpu, oracle, C, N):
    """wide-hidden kernel: empty rows, rows longer than one 64-entry index batch, a row count that is
    not a multiple of the pass, non-unit weights; the sizes take passes of 16, 32 and 64 rows, with two to
    four passes per workgroup (three and more exercise the look-ahead across passes)"""
    from graphnn_amd import ops
    rng = np.random.default_rng(90 + C + N)
    lens = rng.integers(0, 7, N); lens[5] = 700; lens[6] = 0; lens[7] = 0; lens[N - 1] = 130; lens[64:72] = 0
    rp = np.zeros(N + 1, np.int32); np.cumsum(lens, out=rp[1:])
    nnz = int(rp[-1])
    ci = rng.integers(0, N, nnz).astype(np.int32)
    v = (rng.random(nnz) * 0.5).astype(np.float32)
    h_in = np.maximum(rng.standard_normal((N, C)), 0).astype(np.float32)
    W = (rng.standard_normal((C, C)) * 0.1).astype(np.float32)
    msg = rng.standard_normal((N, C)).astype(np.float32)
    want, w64 = _level_want(oracle, rp, ci, v, h_in, W, msg, None)
    got = _n(ops.s2v_level(_t(rp, gpu), _t(ci, gpu), _t(v, gpu), _t(h_in, gpu), _t(W, gpu), _t(msg, gpu)))
    assert_parity("level", got, want, w64)


@pytest.mark.parametrize("C,H,Q", [(64, 32, 2), (16, 8, 3), (32, 100, 70), (48, 16, 2), (128, 64, 5)])
def test_readout_stage(gpu, oracle, C, H, Q):
    from graphnn_amd import ops
    batch, w, a, s = _small_problem(30 + C, 33, 5, C, H, Q, lo=1, hi=300)
    rng = np.random.default_rng(C + H)
    h = np.maximum(rng.standard_normal((batch.num_nodes, C)), 0).astype(np.float32)
    pool, hidden, logits, probs, pred = (_n(t) for t in ops.s2v_readout(*_csr_t(s, gpu), _t(h, gpu), _t(w.W_h1, gpu),
                                                                        _t(w.W_h2, gpu), batch.num_graphs))
    w_pool = oracle.spmm(*s, h, batch.num_graphs)
    w_hidden = np.maximum(oracle.gemm(w_pool, w.W_h1), 0)
    w_logits = oracle.gemm(w_hidden, w.W_h2)
    assert max_rel(pool, w_pool) < PARITY_TOL
    assert max_rel(hidden, w_hidden) < PARITY_TOL
    assert max_rel(logits, w_logits) < PARITY_TOL
    assert max_rel(probs, oracle.row_softmax(w_logits)) < PARITY_TOL
    assert np.array_equal(pred, oracle.row_argmax(logits))      # arg-max of the logits the device produced: exact


@pytest.mark.parametrize("C,H,Q,B", [(64, 32, 2, 1500), (16, 8, 3, 1100), (32, 100, 70, 1030), (128, 64, 5, 300), (256, 128, 2, 260)])
def test_readout_stage_many_graphs(gpu, oracle, C, H, Q, B):
    """batches of many graphs take the kernel with one wavefront per graph (hidden up to 64; wider ones the
    SpMM and the GEMMs).  Graphs of 1 to 60 nodes; the subgraph matrix also gets one empty row and weights
    other than 1"""
    from graphnn_amd import ops
    batch, w, a, s = _small_problem(70 + C, B, 5, C, H, Q, lo=1, hi=60)
    rp, ci, v = (np.array(x) for x in s)
    # graph 3 loses its nodes (an empty row of S), and the weights differ from 1
    lo, hi = int(rp[3]), int(rp[4])
    keep = np.ones(rp[-1], dtype=bool); keep[lo:hi] = False
    ci, v = ci[keep], v[keep]
    rp = rp.copy(); rp[4:] -= (hi - lo)
    rng = np.random.default_rng(C + H + B)
    v = (0.5 + rng.random(v.size)).astype(np.float32)
    s = (rp.astype(np.int32), ci.astype(np.int32), v)
    h = np.maximum(rng.standard_normal((batch.num_nodes, C)), 0).astype(np.float32)
    pool, hidden, logits, probs, pred = (_n(t) for t in ops.s2v_readout(*_csr_t(s, gpu), _t(h, gpu), _t(w.W_h1, gpu),
                                                                        _t(w.W_h2, gpu), batch.num_graphs))
    w_pool = oracle.spmm(*s, h, batch.num_graphs)
    w_hidden = np.maximum(oracle.gemm(w_pool, w.W_h1), 0)
    w_logits = oracle.gemm(w_hidden, w.W_h2)
    assert np.all(pool[3] == 0) and np.all(logits[3] == 0)
    assert max_rel(pool, w_pool) < PARITY_TOL
    assert max_rel(hidden, w_hidden) < PARITY_TOL
    assert max_rel(logits, w_logits) < PARITY_TOL
    assert max_rel(probs, oracle.row_softmax(w_logits)) < PARITY_TOL
    assert np.array_equal(pred, oracle.row_argmax(logits))      # arg-max of the logits the device produced: exact


@pytest.mark.parametrize("C,H,Q,B,hi", [(4, 8, 2, 5, 40), (7, 130, 70, 41, 90), (100, 50, 6, 2051, 9), (255, 20, 3, 2049, 5), (33, 64, 2, 7, 1500), (129, 32, 2, 3, 900)])
def test_readout_of_any_hidden_size(gpu, oracle, C, H, Q, B, hi):
    """a wavefront per graph (from 2,048 small ones on, the last tile of four not full), a workgroup of 256 lanes, one of 512
    for graphs of hundreds of rows; an empty graph, one node, weights other than 1; then the scores of the rows as a product
    with one column, from 4,096 rows on a kernel of its own at any width"""
    from graphnn_amd import ops
    rng = np.random.default_rng(C + B)
    lens = rng.integers(hi // 2, hi + 1, B); lens[1] = 0; lens[2] = 1
    rp = np.zeros(B + 1, np.int32); np.cumsum(lens, out=rp[1:])
    N = int(rp[-1])
    S = (rp, np.arange(N, dtype=np.int32), (0.5 + rng.random(N)).astype(np.float32))
    h = np.maximum(rng.standard_normal((N, C)), 0).astype(np.float32)
    W1 = (rng.standard_normal((C, H)) * 0.2).astype(np.float32); W2 = (rng.standard_normal((H, Q)) * 0.2).astype(np.float32)
    pool, hidden, logits, probs, pred = (_n(t) for t in ops.s2v_readout(*_csr_t(S, gpu), _t(h, gpu), _t(W1, gpu), _t(W2, gpu), B))
    w_pool = oracle.spmm(*S, h, B)
    w_hidden = np.maximum(oracle.gemm(w_pool, W1), 0)
    w_logits = oracle.gemm(w_hidden, W2)
    for got, want in ((pool, w_pool), (hidden, w_hidden), (logits, w_logits), (probs, oracle.row_softmax(w_logits))):
        assert max_rel(got, want) < PARITY_TOL
    assert np.all(pool[1] == 0) and np.array_equal(pred, oracle.row_argmax(logits))
    w = rng.standard_normal((C, 1)).astype(np.float32)
    assert_parity("score", _n(ops.gemm(_t(h, gpu), _t(w, gpu))), *_gemm_want(oracle, h, w))


# ------------------------------------------------------------------ whole forward, configurations 1 and 2
def _forward_case(gpu, oracle, config_id, B=None):
    from graphnn_amd import ops
    batch, w, cfg = synth.make_config(config_id, B=B)
    a = batching.node2node_csr(batch.num_nodes, batch.edge_x, batch.edge_y)
    s = batching.subgraph_csr(batch.num_graphs, batch.subg_id, batch.node_idx)
    X = batch.one_hot()
    lab = batch.label_csr()
    want = _forward_want(oracle, a, s, X, w, cfg["L"], lab)
    bufs = ops.s2v_forward(_csr_t(a, gpu), _csr_t(s, gpu), _t(X, gpu), _t(w.W_n2l, gpu), _t(w.W_conv, gpu),
                           _t(w.W_h1, gpu), _t(w.W_h2, gpu), cfg["L"])
    got = dict(msg=_n(bufs.msg), h_final=_n(bufs.h_final), pool=_n(bufs.pool), hidden=_n(bufs.hidden),
               logits=_n(bufs.logits), probs=_n(bufs.probs), pred=_n(bufs.pred))
    return batch, cfg, a, s, X, w, lab, want, got, bufs


@pytest.mark.parametrize("config_id", [1, 2])
def test_forward_matches_reference_path(gpu, oracle, config_id):
    from graphnn_amd import ops
    batch, cfg, a, s, X, w, lab, want, got, bufs = _forward_case(gpu, oracle, config_id)
    _assert_forward_parity(got, want, cfg["L"])
    assert_stages("", a, s, X, w, {k: got[k] for k in ("msg", "h_final", "pool", "hidden", "logits", "probs")})
    # argmax predictions bit-exact with the reference path
    assert np.array_equal(got["pred"], want["pred"])
    # loss / accuracy tail of the graph, operator by operator on the device
    lab_d = _csr_t(lab, gpu)
    loss_rows = ops.cross_entropy(bufs.probs, *lab_d)
    truth = ops.csr_row_argmax(*lab_d)
    hit = ops.in_top_k(bufs.logits, truth, 1)
    loss = float(_n(ops.reduce("mean", loss_rows))[0])
    acc = float(_n(ops.reduce("mean", ops.cast_i32_f32(hit)))[0])
    assert np.array_equal(_n(truth), want["truth"])
    assert np.array_equal(_n(hit), want["hit"])
    assert np.allclose(_n(loss_rows)[:, 0], want["loss_rows"], rtol=1e-4)
    assert abs(loss - want["scalars"][0]) <= 1e-4 * abs(want["scalars"][0])
    assert abs(acc - want["scalars"][1]) <= 1e-6


@pytest.mark.parametrize("C,H,Q", [(64, 32, 2), (32, 8, 3), (128, 16, 2), (256, 8, 2)])
def test_forward_graph_counts_around_the_readout_thresholds(gpu, oracle, C, H, Q):
    """whole forward (general route) on batches of 1 .. 4,100 small graphs: the readout changes kernel at 1,024
    graphs (one wavefront per graph, hidden <= 64) and at 4,096 graphs (hidden 128/256: workgroup per graph, then
    SpMM + GEMM)"""
    from graphnn_amd import ops
    K, L = 6, 2
    for B in (1, 2, 255, 1023, 1024, 1025, 4096, 4100):
        seed = 31 * C + B
        batch = synth.molecule_batch(seed, B, K, Q, size_mode="uniform", size_lo=1, size_hi=7)
        w = synth.make_weights(synth.Stream(seed), K, C, H, Q)
        a = batching.node2node_csr(batch.num_nodes, batch.edge_x, batch.edge_y)
        s = batching.subgraph_csr(batch.num_graphs, batch.subg_id, batch.node_idx)
        X = batch.one_hot()
        want = _forward_want(oracle, a, s, X, w, L)
        bufs = ops.s2v_forward(_csr_t(a, gpu), _csr_t(s, gpu), _t(X, gpu), _t(w.W_n2l, gpu), _t(w.W_conv, gpu),
                               _t(w.W_h1, gpu), _t(w.W_h2, gpu), L)
        _assert_forward_parity({k: _n(getattr(bufs, k)) for k in ("pool", "hidden", "logits", "probs")}, want, L,
                               tag=" B=%d" % B, keys=("pool", "hidden", "logits", "probs"))
        assert np.array_equal(_n(bufs.pred), want["pred"]), B


def test_forward_on_two_streams_interleaved(gpu, oracle):
    """two forwards queued alternately on two streams (scratch buffers and the plan of the long-row pass are
    kept per stream): each gives what it gives alone"""
    import torch
    from graphnn_amd import ops
    cases = []
    for seed, B, C in ((1, 300, 64), (2, 40, 128)):
        batch = synth.molecule_batch(seed, B, 9, 2, size_mode="uniform", size_lo=5, size_hi=200)
        w = synth.make_weights(synth.Stream(seed), 9, C, 16, 2)
        a = batching.node2node_csr(batch.num_nodes, batch.edge_x, batch.edge_y)
        s = batching.subgraph_csr(batch.num_graphs, batch.subg_id, batch.node_idx)
        args = (_csr_t(a, gpu), _csr_t(s, gpu), _t(batch.one_hot(), gpu), _t(w.W_n2l, gpu), _t(w.W_conv, gpu),
                _t(w.W_h1, gpu), _t(w.W_h2, gpu), 3)
        alone = _n(ops.s2v_forward(*args).logits)
        cases.append((args, alone))
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    outs = [[], []]
    for _ in range(6):
        for k in (0, 1):
            with torch.cuda.stream(streams[k]):
                outs[k].append(ops.s2v_forward(*cases[k][0]).logits)
    torch.cuda.synchronize()
    for k in (0, 1):
        for o in outs[k]:
            assert np.array_equal(_n(o), cases[k][1])


def test_one_launch_forward_with_batches_in_flight_on_several_streams(gpu, oracle):
    """the one-launch forward queued round-robin on three streams through calls bound once (three batches of
    different sizes, 300 graphs and more so that the graph order is made on each stream's own scratch, and small
    ones): every round gives each batch the bits it has alone"""
    import torch
    from graphnn_amd import ops
    cases = []
    for seed, B in ((11, 300), (12, 77), (13, 700)):
        batch = synth.molecule_batch(seed, B, 9, 2, size_mode="uniform", size_lo=3, size_hi=90)
        w = synth.make_weights(synth.Stream(seed), 9, 64, 16, 2)
        a = batching.node2node_csr(batch.num_nodes, batch.edge_x, batch.edge_y)
        s = batching.subgraph_csr(batch.num_graphs, batch.subg_id, batch.node_idx)
        args = (_csr_t(a, gpu), _csr_t(s, gpu), _t(batch.one_hot(), gpu), _t(w.W_n2l, gpu), _t(w.W_conv, gpu),
                _t(w.W_h1, gpu), _t(w.W_h2, gpu), 3, int(batch.graph_sizes.max()))
        alone = ops.s2v_forward_batched(*args)
        assert int(_n(alone.status)[0]) == 0
        cases.append((args, {k: _n(getattr(alone, k)) for k in ("h_final", "logits", "probs", "pred")}, batch))
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in cases]
    bufs = [ops.BatchedBuffers(c[2].num_nodes, c[2].num_graphs, 64, 16, 2, gpu) for c in cases]
    calls = [ops.bind_s2v_forward_batched(*cases[k][0], bufs[k], streams[k]) for k in range(len(cases))]
    for rnd in range(5):
        for b in bufs:
            b.logits.fill_(-1.0)
        torch.cuda.synchronize()
        for _ in range(4):
            for call in calls:
                call()
        torch.cuda.synchronize()
        for k, b in enumerate(bufs):
            assert int(_n(b.status)[0]) == 0
            for key, want in cases[k][1].items():
                assert np.array_equal(_n(getattr(b, key)), want), (rnd, k, key)


def test_forwards_replay_from_a_captured_graph(gpu, oracle):
    """once a stream has its scratch (a first eager call), the forwards queue kernels only (no allocation, no
    memset nodes): captured into a HIP graph through torch and replayed five times, with eager forwards and
    synchronisations between the replays, every replay gives the eager bits; both routes, and a batch of 300
    graphs whose one-launch forward has the graph-order launch ahead of it"""
    import torch
    from graphnn_amd import ops
    for B in (64, 300):
        batch, w, cfg = synth.make_config(2, B=B)
        a = batching.node2node_csr(batch.num_nodes, batch.edge_x, batch.edge_y)
        s = batching.subgraph_csr(batch.num_graphs, batch.subg_id, batch.node_idx)
        args = (_csr_t(a, gpu), _csr_t(s, gpu), _t(batch.one_hot(), gpu), _t(w.W_n2l, gpu), _t(w.W_conv, gpu),
                _t(w.W_h1, gpu), _t(w.W_h2, gpu), cfg["L"])
        nmax = int(batch.graph_sizes.max())
        stream = torch.cuda.Stream()
        gen = ops.ForwardBuffers(batch.num_nodes, B, cfg["C"], cfg["H"], cfg["Q"], gpu)
        one = ops.BatchedBuffers(batch.num_nodes, B, cfg["C"], cfg["H"], cfg["Q"], gpu)
        def both():
            ops.s2v_forward(*args, bufs=gen)
            ops.s2v_forward_batched(*args, nmax, bufs=one)
        with torch.cuda.stream(stream):
            both()
        torch.cuda.synchronize()
        want = (_n(gen.logits), _n(gen.pred), _n(one.logits), _n(one.h_final))
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            both()
        torch.cuda.synchronize()
        for rep in range(5):
            for t in (gen.logits, one.logits, one.h_final):
                t.fill_(-3.0)
            gen.pred.fill_(-1)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            got = (_n(gen.logits), _n(gen.pred), _n(one.logits), _n(one.h_final))
            for g_, w_ in zip(got, want):
                assert np.array_equal(g_, w_), (B, rep)
            with torch.cuda.stream(stream):
                both()                                       # the program's own eager work between replays
            torch.cuda.synchronize()
        assert int(_n(one.status)[0]) == 0


def test_forward_every_level_matches(gpu, oracle):
    """level by level through the per-level entry point, against each of the oracle's stored h_l"""
    from graphnn_amd import ops
    batch, w, cfg = synth.make_config(2, B=64)
    a = batching.node2node_csr(batch.num_nodes, batch.edge_x, batch.edge_y)
    s = batching.subgraph_csr(batch.num_graphs, batch.subg_id, batch.node_idx)
    X = batch.one_hot()
    want = oracle.forward(a, s, X, w, cfg["L"], batch.label_csr())
    a_d = _csr_t(a, gpu)
    msg, h = ops.s2v_input(_t(X, gpu), _t(w.W_n2l, gpu))
    assert max_rel(_n(h), want["h"][0]) < PARITY_TOL
    Wc = _t(w.W_conv, gpu)
    levels = [_n(h)]
    for lv in range(cfg["L"]):
        h = ops.s2v_level(*a_d, h, Wc, msg)
        assert max_rel(_n(h), want["h"][lv + 1]) < PARITY_TOL, lv
        levels.append(_n(h))
    assert_stages(" (level entry)", a, s, X, w, dict(msg=_n(msg), h=np.stack(levels)))


def test_forward_unfused_operator_route_agrees(gpu, oracle):
    """the same forward built from the general operators (the route FactorGraph takes op by op)"""
    from graphnn_amd import ops
    batch, cfg, a, s, X, w, lab, want, got, bufs = _forward_case(gpu, oracle, 1)
    a_d, s_d = _csr_t(a, gpu), _csr_t(s, gpu)
    Wn, Wc, W1, W2 = (_t(m, gpu) for m in (w.W_n2l, w.W_conv, w.W_h1, w.W_h2))
    msg = ops.gemm(_t(X, gpu), Wn)
    h = ops.relu(msg)
    for _ in range(cfg["L"]):
        pool = ops.spmm(*a_d, h, batch.num_nodes)
        lin = ops.gemm(pool, Wc)
        merged = ops.add(lin, msg)
        h = ops.relu(merged)
    y = ops.spmm(*s_d, h, batch.num_graphs)
    hidden = ops.relu(ops.gemm(y, W1))
    logits = ops.gemm(hidden, W2)
    probs = ops.row_softmax(logits.clone())
    assert max_rel(_n(logits), want["logits"]) < PARITY_TOL
    assert max_rel(_n(probs), want["probs"]) < PARITY_TOL
    assert max_rel(_n(logits), got["logits"]) < PARITY_TOL
    assert np.array_equal(_n(ops.row_argmax(logits)), want["pred"])


def test_forward_is_deterministic_and_reuses_buffers(gpu, oracle):
    from graphnn_amd import ops
    batch, cfg, a, s, X, w, lab, want, got, bufs = _forward_case(gpu, oracle, 1)
    args = (_csr_t(a, gpu), _csr_t(s, gpu), _t(X, gpu), _t(w.W_n2l, gpu), _t(w.W_conv, gpu), _t(w.W_h1, gpu), _t(w.W_h2, gpu))
    for _ in range(3):
        ops.s2v_forward(*args, cfg["L"], bufs=bufs)
        assert np.array_equal(_n(bufs.logits), got["logits"])
        assert np.array_equal(_n(bufs.h_final), got["h_final"])


# ------------------------------------------------------------------ pool allocator
def test_pool_recycles_blocks(gpu):
    import ctypes
    from graphnn_amd import _lib as binding
    lib = binding.load_library()
    used0, parked0, allocs0 = ctypes.c_size_t(), ctypes.c_size_t(), ctypes.c_size_t()
    lib.gnnhip_pool_stats(ctypes.byref(used0), ctypes.byref(parked0), ctypes.byref(allocs0))
    p = ctypes.c_void_p(); q = ctypes.c_void_p()
    assert lib.gnnhip_malloc(ctypes.byref(p), 1 << 20) == 0
    assert lib.gnnhip_recycle(p) == 0
    assert lib.gnnhip_malloc(ctypes.byref(q), (1 << 20) - 4096) == 0     # smallest parked block that is large enough
    assert q.value == p.value
    used, parked, allocs = ctypes.c_size_t(), ctypes.c_size_t(), ctypes.c_size_t()
    lib.gnnhip_pool_stats(ctypes.byref(used), ctypes.byref(parked), ctypes.byref(allocs))
    assert allocs.value == allocs0.value + 1
    # h2d / d2h round trip through the library's own copies
    src = np.arange(1000, dtype=np.float32); dst = np.zeros_like(src)
    P = lambda arr: arr.ctypes.data_as(ctypes.c_void_p)
    assert lib.gnnhip_memcpy_h2d(q, P(src), src.nbytes, None) == 0
    assert lib.gnnhip_memcpy_d2h(P(dst), q, src.nbytes, None) == 0
    assert np.array_equal(src, dst)
    assert lib.gnnhip_free(q) == 0
    assert lib.gnnhip_recycle(q) == -1                                   # no longer owned by the pool


# ------------------------------------------------------------------ graph-resident (one-launch) forward
def _batched_case(gpu, oracle, batch, w, L):
    from graphnn_amd import ops
    a = batching.node2node_csr(batch.num_nodes, batch.edge_x, batch.edge_y)
    s = batching.subgraph_csr(batch.num_graphs, batch.subg_id, batch.node_idx)
    X = batch.one_hot()
    want = _forward_want(oracle, a, s, X, w, L, batch.label_csr())
    want["_inputs"] = (a, s, X, w)
    bufs = ops.s2v_forward_batched(_csr_t(a, gpu), _csr_t(s, gpu), _t(X, gpu), _t(w.W_n2l, gpu), _t(w.W_conv, gpu),
                                   _t(w.W_h1, gpu), _t(w.W_h2, gpu), L, int(batch.graph_sizes.max()))
    return want, bufs


def _assert_batched_matches(want, bufs, L):
    assert int(_n(bufs.status)[0]) == 0
    got = {k: _n(getattr(bufs, k)) for k in ("msg", "h_final", "pool", "hidden", "logits", "probs")}
    _assert_forward_parity(got, want, L)
    if "_inputs" in want:
        assert_stages(" (one launch)", *want["_inputs"], got)
    assert np.array_equal(_n(bufs.pred), want["pred"])


@pytest.mark.parametrize("config_id", [1, 2])
def test_batched_forward_matches_reference_path(gpu, oracle, config_id):
    batch, w, cfg = synth.make_config(config_id)
    want, bufs = _batched_case(gpu, oracle, batch, w, cfg["L"])
    _assert_batched_matches(want, bufs, cfg["L"])


@pytest.mark.parametrize("C,K,H,Q,L", [(16, 7, 8, 3, 2), (32, 20, 16, 2, 3), (64, 64, 32, 5, 1), (64, 3, 100, 70, 0),
                                       (32, 48, 8, 2, 5), (16, 33, 4, 2, 1),
                                       # label counts around the steps of the input stage (two columns per 64-bit read)
                                       (64, 1, 8, 2, 2), (32, 2, 8, 2, 1), (64, 17, 16, 3, 2), (16, 49, 8, 2, 1),
                                       # hidden 128: eight wavefronts, a lane carries two columns through the readout
                                       (128, 7, 16, 2, 2), (128, 38, 32, 2, 4), (128, 64, 100, 70, 1), (128, 3, 8, 2, 0)])
def test_batched_forward_shapes(gpu, oracle, C, K, H, Q, L):
    seed = 1000 + C + K + L
    batch = synth.molecule_batch(seed, 37, K, Q, size_mode="uniform", size_lo=1, size_hi=70)
    w = synth.make_weights(synth.Stream(seed), K, C, H, Q)
    want, bufs = _batched_case(gpu, oracle, batch, w, L)
    _assert_batched_matches(want, bufs, L)


@pytest.mark.parametrize("C", [16, 64])
def test_batched_forward_graph_counts(gpu, oracle, C):
    """one graph, more graphs than compute units, exactly and more than the 1,024 workgroups of a launch (each
    workgroup then walks several graphs); graphs of 1..20 nodes, one of them empty of edges"""
    K, H, Q, L = 11, 8, 2, 3
    for B in (1, 257, 1024, 1025, 2500):
        seed = 17 * C + B
        batch = synth.molecule_batch(seed, B, K, Q, size_mode="uniform", size_lo=1, size_hi=20)
        w = synth.make_weights(synth.Stream(seed), K, C, H, Q)
        want, bufs = _batched_case(gpu, oracle, batch, w, L)
        _assert_batched_matches(want, bufs, L)


def test_batched_forward_large_and_dense_graphs(gpu, oracle):
    """a 200-node graph (more than 64 KB of LDS) next to a complete graph whose edge list is not staged in LDS"""
    from graphnn_amd import ops
    rng = np.random.default_rng(77)
    sizes = np.array([200, 100, 1, 17], np.int64)
    off = np.concatenate([[0], np.cumsum(sizes)])
    N, B, K, C, H, Q, L = int(off[-1]), 4, 9, 64, 32, 2, 3
    ex, ey = [], []
    for g, n in enumerate(sizes):
        if g == 1:                                   # complete graph: 9,900 directed edges
            a, b = np.meshgrid(np.arange(n), np.arange(n), indexing="ij")
            m = a != b
            ex.append(off[g] + a[m]); ey.append(off[g] + b[m])
        elif n > 1:                                  # ring plus chords
            i = np.arange(n)
            for step in (1, 7):
                ex += [off[g] + i, off[g] + (i + step) % n]; ey += [off[g] + (i + step) % n, off[g] + i]
    ex = np.concatenate(ex).astype(np.int32); ey = np.concatenate(ey).astype(np.int32)
    order = np.lexsort((ey, ex)); ex, ey = ex[order], ey[order]
    a = batching.node2node_csr(N, ex, ey)
    s = batching.subgraph_csr(B, np.repeat(np.arange(B), sizes).astype(np.int32), np.arange(N, dtype=np.int32))
    a = (a[0], a[1], (rng.random(a[1].size) * 0.05).astype(np.float32))           # non-unit edge weights
    s = (s[0], s[1], (rng.random(N) * 0.5).astype(np.float32))                    # weighted pooling
    X = rng.standard_normal((N, K)).astype(np.float32)
    w = synth.make_weights(synth.Stream(5), K, C, H, Q)
    want = _forward_want(oracle, a, s, X, w, L)
    bufs = ops.s2v_forward_batched(_csr_t(a, gpu), _csr_t(s, gpu), _t(X, gpu), _t(w.W_n2l, gpu), _t(w.W_conv, gpu),
                                   _t(w.W_h1, gpu), _t(w.W_h2, gpu), L, 200)
    _assert_batched_matches(want, bufs, L)
    # the general multi-launch forward gives the same answer on this batch
    gen = ops.s2v_forward(_csr_t(a, gpu), _csr_t(s, gpu), _t(X, gpu), _t(w.W_n2l, gpu), _t(w.W_conv, gpu),
                          _t(w.W_h1, gpu), _t(w.W_h2, gpu), L)
    assert max_rel(_n(gen.logits), _n(bufs.logits)) < PARITY_TOL


@pytest.mark.parametrize("B,C,hi", [(257, 64, 110), (300, 16, 40), (511, 64, 60), (512, 64, 60), (1023, 64, 70), (1500, 32, 33),
                                    (1024, 16, 20), (4096, 64, 40), (4097, 64, 40), (9000, 64, 24), (700, 64, 140)])
def test_batched_forward_of_more_graphs_than_compute_units(gpu, oracle, B, C, hi):
    """257 to 511 graphs: the one-launch forward hands the graphs to its workgroups largest first (an order a small
    launch ahead of it derives from the sizes).  From 512 graphs on, runs of consecutive graphs are packed into
    bins of 128 to 208 nodes that a workgroup carries through the levels as one block-diagonal graph, the readout
    running per graph (a small launch cuts the batch into bins, each 64 graphs on their own).  Either way every
    graph must come out exactly once: node outputs with the bits they have in a batch of at most 256 graphs
    (which is taken graph by graph, in batch order), graph outputs with those bits where the graphs are not
    packed and the same values where they are (the packed readout adds a graph's rows in order, as the reference
    path does).  Sizes 1..hi: several size classes, bins of one graph and of dozens"""
    from graphnn_amd import ops
    K, H, Q, L = 11, 16, 3, 2
    seed = 7000 + B
    batch = synth.molecule_batch(seed, B, K, Q, size_mode="uniform", size_lo=1, size_hi=hi)
    w = synth.make_weights(synth.Stream(seed), K, C, H, Q)
    a = batching.node2node_csr(batch.num_nodes, batch.edge_x, batch.edge_y)
    s = batching.subgraph_csr(batch.num_graphs, batch.subg_id, batch.node_idx)
    X = batch.one_hot()
    sizes = np.asarray(batch.graph_sizes).astype(np.int64)
    off = np.concatenate([[0], np.cumsum(sizes)])
    nmax = int(sizes.max())
    wts = (_t(w.W_n2l, gpu), _t(w.W_conv, gpu), _t(w.W_h1, gpu), _t(w.W_h2, gpu))
    keys = ("msg", "h_final", "pool", "hidden", "logits", "probs", "pred")
    packed = B >= 512
    big = ops.s2v_forward_batched(_csr_t(a, gpu), _csr_t(s, gpu), _t(X, gpu), *wts, L, nmax)
    assert int(_n(big.status)[0]) == 0
    got = {k: _n(getattr(big, k)) for k in keys}
    for b0 in range(0, B, 256):
        b1 = min(B, b0 + 256)
        n0, n1 = int(off[b0]), int(off[b1])
        e0, e1 = int(a[0][n0]), int(a[0][n1])
        a_part = (a[0][n0:n1 + 1] - e0, a[1][e0:e1] - n0, a[2][e0:e1])
        s_part = ((off[b0:b1 + 1] - n0).astype(np.int32), np.arange(n1 - n0, dtype=np.int32), np.ones(n1 - n0, np.float32))
        part = ops.s2v_forward_batched(_csr_t(a_part, gpu), _csr_t(s_part, gpu), _t(X[n0:n1], gpu), *wts, L, nmax)
        assert int(_n(part.status)[0]) == 0
        for k in keys:
            rows = slice(n0, n1) if k in ("msg", "h_final") else slice(b0, b1)
            ref = _n(getattr(part, k))
            if not packed or k in ("msg", "h_final"):
                assert np.array_equal(got[k][rows], ref), (k, b0)
        if packed:
            # the graph outputs of the packed readout against the reference path (float64 settles a miss)
            want_p = _forward_want(oracle, a_part, s_part, X[n0:n1], w, L)
            gk = ("pool", "hidden", "logits", "probs")
            _assert_forward_parity({k: got[k][b0:b1] for k in gk}, want_p, L, tag=" graphs %d.." % b0, keys=gk)
            # arg-max: equal unless the two largest logits are within rounding of each other
            lg = want_p["logits"].astype(np.float64)
            top2 = np.sort(lg, axis=1)[:, -2:]
            clear = (top2[:, 1] - top2[:, 0]) > 1e-4 * np.abs(lg).max()
            assert clear.sum() > 0.9 * (b1 - b0)
            assert np.array_equal(got["pred"][b0:b1][clear], want_p["pred"][clear]), b0
    if B <= 700 and not packed:
        want = _forward_want(oracle, a, s, X, w, L)
        _assert_forward_parity({k: got[k] for k in ("msg", "h_final", "pool", "hidden", "logits", "probs")}, want, L)
    # a promise one tile short of the largest graphs: they are refused, every other graph keeps its values.
    # (Packed batches take the promise as at least the bin size, 128 to 208 nodes: see the test below.)
    short = (nmax - 1) // 16 * 16
    if short >= 16 and not packed:
        fresh = ops.BatchedBuffers(batch.num_nodes, B, C, H, Q, gpu)
        for k in ("pool", "logits"):
            getattr(fresh, k).fill_(-7.0)
        ops.s2v_forward_batched(_csr_t(a, gpu), _csr_t(s, gpu), _t(X, gpu), *wts, L, short, bufs=fresh)
        assert int(_n(fresh.status)[0]) & 1
        fits = sizes <= short
        assert 0 < fits.sum() < B
        # (a smaller promise may pick a workgroup shape that adds in another order: the same values, not the same bits)
        assert max_rel(_n(fresh.logits)[fits], got["logits"][fits]) < PARITY_TOL
        assert max_rel(_n(fresh.pool)[fits], got["pool"][fits]) < PARITY_TOL
        assert np.all(_n(fresh.logits)[~fits] == -7.0)


@pytest.mark.parametrize("C,K,B", [(16, 60, 700), (32, 7, 900), (32, 60, 700), (32, 200, 700), (64, 7, 600), (16, 7, 300), (32, 40, 400)])
@pytest.mark.parametrize("degree", [2, 9, 30])
def test_batched_forward_whatever_the_entry_count_is_said_to_be(gpu, oracle, C, K, B, degree):
    """the host's entry count decides how many workgroups share a compute unit's LDS, and with it how many entries fit the edge
    cache: batches whose bins fit it, half fit it and never fit it, with the count said to be right, none, enormous and
    (the entries without it) unknown: the same bits every time, and the oracle's values.  K = 200: labels"""
    import torch
    from graphnn_amd import ops
    rng = np.random.default_rng(1000 * C + 10 * K + degree)
    H, Q, L = 16, 3, 2
    sizes = rng.integers(30, 61, B)
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    N = int(off[-1])
    per_row = rng.integers(0, 2 * degree + 1, N)
    a_rp = np.concatenate([[0], np.cumsum(per_row)]).astype(np.int32)
    graph = np.repeat(np.repeat(np.arange(B), sizes), per_row)
    a = (a_rp, (off[graph] + (rng.random(graph.size) * sizes[graph]).astype(np.int64)).astype(np.int32),
         (rng.random(graph.size) / degree).astype(np.float32))
    s = (off, np.arange(N, dtype=np.int32), np.ones(N, np.float32))
    w = synth.make_weights(synth.Stream(C + K), K, C, H, Q)
    label = rng.integers(0, K, N).astype(np.int32)
    labels = K > 64
    X = np.eye(K, dtype=np.float32)[label]
    a_d, s_d = _csr_t(a, gpu), _csr_t(s, gpu)
    wts = [_t(m, gpu) for m in (w.W_n2l, w.W_conv, w.W_h1, w.W_h2)]
    x = _t(label if labels else X, gpu)
    run = (ops.s2v_forward_batched_labels if labels else ops.s2v_forward_batched)
    keys = ("msg", "h_final", "pool", "hidden", "logits", "probs", "pred")
    bufs = run(a_d, s_d, x, *wts, L, 60)
    got = {k: _n(getattr(bufs, k)) for k in keys}
    assert int(_n(bufs.status)[0]) == 0
    sized = getattr(ops._bound(), "s2v_forward_batched_labels_sized_f32" if labels else "s2v_forward_batched_sized_f32")
    plain = getattr(ops._lib(), "gnnhip_s2v_forward_batched_labels_f32" if labels else "gnnhip_s2v_forward_batched_f32")
    for count in (0, 2 ** 31 - 1, None):
        o = ops.BatchedBuffers(N, B, C, H, Q, gpu)
        args = [*a_d, *s_d, x, *wts, o.msg, o.h_final, o.pool, o.hidden, o.logits, o.probs, o.pred, o.status]
        if count is not None:
            sized(N, B, K, C, H, Q, L, 60, count, *args)
        else:
            assert plain(N, B, K, C, H, Q, L, 60, *[ctypes.c_void_p(t.data_ptr()) for t in args], ops._stream()) == 0
        torch.cuda.synchronize()
        for k in keys:
            assert np.array_equal(_n(getattr(o, k)), got[k]), (count, k)
    want = _forward_want(oracle, a, s, X, w, L)
    _assert_forward_parity({k: got[k] for k in keys[:-1]}, want, L)


def test_packed_batch_refuses_a_graph_larger_than_a_bin(gpu, oracle):
    """600 graphs of up to 40 nodes, one of them grown to 300 nodes, promise 40: the batch is packed into bins, the
    large graph is a bin of its own that no workgroup can hold: status bit 0, its outputs untouched, every other
    graph as without it"""
    from graphnn_amd import ops
    K, C, H, Q, L = 7, 32, 8, 2, 2
    sizes = np.random.default_rng(3).integers(1, 41, 600)
    sizes[321] = 300
    # chains: node i of a graph is joined to node i + 1
    off = np.concatenate([[0], np.cumsum(sizes)])
    ex, ey = [], []
    for g, n in enumerate(sizes):
        i = np.arange(n - 1) + off[g]
        ex += [i, i + 1]; ey += [i + 1, i]
    ex = np.concatenate(ex).astype(np.int32); ey = np.concatenate(ey).astype(np.int32)
    order = np.lexsort((ey, ex)); ex, ey = ex[order], ey[order]
    N, B = int(off[-1]), sizes.size
    a = batching.node2node_csr(N, ex, ey)
    s = batching.subgraph_csr(B, np.repeat(np.arange(B), sizes).astype(np.int32), np.arange(N, dtype=np.int32))
    rng = np.random.default_rng(4)
    X = rng.standard_normal((N, K)).astype(np.float32)
    w = synth.make_weights(synth.Stream(77), K, C, H, Q)
    wts = (_t(w.W_n2l, gpu), _t(w.W_conv, gpu), _t(w.W_h1, gpu), _t(w.W_h2, gpu))
    bufs = ops.BatchedBuffers(N, B, C, H, Q, gpu)
    bufs.logits.fill_(-7.0)
    ops.s2v_forward_batched(_csr_t(a, gpu), _csr_t(s, gpu), _t(X, gpu), *wts, L, 40, bufs=bufs)
    assert int(_n(bufs.status)[0]) == 1
    lg = _n(bufs.logits)
    assert np.all(lg[321] == -7.0)
    want = _forward_want(oracle, a, s, X, w, L)
    keep = np.arange(B) != 321
    assert max_rel(lg[keep], want["logits"][keep]) < PARITY_TOL
    assert np.array_equal(_n(bufs.pred)[keep], want["pred"][keep])


@pytest.mark.parametrize("B", [40, 300, 600, 1100])
def test_batched_forward_with_graphs_of_no_nodes(gpu, oracle, B):
    """graphs without nodes between the others (rows of S without entries; GetBatch never makes them, the operand
    allows them): pooled features of zero and the logits of a zero vector, through every way the one-launch forward
    hands out its graphs (in batch order, largest first, packed into bins), the first and the last graph among them"""
    from graphnn_amd import ops
    K, C, H, Q, L = 9, 32, 16, 3, 2
    rng = np.random.default_rng(50 + B)
    sizes = rng.integers(1, 31, B)
    sizes[rng.random(B) < 0.2] = 0
    sizes[[0, B - 1, B // 2, B // 2 + 1]] = 0
    off = np.concatenate([[0], np.cumsum(sizes)])
    ex, ey = [], []
    for g, n in enumerate(sizes):
        if n < 2:
            continue
        i = np.arange(n - 1) + off[g]
        ex += [i, i + 1]; ey += [i + 1, i]
    ex = np.concatenate(ex).astype(np.int32); ey = np.concatenate(ey).astype(np.int32)
    N = int(off[-1])
    a = batching.node2node_csr(N, ex, ey)
    s = (off.astype(np.int32), np.arange(N, dtype=np.int32), np.ones(N, np.float32))
    X = rng.standard_normal((N, K)).astype(np.float32)
    w = synth.make_weights(synth.Stream(78), K, C, H, Q)
    wts = (_t(w.W_n2l, gpu), _t(w.W_conv, gpu), _t(w.W_h1, gpu), _t(w.W_h2, gpu))
    bufs = ops.s2v_forward_batched(_csr_t(a, gpu), _csr_t(s, gpu), _t(X, gpu), *wts, L, 32)
    assert int(_n(bufs.status)[0]) == 0
    want = _forward_want(oracle, a, s, X, w, L)
    keys = ("msg", "h_final", "pool", "hidden", "logits", "probs")
    _assert_forward_parity({k: _n(getattr(bufs, k)) for k in keys}, want, L)
    none = sizes == 0
    assert np.all(_n(bufs.pool)[none] == 0) and np.all(_n(bufs.logits)[none] == 0)
    assert np.array_equal(_n(bufs.pred)[none], want["pred"][none])


@pytest.mark.parametrize("C,L,B", [(64, 4, 256), (16, 1, 37), (32, 3, 300), (64, 0, 9), (128, 3, 100), (128, 4, 256)])
def test_batched_forward_keeps_every_level_for_training(gpu, oracle, C, L, B):
    """the one-launch forward of a training iteration: h_0 .. h_L as the per-level entry points give them (which
    have their own parity tests), every other output with the bits of the inference entry"""
    from graphnn_amd import ops
    K, H, Q = 9, 16, 2
    batch = synth.molecule_batch(4000 + C + B, B, K, Q, size_mode="uniform", size_lo=2, size_hi=90)
    w = synth.make_weights(synth.Stream(4000 + C), K, C, H, Q)
    a = batching.node2node_csr(batch.num_nodes, batch.edge_x, batch.edge_y)
    s = batching.subgraph_csr(batch.num_graphs, batch.subg_id, batch.node_idx)
    args = (_csr_t(a, gpu), _csr_t(s, gpu), _t(batch.one_hot(), gpu), _t(w.W_n2l, gpu), _t(w.W_conv, gpu),
            _t(w.W_h1, gpu), _t(w.W_h2, gpu), L, int(batch.graph_sizes.max()))
    plain = ops.s2v_forward_batched(*args)
    bufs, hl = ops.s2v_forward_batched_train(*args)
    assert int(_n(bufs.status)[0]) == 0 and tuple(hl.shape) == (L + 1, batch.num_nodes, C)
    for k in ("msg", "pool", "hidden", "logits", "probs", "pred"):
        assert np.array_equal(_n(getattr(bufs, k)), _n(getattr(plain, k))), k
    assert np.array_equal(_n(hl[L]), _n(plain.h_final))
    want = _forward_want(oracle, a, s, batch.one_hot(), w, L, None)
    for l in range(L + 1):
        assert_parity("h%d" % l, _n(hl[l]), want["h"][l], want["_f64"]["h"][l])
    assert np.array_equal(_n(hl[0]), np.maximum(_n(bufs.msg), 0))
    assert_stages(" (one launch, levels kept)", a, s, batch.one_hot(), w,
                  dict(msg=_n(bufs.msg), h=_n(hl), pool=_n(bufs.pool), hidden=_n(bufs.hidden), logits=_n(bufs.logits), probs=_n(bufs.probs)))


def test_batched_forward_dense_features_past_the_staging_registers(gpu, oracle):
    """64 real-valued feature columns on graphs of up to 190 nodes: a graph's block of X (12,160 floats) is longer
    than what the lanes stage in one go, and its rows outnumber the gather rounds kept in registers"""
    from graphnn_amd import ops
    rng = np.random.default_rng(123)
    K, C, H, Q, L = 64, 64, 32, 2, 2
    batch = synth.molecule_batch(321, 9, K, Q, size_mode="uniform", size_lo=150, size_hi=190)
    w = synth.make_weights(synth.Stream(321), K, C, H, Q)
    a = batching.node2node_csr(batch.num_nodes, batch.edge_x, batch.edge_y)
    s = batching.subgraph_csr(batch.num_graphs, batch.subg_id, batch.node_idx)
    X = rng.standard_normal((batch.num_nodes, K)).astype(np.float32)
    want = _forward_want(oracle, a, s, X, w, L)
    bufs = ops.s2v_forward_batched(_csr_t(a, gpu), _csr_t(s, gpu), _t(X, gpu), _t(w.W_n2l, gpu), _t(w.W_conv, gpu),
                                   _t(w.W_h1, gpu), _t(w.W_h2, gpu), L, int(batch.graph_sizes.max()))
    _assert_batched_matches(want, bufs, L)


def test_batched_forward_reports_broken_promises(gpu, oracle):
    from graphnn_amd import ops
    from graphnn_amd._lib import GnnHipError
    batch, w, cfg = synth.make_config(1, B=8)
    a = batching.node2node_csr(batch.num_nodes, batch.edge_x, batch.edge_y)
    s = batching.subgraph_csr(batch.num_graphs, batch.subg_id, batch.node_idx)
    X = batch.one_hot()
    dev_w = (_t(w.W_n2l, gpu), _t(w.W_conv, gpu), _t(w.W_h1, gpu), _t(w.W_h2, gpu))
    nmax = int(batch.graph_sizes.max())
    # a graph larger than promised: bit 0, nothing overruns
    assert nmax > 16                                          # the promise is checked at 16-row granularity
    bufs = ops.s2v_forward_batched(_csr_t(a, gpu), _csr_t(s, gpu), _t(X, gpu), *dev_w, cfg["L"], 16)
    assert int(_n(bufs.status)[0]) & 1
    # an edge that joins two graphs: bit 1
    bad_col = a[1].copy()
    bad_col[0] = batch.num_nodes - 1
    bufs = ops.s2v_forward_batched((_t(a[0], gpu), _t(bad_col, gpu), _t(a[2], gpu)), _csr_t(s, gpu), _t(X, gpu), *dev_w,
                                   cfg["L"], nmax)
    assert int(_n(bufs.status)[0]) & 2
    # a pooling matrix that is not the identity layout: bit 2
    bad_s = s[1].copy(); bad_s[[0, 1]] = bad_s[[1, 0]]
    bufs = ops.s2v_forward_batched(_csr_t(a, gpu), (_t(s[0], gpu), _t(bad_s, gpu), _t(s[2], gpu)), _t(X, gpu), *dev_w,
                                   cfg["L"], nmax)
    assert int(_n(bufs.status)[0]) & 4
    # shapes outside the kernel's range are refused without launching
    with pytest.raises(GnnHipError) as err:
        ops.s2v_forward_batched(_csr_t(a, gpu), _csr_t(s, gpu), _t(X, gpu), *dev_w, cfg["L"], 5000)
    assert err.value.code == -5


# ------------------------------------------------------------------ label input (one int per node instead of one-hot X)
@pytest.mark.parametrize("C,K,N", [(64, 38, 7450), (16, 7, 333), (128, 64, 5001), (256, 3, 1000), (48, 100, 777), (7, 5, 100)])
def test_input_labels_is_the_one_hot_product_bit_for_bit(gpu, oracle, C, K, N):
    import torch
    from graphnn_amd import ops
    rng = np.random.default_rng(C + K)
    lab = rng.integers(0, K, N).astype(np.int32)
    W = (rng.standard_normal((K, C)) * 0.1).astype(np.float32)
    W[0, :3] = -0.0                                              # the product turns -0.0 into +0.0; so must the lookup
    lab[:5] = 0
    X = np.zeros((N, K), np.float32); X[np.arange(N), lab] = 1.0
    want = oracle.gemm(X, W)
    status = torch.zeros(1, dtype=torch.int32, device=gpu)
    msg, h0 = ops.s2v_input_labels(_t(lab, gpu), _t(W, gpu), status)
    assert np.array_equal(_n(msg).view(np.int32), want.view(np.int32))
    assert np.array_equal(_n(h0).view(np.int32), np.maximum(want, 0).view(np.int32))
    assert int(_n(status)[0]) == 0
    # the dense input stage of the library gives the same bits
    msg_d, h0_d = ops.s2v_input(_t(X, gpu), _t(W, gpu))
    assert np.array_equal(_n(msg_d).view(np.int32), _n(msg).view(np.int32))
    # a label outside [0, K) is reported and clamped
    bad = lab.copy(); bad[7] = K; bad[8] = -3
    msg_b, _ = ops.s2v_input_labels(_t(bad, gpu), _t(W, gpu), status)
    assert int(_n(status)[0]) == 8
    assert np.array_equal(_n(msg_b)[7], want[lab == K - 1][0] if (lab == K - 1).any() else _n(msg_b)[7])
    assert np.array_equal(_n(msg_b)[8].view(np.int32), want[0].view(np.int32))


@pytest.mark.parametrize("config_id", [1, 2])
def test_batched_forward_from_labels_has_the_bits_of_the_one_hot_route(gpu, oracle, config_id):
    from graphnn_amd import ops
    batch, w, cfg = synth.make_config(config_id)
    want, bufs = _batched_case(gpu, oracle, batch, w, cfg["L"])
    a = batching.node2node_csr(batch.num_nodes, batch.edge_x, batch.edge_y)
    s = batching.subgraph_csr(batch.num_graphs, batch.subg_id, batch.node_idx)
    lab = batch.node_label.astype(np.int32)
    got = ops.s2v_forward_batched_labels(_csr_t(a, gpu), _csr_t(s, gpu), _t(lab, gpu), _t(w.W_n2l, gpu), _t(w.W_conv, gpu),
                                         _t(w.W_h1, gpu), _t(w.W_h2, gpu), cfg["L"], int(batch.graph_sizes.max()))
    assert int(_n(got.status)[0]) == 0
    for key in ("msg", "h_final", "pool", "hidden", "logits", "probs", "pred"):
        assert np.array_equal(_n(getattr(got, key)), _n(getattr(bufs, key))), key
    _assert_batched_matches(want, got, cfg["L"])


@pytest.mark.parametrize("C,K,H,Q,L,B", [(16, 7, 8, 3, 2, 37), (32, 200, 16, 2, 3, 300), (64, 64, 32, 5, 1, 1025), (64, 1, 8, 2, 0, 9),
                                         (64, 130, 32, 2, 2, 40), (128, 38, 32, 2, 4, 256), (128, 100, 16, 3, 2, 300)])
def test_batched_forward_from_labels_shapes(gpu, oracle, C, K, H, Q, L, B):
    """label tables that fit LDS (K C <= 8192 floats) and ones read from L2, more than 64 label types (the dense
    route stops at 64 columns), no level, more graphs than workgroups; a label out of range sets status bit 3"""
    from graphnn_amd import ops
    seed = 2000 + C + K + L
    batch = synth.molecule_batch(seed, B, K, Q, size_mode="uniform", size_lo=1, size_hi=70)
    w = synth.make_weights(synth.Stream(seed), K, C, H, Q)
    a = batching.node2node_csr(batch.num_nodes, batch.edge_x, batch.edge_y)
    s = batching.subgraph_csr(batch.num_graphs, batch.subg_id, batch.node_idx)
    want = _forward_want(oracle, a, s, batch.one_hot(), w, L)
    lab = batch.node_label.astype(np.int32)
    args = (_csr_t(a, gpu), _csr_t(s, gpu))
    wts = (_t(w.W_n2l, gpu), _t(w.W_conv, gpu), _t(w.W_h1, gpu), _t(w.W_h2, gpu))
    got = ops.s2v_forward_batched_labels(*args, _t(lab, gpu), *wts, L, int(batch.graph_sizes.max()))
    _assert_batched_matches(want, got, L)
    bad = lab.copy(); bad[batch.num_nodes // 2] = K + 5
    got = ops.s2v_forward_batched_labels(*args, _t(bad, gpu), *wts, L, int(batch.graph_sizes.max()))
    assert int(_n(got.status)[0]) == 8


# ------------------------------------------------------------------ backward-pass kernels
@pytest.mark.parametrize("n", [2, 7, 64, 128])
def test_spmm_transposed(gpu, oracle, n):
    from graphnn_amd import ops
    rng = np.random.default_rng(300 + n)
    m, k = 411, 233
    csr = _random_csr(rng, m, k, 3000)                       # duplicates present
    B = rng.standard_normal((m, n)).astype(np.float32)
    C0 = rng.standard_normal((k, n)).astype(np.float32)
    got = _n(ops.spmm_t(*_csr_t(csr, gpu), _t(B, gpu), m, k))
    assert max_rel(got, oracle.spmm_T(*csr, B, m, k)) < PARITY_TOL
    got2 = _n(ops.spmm_t(*_csr_t(csr, gpu), _t(B, gpu), m, k, alpha=0.5, beta=2.0, out=_t(C0, gpu)))
    assert max_rel(got2, oracle.spmm_T(*csr, B, m, k, alpha=0.5, beta=2.0, C=C0)) < PARITY_TOL
    # the reference's own SparseMM case (A^T B), test/gpu_tensor_test.cpp:311-336
    g = json.load(open(os.path.join(GOLDEN, "sparse_mm_known_answer.json")))
    kc = (np.array(g["row_ptr"], np.int32), np.array(g["col_idx"], np.int32), np.array(g["val"], np.float32))
    got3 = _n(ops.spmm_t(*_csr_t(kc, gpu), _t(np.array(g["b_for_transpose"], np.float32), gpu), g["a_rows"], g["a_cols"]))
    assert np.array_equal(got3, np.array(g["expected_At_b"], np.float32))


def test_gradient_elementwise_kernels(gpu):
    from graphnn_amd import ops
    rng = np.random.default_rng(31)
    n = 10007
    out = rng.standard_normal(n).astype(np.float32); out[::5] = 0.0
    grad = rng.standard_normal(n).astype(np.float32)
    dst = rng.standard_normal(n).astype(np.float32)
    got = _n(ops.relu_deriv(_t(dst, gpu), _t(out, gpu), _t(grad, gpu)))
    assert np.array_equal(got, np.where(out > 0, dst + grad, dst))
    x = rng.standard_normal(n).astype(np.float32); y = rng.standard_normal(n).astype(np.float32)
    assert np.array_equal(_n(ops.mul(_t(x, gpu), _t(y, gpu))), x * y)
    M = rng.standard_normal((37, 5)).astype(np.float32); s = rng.standard_normal(37).astype(np.float32)
    assert np.array_equal(_n(ops.row_scale(_t(s, gpu), _t(M, gpu))), M * s[:, None])
    # dense += a * sparse, duplicates in a row accumulate in order
    rp = np.array([0, 2, 2, 5], np.int32); ci = np.array([1, 1, 0, 3, 0], np.int32); v = np.array([1, 2, 3, 4, 5], np.float32)
    D = np.zeros((3, 4), np.float32)
    want = D.copy()
    for r in range(3):
        for t in range(rp[r], rp[r + 1]):
            want[r, ci[t]] += np.float32(-0.5) * v[t]
    assert np.array_equal(_n(ops.csr_axpy(-0.5, _t(rp, gpu), _t(ci, gpu), _t(v, gpu), _t(D, gpu))), want)
    big = (rng.random(300001) * 2 - 1).astype(np.float32)
    ss = float(_n(ops.reduce("sumsq", _t(big, gpu)))[0])
    assert abs(ss - float((big.astype(np.float64) ** 2).sum())) <= 1e-5 * ss


# ------------------------------------------------------------------ skewed degrees (hub rows)
def _hub_matrix(rng, m, k, long_rows):
    """CSR with short random rows and a few very long ones next to each other"""
    lens = rng.integers(0, 5, m)
    for r, d in long_rows:
        lens[r] = d
    rp = np.zeros(m + 1, np.int32); np.cumsum(lens, out=rp[1:])
    nnz = int(rp[-1])
    ci = rng.integers(0, k, nnz).astype(np.int32)
    v = (rng.random(nnz) * 0.5 + 0.25).astype(np.float32)
    return rp, ci, v


@pytest.mark.parametrize("n", [4, 64, 100])
def test_spmm_long_rows_around_the_row_count_threshold(gpu, oracle, n):
    """the balanced pass over long rows starts at 32,768 rows; below it a long row is split inside one workgroup.
    The same long rows (65, 2,048, 2,049, 5,000 entries, first and last row) one row below, at and above it."""
    from graphnn_amd import ops
    for m in (32_767, 32_768, 32_769):
        rng = np.random.default_rng(m + n)
        k = 5000
        csr = _hub_matrix(rng, m, k, [(0, 5000), (9, 65), (10, 2048), (11, 2049), (m // 2, 64), (m - 1, 3000)])
        B = rng.standard_normal((k, n)).astype(np.float32)
        got = _n(ops.spmm(*_csr_t(csr, gpu), _t(B, gpu), m))
        want, w64 = _spmm_want(oracle, *csr, B, m)
        assert_parity("spmm m=%d" % m, got, want, w64)


@pytest.mark.parametrize("n", [64, 128, 7, 36, 300])
def test_spmm_hub_rows_balanced_pass(gpu, oracle, n):
    """matrix large enough for the balanced pass over long rows: rows of 65 and 257 (one chunk), 2048, 2049 and
    9000 entries (several chunks), 64 (just below the threshold), neighbours at the low indices, an empty row between them"""
    from graphnn_amd import ops
    rng = np.random.default_rng(500 + n)
    m = k = 40000
    csr = _hub_matrix(rng, m, k, [(0, 9000), (1, 2049), (2, 0), (3, 2048), (4, 257), (5, 256), (6, 65), (7, 64), (17000, 5000), (m - 1, 700)])
    B = rng.standard_normal((k, n)).astype(np.float32)
    C0 = rng.standard_normal((m, n)).astype(np.float32)
    got = _n(ops.spmm(*_csr_t(csr, gpu), _t(B, gpu), m))
    want, w64 = _spmm_want(oracle, *csr, B, m)
    assert_parity("spmm", got, want, w64)
    got2 = _n(ops.spmm(*_csr_t(csr, gpu), _t(B, gpu), m, alpha=-0.5, beta=1.5, out=_t(C0, gpu)))
    assert_parity("spmm", got2, *_spmm_want(oracle, *csr, B, m, alpha=-0.5, beta=1.5, C=C0))
    # deterministic: the same bits on a second run
    assert np.array_equal(got, _n(ops.spmm(*_csr_t(csr, gpu), _t(B, gpu), m)))


@pytest.mark.parametrize("n", [3, 5, 13, 17, 31, 101, 259, 1026])
def test_spmm_rows_of_any_alignment(gpu, oracle, n):
    """widths whose rows end inside a lane's four columns (the last unit is moved back, also across two sets of columns per
    lane and in a last slab of two), and narrow ones, whose wavefronts copy their rows' entries first: runs of rows just
    inside and past what is copied at once (768 entries), empty rows, a deferred row and a ragged end; also above
    32,768 rows, where long rows come from the balanced pass"""
    from graphnn_amd import ops
    for m in (1_003, 32_801):
        if m > 2_000 and n > 300:
            continue
        rng = np.random.default_rng(1200 + n + m)
        k = 701
        long_rows = [(r, 48) for r in range(64, 80)] + [(r, 49) for r in range(128, 144)] + [(200, 0), (201, 2_500), (m - 2, 0), (m - 1, 70)]
        csr = _hub_matrix(rng, m, k, long_rows)
        B = rng.standard_normal((k, n)).astype(np.float32)
        C0 = rng.standard_normal((m, n)).astype(np.float32)
        got = _n(ops.spmm(*_csr_t(csr, gpu), _t(B, gpu), m))
        assert_parity("spmm", got, *_spmm_want(oracle, *csr, B, m))
        got2 = _n(ops.spmm(*_csr_t(csr, gpu), _t(B, gpu), m, alpha=-0.5, beta=1.5, out=_t(C0, gpu)))
        assert_parity("spmm", got2, *_spmm_want(oracle, *csr, B, m, alpha=-0.5, beta=1.5, C=C0))


@pytest.mark.parametrize("m,n", [(37, 64), (300, 7), (1, 128), (2000, 300), (4096, 4)])
def test_spmm_few_long_rows_take_a_workgroup_each(gpu, oracle, m, n):
    """rows of several hundred entries on average and fewer than 32,768 of them (sum-pooling into subgraphs): every
    row is summed by a whole workgroup; empty rows, a row of one entry and a row of 5,000 among them; alpha, beta"""
    from graphnn_amd import ops
    rng = np.random.default_rng(900 + m + n)
    k = 20_000
    lens = rng.integers(200, 700, m)
    lens[0] = 5_000
    if m > 3:
        lens[1] = 0; lens[2] = 1; lens[m - 1] = 0
    rp = np.zeros(m + 1, np.int32); np.cumsum(lens, out=rp[1:])
    nnz = int(rp[-1])
    assert nnz >= 256 * m
    ci = rng.integers(0, k, nnz).astype(np.int32)
    v = (rng.random(nnz) * 0.2 - 0.05).astype(np.float32)
    csr = (rp, ci, v)
    B = rng.standard_normal((k, n)).astype(np.float32)
    C0 = rng.standard_normal((m, n)).astype(np.float32)
    got = _n(ops.spmm(*_csr_t(csr, gpu), _t(B, gpu), m))
    assert_parity("spmm", got, *_spmm_want(oracle, *csr, B, m))
    got2 = _n(ops.spmm(*_csr_t(csr, gpu), _t(B, gpu), m, alpha=-0.5, beta=1.5, out=_t(C0, gpu)))
    assert_parity("spmm", got2, *_spmm_want(oracle, *csr, B, m, alpha=-0.5, beta=1.5, C=C0))
    assert np.array_equal(got, _n(ops.spmm(*_csr_t(csr, gpu), _t(B, gpu), m)))
    if m > 3:
        assert np.all(got[1] == 0) and np.array_equal(got2[1], (1.5 * C0[1]).astype(np.float32))


@pytest.mark.parametrize("n", [64, 128, 9, 36, 300, 32, 4, 520, 150])
def test_spmm_column_ordered_pieces_on_a_power_law_matrix(gpu, oracle, n):
    """R-MAT, 65,536 rows, 16 entries per row on average (rows of up to 13,000 entries, a third of the rows
    empty): large and dense enough for the route that cuts rows into pieces of 32 entries and sums them in the
    order of their first column (operands of at least eight column units; width 4 stays with the row-group
    route); random weights, alpha and beta, the same bits on a second run"""
    from graphnn_amd import ops
    rng = np.random.default_rng(600 + n)
    a = synth.rmat_csr(0x5EED0005, 16, 16 << 16)
    N = 1 << 16
    assert (np.diff(a[0]) == 0).sum() > 1000 and np.diff(a[0]).max() > 5000
    v = (rng.random(a[1].size) * 0.2 - 0.05).astype(np.float32)
    csr = (a[0], a[1], v)
    B = rng.standard_normal((N, n)).astype(np.float32)
    C0 = rng.standard_normal((N, n)).astype(np.float32)
    got = _n(ops.spmm(*_csr_t(csr, gpu), _t(B, gpu), N))
    want, w64 = _spmm_want(oracle, *csr, B, N)
    assert_parity("spmm", got, want, w64)
    got2 = _n(ops.spmm(*_csr_t(csr, gpu), _t(B, gpu), N, alpha=-0.5, beta=1.5, out=_t(C0, gpu)))
    assert_parity("spmm", got2, *_spmm_want(oracle, *csr, B, N, alpha=-0.5, beta=1.5, C=C0))
    assert np.array_equal(got, _n(ops.spmm(*_csr_t(csr, gpu), _t(B, gpu), N)))
    # rows of at most 32 entries are one piece each: their sums are the row-order sums of the reference path
    short = np.diff(a[0]) <= 32
    unit = (a[0], a[1], np.ones_like(v))
    got_u = _n(ops.spmm(*_csr_t(unit, gpu), _t(B, gpu), N))
    assert np.array_equal(got_u[short], oracle.spmm(*unit, B, N)[short])
    # a host-side entry count below the matrix's own (but still dense enough for this route): the plan covers the
    # rows that end inside it, the last rows are summed from the CSR arrays
    for hint in (a[1].size - 1, 13 * N):
        got_h = _n(ops.spmm(*_csr_t(csr, gpu), _t(B, gpu), N, alpha=-0.5, beta=1.5, out=_t(C0, gpu), nnz_hint=hint))
        inside = a[0][1:] <= hint
        assert 0 < inside.sum() < N
        assert np.array_equal(got_h[inside], got2[inside]), hint
        assert_parity("spmm", got_h, *_spmm_want(oracle, *csr, B, N, alpha=-0.5, beta=1.5, C=C0))


@pytest.mark.parametrize("k", [1, 256, 257, 1 << 20, (1 << 20) + 1])
def test_spmm_pieces_whatever_bits_their_order_takes(gpu, oracle, k):
    """rows cut into pieces, as above, with as many columns as the eight bits their order takes up to 2^20 columns, one more,
    and either side of that line; rows of at most 32 entries have the bits of the row-order sums whatever the order"""
    from graphnn_amd import ops
    rng = np.random.default_rng(k)
    m, n = 32768, 32
    deg = rng.integers(4, 33, m)
    row_ptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    col = rng.integers(0, k, row_ptr[-1]).astype(np.int32)
    val = np.ones(col.size, np.float32)               # products without rounding: the oracle's are not fused with its sums
    B = rng.standard_normal((k, n)).astype(np.float32)
    got = _n(ops.spmm(*_csr_t((row_ptr, col, val), gpu), _t(B, gpu), m))
    assert np.array_equal(got, oracle.spmm(row_ptr, col, val, B, m))


@pytest.mark.parametrize("k", [257, 1 << 19, (1 << 19) + 1, 1 << 20, (1 << 20) + 1])
def test_kept_plans_whatever_bits_their_order_takes(gpu, k):
    """a plan that is kept orders its pieces by eight, eleven or sixteen bits of their first column, by the number of columns, a call
    without one by eight up to 2^20: the same bits, whatever the order, with rows of one piece and of several"""
    from graphnn_amd import ops
    import torch
    m, n = 32768, 33
    gen = torch.Generator(device=gpu).manual_seed(k)
    deg = torch.randint(4, 60, (m,), device=gpu, generator=gen)
    row_ptr = torch.cat([torch.zeros(1, dtype=torch.int64, device=gpu), deg.cumsum(0)]).int()
    col = torch.randint(0, k, (int(row_ptr[-1]),), device=gpu, generator=gen).int()
    val, B = torch.randn(col.numel(), device=gpu, generator=gen), torch.randn(k, n, device=gpu, generator=gen)
    want = ops.spmm(row_ptr, col, val, B, m)
    with ops.CsrPlan(row_ptr, col, val, m, k) as plan:
        assert torch.equal(plan.spmm(B), want)


@pytest.mark.parametrize("m", [33_790, 33_791, 33_792, 34_000, 2_097_153])
def test_spmm_pieces_at_the_edges_of_their_scans(gpu, m):
    """rows whose counts fill segments of 1,024 to the last element, pass one by an element, and pass the 2,048 segments that a
    workgroup adds up by itself; small whole numbers, whose sums are exact in any order, against the sums of 64-bit integers"""
    from graphnn_amd import ops
    import torch
    n = 32
    gen = torch.Generator(device=gpu).manual_seed(m)
    deg = torch.randint(0, 29, (m,), device=gpu, generator=gen)
    deg[m // 2] = 5_000
    deg[-1] = 40
    row_ptr = torch.cat([torch.zeros(1, dtype=torch.int64, device=gpu), deg.cumsum(0)])
    col = torch.randint(0, m, (int(row_ptr[-1]),), device=gpu, generator=gen)
    assert col.numel() >= 12 * m
    B = torch.randint(-8, 9, (m, n), device=gpu, generator=gen)
    got = ops.spmm(row_ptr.int(), col.int(), torch.ones(col.numel(), device=gpu), B.float(), m)
    for at in range(0, n, 8):                                 # differences of running sums, a few columns at a time
        run = torch.cat([torch.zeros(1, 8, dtype=torch.int64, device=gpu), B[:, at:at + 8][col].cumsum(0)])
        assert torch.equal(got[:, at:at + 8].long(), run[row_ptr[1:]] - run[row_ptr[:-1]]), at
        del run


@pytest.mark.parametrize("n", [64, 128, 36, 9, 4, 300, 1100])
def test_spmm_with_a_plan_has_the_bits_of_the_call_without(gpu, oracle, n):
    """gnnhip_csr_plan_create + gnnhip_spmm_csr_planned_f32 on the power-law matrix of the test above: the plan sizes its
    arrays for the pieces the matrix really has, the product runs the same kernels in the same order, so every bit
    equals gnnhip_spmm_csr_f32's; also with beta, on a second and third call, at another width through the same plan
    (its partial sums grow), and against the oracle"""
    from graphnn_amd import ops
    rng = np.random.default_rng(900 + n)
    a = synth.rmat_csr(0x5EED0005, 16, 16 << 16)
    N = 1 << 16
    v = (rng.random(a[1].size) * 0.2 - 0.05).astype(np.float32)
    csr = (a[0], a[1], v)
    csr_d = _csr_t(csr, gpu)
    B = rng.standard_normal((N, n)).astype(np.float32)
    C0 = rng.standard_normal((N, n)).astype(np.float32)
    B_d = _t(B, gpu)
    plain = _n(ops.spmm(*csr_d, B_d, N))
    plain2 = _n(ops.spmm(*csr_d, B_d, N, alpha=-0.5, beta=1.5, out=_t(C0, gpu)))
    with ops.CsrPlan(*csr_d, N, N) as plan:
        first_bytes = plan.bytes()
        got = _n(plan.spmm(B_d))
        assert np.array_equal(got, plain)
        assert np.array_equal(_n(plan.spmm(B_d, alpha=-0.5, beta=1.5, out=_t(C0, gpu))), plain2)
        assert np.array_equal(_n(plan.spmm(B_d)), plain)
        # another width through the same plan, then the first one again
        B8 = rng.standard_normal((N, 72)).astype(np.float32)
        assert np.array_equal(_n(plan.spmm(_t(B8, gpu))), _n(ops.spmm(*csr_d, _t(B8, gpu), N)))
        assert np.array_equal(_n(plan.spmm(B_d)), plain)
        assert plan.bytes() >= first_bytes
        # the plan's arrays: 8 bytes per entry, 8 per row, 16 per piece and less than that again for the balanced pass
        pieces = int(np.ceil(np.diff(a[0]) / 32).sum())
        assert first_bytes <= 8 * a[1].size + 8 * (N + 1) + 16 * pieces + (1 << 16)
    want, w64 = _spmm_want(oracle, *csr, B, N)
    assert_parity("spmm", got, want, w64)


@pytest.mark.parametrize("slot", [1, 3, 4])
def test_spmm_falls_back_with_the_output_untouched_when_scratch_cannot_be_had(gpu, oracle, slot):
    """The column-ordered route takes all its scratch (slot 3: plan, 4: partial sums, 1: the balanced pass over rows of
    many pieces) before its first launch.  When one of the requests fails (injected through the library's test hook, as
    a full device would fail it), the product falls back to the row-group route with C as the caller left it: with
    beta != 0, beta is applied exactly once."""
    import ctypes
    from graphnn_amd import ops
    from graphnn_amd._lib import load_library
    rng = np.random.default_rng(950 + slot)
    a = synth.rmat_csr(0x5EED0005, 16, 16 << 16)
    N, n = 1 << 16, 64
    v = (rng.random(a[1].size) * 0.2 - 0.05).astype(np.float32)
    csr = (a[0], a[1], v)
    csr_d = _csr_t(csr, gpu)
    B = rng.standard_normal((N, n)).astype(np.float32)
    C0 = rng.standard_normal((N, n)).astype(np.float32)
    normal = _n(ops.spmm(*csr_d, _t(B, gpu), N, alpha=-0.5, beta=1.5, out=_t(C0, gpu)))
    lib = load_library()
    lib.gnnhip_test_fail_next_scratch.argtypes = [ctypes.c_int]
    lib.gnnhip_test_fail_next_scratch.restype = None
    lib.gnnhip_test_fail_next_scratch(slot)
    try:
        got = _n(ops.spmm(*csr_d, _t(B, gpu), N, alpha=-0.5, beta=1.5, out=_t(C0, gpu)))
    finally:
        lib.gnnhip_test_fail_next_scratch(-1)
    want, w64 = _spmm_want(oracle, *csr, B, N, alpha=-0.5, beta=1.5, C=C0)
    assert_parity("spmm after a failed scratch request", got, want, w64)
    # the fallback is another route (its sums run in another order), so the bits differ from the normal call's somewhere,
    # while a beta applied twice would be off by |0.75 C0| ~ 1 everywhere
    assert not np.array_equal(got, normal)
    assert np.abs(got - normal).max() < 1e-3
    # and the next call takes the normal route again
    assert np.array_equal(_n(ops.spmm(*csr_d, _t(B, gpu), N, alpha=-0.5, beta=1.5, out=_t(C0, gpu))), normal)


def test_plan_of_matrices_that_take_the_other_routes(gpu, oracle):
    """a plan is made for any matrix: small ones, sparse ones and ones with a few very long rows keep the row-group
    route (with the balanced pass over long rows, whose plan is then kept); no rows, no entries"""
    from graphnn_amd import ops
    rng = np.random.default_rng(901)
    cases = [_random_csr(rng, 517, 389, 4000), _random_csr(rng, 40_000, 40_000, 90_000),
             _hub_matrix(rng, 36_000, 36_000, [(0, 12000), (5, 300), (17, 65), (20000, 3000), (35_999, 1000)]),
             (np.zeros(8, np.int32), np.zeros(0, np.int32), np.zeros(0, np.float32))]
    for rp, ci, v in cases:
        m = rp.size - 1
        k = 389 if m == 517 else max(m, 1)
        B = rng.standard_normal((k, 64)).astype(np.float32)
        csr_d = _csr_t((rp, ci, v), gpu)
        with ops.CsrPlan(*csr_d, m, k) as plan:
            for _ in range(2):
                got = _n(plan.spmm(_t(B, gpu)))
                assert np.array_equal(got, _n(ops.spmm(*csr_d, _t(B, gpu), m)))
            if m == k and m > 7:
                h = np.maximum(B, 0)
                W = (rng.standard_normal((64, 64)) * 0.1).astype(np.float32)
                lv = _n(plan.level(_t(h, gpu), _t(W, gpu), _t(B, gpu)))
                assert np.array_equal(lv, _n(ops.s2v_level(*csr_d, _t(h, gpu), _t(W, gpu), _t(B, gpu))))
        assert_parity("spmm", got, *_spmm_want(oracle, rp, ci, v, B, m))
    with ops.CsrPlan(*_csr_t((np.zeros(1, np.int32), np.zeros(0, np.int32), np.zeros(0, np.float32)), gpu), 0, 5) as plan:
        assert plan.spmm(_t(np.ones((5, 3), np.float32), gpu)).shape == (0, 3)


def test_plans_give_their_memory_back(gpu):
    """plans of a power-law matrix made, used at two widths (the partial sums and the balanced pass grow with the width) and
    destroyed, several times over: the pool holds what it held before, and the bytes a plan reports are what it took"""
    import ctypes
    from graphnn_amd import ops
    lib = ops._lib()
    rng = np.random.default_rng(77)
    a = synth.rmat_csr(0x5EED0005, 16, 16 << 16)
    N = 1 << 16
    csr_d = _csr_t((a[0], a[1], np.ones(a[1].size, np.float32)), gpu)
    B32, B128 = _t(rng.standard_normal((N, 32)).astype(np.float32), gpu), _t(rng.standard_normal((N, 128)).astype(np.float32), gpu)
    def in_use():
        z = [ctypes.c_size_t() for _ in range(3)]
        ops.check(lib.gnnhip_pool_stats(*[ctypes.byref(c) for c in z]))
        return z[0].value
    import torch
    torch.cuda.synchronize()
    before = in_use()
    first = None
    for _ in range(4):
        with ops.CsrPlan(*csr_d, N, N) as plan:
            held = plan.bytes()
            assert in_use() - before == held
            got = plan.spmm(B32)
            got128 = plan.spmm(B128)
            assert plan.bytes() > held and in_use() - before == plan.bytes()
            if first is None:
                first = (got.clone(), got128.clone())
            assert torch.equal(got, first[0]) and torch.equal(got128, first[1])
        assert in_use() == before


@pytest.mark.parametrize("C", [16, 32, 64, 128])
def test_level_on_a_power_law_graph_leaves_no_trace_of_the_output_buffer(gpu, oracle, C):
    """the two-launch level on the R-MAT matrix (a third of its rows empty): the product skips the rows without
    entries and the contraction takes them as zero without reading them, so whatever the output buffer held before
    the call (NaN here) must not show; with and without a plan, the same bits; against the oracle"""
    import torch
    from graphnn_amd import ops
    rng = np.random.default_rng(910 + C)
    a = synth.rmat_csr(0x5EED0005, 16, 16 << 16)
    N = 1 << 16
    v = (rng.random(a[1].size) * 0.1).astype(np.float32)
    csr = (a[0], a[1], v)
    csr_d = _csr_t(csr, gpu)
    h_in = np.maximum(rng.standard_normal((N, C)), 0).astype(np.float32)
    W = (rng.standard_normal((C, C)) * 0.1).astype(np.float32)
    msg = rng.standard_normal((N, C)).astype(np.float32)
    out = torch.full((N, C), float("nan"), device=gpu)
    got = _n(ops.s2v_level(*csr_d, _t(h_in, gpu), _t(W, gpu), _t(msg, gpu), out=out))
    assert not np.isnan(got).any()
    empty = np.diff(a[0]) == 0
    assert empty.sum() > 1000 and np.array_equal(got[empty], np.maximum(msg[empty], 0))
    with ops.CsrPlan(*csr_d, N, N) as plan:
        out2 = torch.full((N, C), float("nan"), device=gpu)
        assert np.array_equal(_n(plan.level(_t(h_in, gpu), _t(W, gpu), _t(msg, gpu), out=out2)), got)
        assert np.array_equal(_n(plan.level(_t(h_in, gpu), _t(W, gpu), _t(msg, gpu), out=out2)), got)
        if C == 64:
            # the whole forward with the caller's plan: the bits of the forward that plans for itself
            K, H, Q, L, B = 6, 16, 3, 2, 64
            w = synth.make_weights(synth.Stream(910), K, C, H, Q)
            X = np.zeros((N, K), np.float32); X[np.arange(N), rng.integers(0, K, N)] = 1.0
            s_d = _csr_t(synth.contiguous_subgraph_csr(N, B), gpu)
            dev_w = [_t(x, gpu) for x in (w.W_n2l, w.W_conv * 0.1, w.W_h1, w.W_h2)]
            f1 = ops.s2v_forward(csr_d, s_d, _t(X, gpu), *dev_w, L)
            f2 = ops.s2v_forward_planned(plan, s_d, _t(X, gpu), *dev_w, L)
            for key in ("msg", "pool", "hidden", "logits", "probs", "pred"):
                assert np.array_equal(_n(getattr(f1, key)), _n(getattr(f2, key))), key
            assert np.array_equal(_n(f1.h_final), _n(f2.h_final))
    want, w64 = _level_want(oracle, *csr, h_in, W, msg, None)
    short = np.diff(a[0]) <= 256
    assert_parity("level, rows of up to 256 entries", got[short], want[short], w64[short])
    assert_condition("level, all rows", got, w64(), w64.cond())


@pytest.mark.parametrize("C", [16, 64])
def test_level_hub_rows_balanced_pass(gpu, oracle, C):
    from graphnn_amd import ops
    rng = np.random.default_rng(600 + C)
    N = 36000
    csr = _hub_matrix(rng, N, N, [(0, 12000), (1, 4100), (7, 300), (15, 257), (16, 2048), (17, 65), (18, 64), (19, 49), (20000, 3000), (N - 1, 1000)])
    h_in = np.maximum(rng.standard_normal((N, C)), 0).astype(np.float32)
    W = (rng.standard_normal((C, C)) * 0.1).astype(np.float32)
    msg = rng.standard_normal((N, C)).astype(np.float32)
    want, w64 = _level_want(oracle, *csr, h_in, W, msg, None)
    got = _n(ops.s2v_level(*_csr_t(csr, gpu), _t(h_in, gpu), _t(W, gpu), _t(msg, gpu)))
    assert_parity("level", got, want, w64)
    assert np.array_equal(got, _n(ops.s2v_level(*_csr_t(csr, gpu), _t(h_in, gpu), _t(W, gpu), _t(msg, gpu))))


@pytest.mark.parametrize("C,L", [(64, 2), (16, 1), (32, 3), (128, 2), (256, 1)])
def test_forward_first_level_reads_msg_with_long_rows(gpu, oracle, C, L):
    """sparse graph of 36,000 nodes with a few very long rows: the forward does not store h0, the first level
    and the balanced pass over the long rows read ReLU(msg) from msg; every level's embedding, the pooled
    features and the logits against the reference path"""
    from graphnn_amd import ops
    rng = np.random.default_rng(700 + C)
    N, K, H, Q, B = 36000, 9, 16, 3, 36
    a = _hub_matrix(rng, N, N, [(0, 9000), (1, 2100), (7, 300), (16, 2048), (17, 65), (18, 64), (19, 49), (20000, 3000), (N - 1, 1000)])
    s = synth.contiguous_subgraph_csr(N, B)
    lab = rng.integers(0, K, N)
    X = np.zeros((N, K), np.float32); X[np.arange(N), lab] = 1.0
    X += (rng.standard_normal(X.shape) * 0.05).astype(np.float32)              # msg with both signs everywhere
    w = synth.make_weights(synth.Stream(700 + C), K, C, H, Q)
    w.W_conv = (w.W_conv * 0.02).astype(np.float32)                              # rows of thousands of entries: keep the levels bounded
    want = _forward_want(oracle, a, s, X, w, L)
    bufs = ops.s2v_forward(_csr_t(a, gpu), _csr_t(s, gpu), _t(X, gpu), _t(w.W_n2l, gpu), _t(w.W_conv, gpu),
                           _t(w.W_h1, gpu), _t(w.W_h2, gpu), L)
    # the reference path adds a row of thousands of entries sequentially in fp32 and is itself about 1e-4 from
    # the exact sum there: where the device misses the oracle by more than 1e-4, the float64 model decides
    # (the device must be no further from it than the oracle is)
    _assert_forward_parity({k: _n(getattr(bufs, k)) for k in ("msg", "h_final", "pool", "hidden", "logits", "probs")}, want, L)


def test_rmat_forward_with_jagged_softmax(gpu, oracle):
    """the skewed-degree workload at reduced scale: R-MAT (a=0.57, b=c=0.19), 16 entries per row on
    average, subgraphs = contiguous ranges of 1024 nodes; three levels, node score = h . w, jagged
    softmax of the scores per subgraph, sum-pool of h per subgraph"""
    from graphnn_amd import ops
    scale, ef, C, K, L = 16, 16, 64, 12, 3
    N = 1 << scale
    a = synth.rmat_csr(0x5EED0005, scale, ef << scale)
    assert int(np.diff(a[0]).max()) > 2048                      # hubs well past every in-kernel threshold
    nsub = N // 1024
    s = synth.contiguous_subgraph_csr(N, nsub)
    st = synth.Stream(0x5EED0005)
    lab = (st.child(100).uniform(N) * K).astype(np.int64) % K
    X = np.zeros((N, K), np.float32); X[np.arange(N), lab] = 1.0
    w = synth.make_weights(st, K, C, 8, 2)
    wsc = (np.random.default_rng(5).standard_normal((C, 1)) * 0.1).astype(np.float32)
    # oracle, and the same network in float64 (unit edge weights and hub rows make the embeddings grow
    # by orders of magnitude per level, so after three levels two correct fp32 summation orders differ
    # by more than 1e-4 in places: each level is checked from identical inputs, the end of the chain
    # against the float64 model)
    import scipy.sparse as sp
    A64 = sp.csr_matrix((a[2].astype(np.float64), a[1], a[0]), shape=(N, N))
    msg = oracle.gemm(X, w.W_n2l)
    h = np.maximum(msg, 0)
    h64 = h.astype(np.float64)
    a_d, s_d = _csr_t(a, gpu), _csr_t(s, gpu)
    msg_d, h_d = ops.s2v_input(_t(X, gpu), _t(w.W_n2l, gpu))
    assert max_rel(_n(msg_d), msg) < PARITY_TOL
    Wc_d = _t(w.W_conv, gpu)
    short = np.diff(a[0]) <= 256
    W64, msg64 = w.W_conv.astype(np.float64), msg.astype(np.float64)
    for _ in range(L):
        # one level from identical inputs.  The reference path adds a row's entries one after the other
        # in fp32, which on a row of 13,000 entries is itself 1e-4 away from the exact sum; the device
        # sums such rows in chunks and lands closer to it.  So: every row against the float64 result,
        # and the rows of up to 256 entries against the reference path as everywhere else.
        h_next = oracle.level(*a, h, w.W_conv, msg, None)
        exact = np.maximum((A64 @ h.astype(np.float64)) @ W64 + msg64, 0).astype(np.float32)
        got = _n(ops.s2v_level(*a_d, _t(h, gpu), Wc_d, msg_d))
        assert max_rel(got, exact) < PARITY_TOL
        assert_parity("level, short rows", got[short], h_next[short], exact[short])
        h_d = ops.s2v_level(*a_d, h_d, Wc_d, msg_d)                                                # chained
        h = h_next
        h64 = np.maximum((A64 @ h64) @ W64 + msg64, 0)
    err_ref = max_rel(h, h64.astype(np.float32))
    err_gpu = max_rel(_n(h_d), h64.astype(np.float32))
    assert err_gpu <= max(err_ref, PARITY_TOL), (err_gpu, err_ref)
    score = oracle.gemm(h, wsc)
    lens = np.full(nsub, 1024, np.int32)
    soft = oracle.jagged_softmax(score.copy(), lens)
    pool = oracle.spmm(*s, h, nsub)
    # reductions from identical inputs
    h_same = _t(h, gpu)
    score_d = ops.gemm(h_same, _t(wsc, gpu))
    assert max_rel(_n(score_d), score) < PARITY_TOL
    soft_d = ops.jagged_softmax(_t(score, gpu), _t(lens, gpu))
    pool_d = ops.spmm(*s_d, h_same, nsub)
    assert max_rel(_n(pool_d), pool) < PARITY_TOL
    got_soft = _n(soft_d).reshape(nsub, 1024)
    assert np.allclose(got_soft.sum(axis=1), 1.0, atol=1e-5)
    assert np.abs(got_soft - soft.reshape(nsub, 1024)).max() < 1e-4


@pytest.mark.parametrize("C", [16, 32, 64])
def test_level_dense_graph_two_launch_route(gpu, oracle, C):
    """a large graph with 14 entries per row takes the SpMM-then-contraction route; same result as the
    reference path"""
    from graphnn_amd import ops
    rng = np.random.default_rng(77 + C)
    N, deg = 40000, 14
    rp, ci, v = synth.erdos_renyi_csr(77, N, N * deg)
    v = (rng.random(v.size) * 0.2).astype(np.float32)
    h_in = np.maximum(rng.standard_normal((N, C)), 0).astype(np.float32)
    W = (rng.standard_normal((C, C)) * 0.1).astype(np.float32)
    msg = rng.standard_normal((N, C)).astype(np.float32)
    bias = rng.standard_normal(C).astype(np.float32)
    want, w64 = _level_want(oracle, rp, ci, v, h_in, W, msg, bias)
    got = _n(ops.s2v_level(_t(rp, gpu), _t(ci, gpu), _t(v, gpu), _t(h_in, gpu), _t(W, gpu), _t(msg, gpu), _t(bias, gpu)))
    assert_parity("level", got, want, w64)


def test_edge_embedding_step_with_edge_based_operands(gpu, oracle):
    """one loopy-BP style update on edge states, built from the edge-to-edge, node-to-edge and edge-to-node
    operands (src/nn/msg_pass.cpp:72-152) and the same SpMM / GEMM / element-wise entry points"""
    from graphnn_amd import ops
    batch = synth.molecule_batch(321, 40, 6, 2)
    N, E, K, C = batch.num_nodes, batch.num_edges, 6, 32
    rng = np.random.default_rng(4)
    n2e = batching.node2edge_csr(batch.edge_x)
    e2e = batching.edge2edge_csr(N, batch.edge_x, batch.edge_y)
    e2n = batching.edge2node_csr(N, batch.edge_y, average=True)
    X = batch.one_hot()
    W1 = (rng.standard_normal((K, C)) * 0.3).astype(np.float32)
    W2 = (rng.standard_normal((C, C)) * 0.3).astype(np.float32)
    m0 = np.maximum(rng.standard_normal((E, C)), 0).astype(np.float32)
    # reference path
    inp = oracle.spmm(*n2e, oracle.gemm(X, W1), E)
    m1 = np.maximum(oracle.gemm(oracle.spmm(*e2e, m0, E), W2) + inp, 0)
    node = oracle.spmm(*e2n, m1, N)
    # device
    inp_d = ops.spmm(*_csr_t(n2e, gpu), ops.gemm(_t(X, gpu), _t(W1, gpu)), E)
    lin_d = ops.gemm(ops.spmm(*_csr_t(e2e, gpu), _t(m0, gpu), E), _t(W2, gpu))
    m1_d = ops.relu(ops.add(lin_d, inp_d))
    node_d = ops.spmm(*_csr_t(e2n, gpu), m1_d, N)
    assert max_rel(_n(m1_d), m1) < PARITY_TOL
    assert max_rel(_n(node_d), node) < PARITY_TOL
    # the same update through the fused level entry: A = edge-to-edge, h = edge states, msg = inp
    fused = ops.s2v_level(*_csr_t(e2e, gpu), _t(m0, gpu), _t(W2, gpu), inp_d)
    assert max_rel(_n(fused), m1) < PARITY_TOL


# ------------------------------------------------------------------ device-side CSR construction
@pytest.mark.parametrize("average", [False, True])
def test_device_csr_group_matches_host_builders(gpu, oracle, average):
    from graphnn_amd import ops
    rng = np.random.default_rng(808)
    # random multigraph with empty rows, a hub, keys needing two radix passes
    N, E = 3000, 20000
    ex = rng.integers(0, N, E).astype(np.int32); ey = rng.integers(0, N, E).astype(np.int32)
    ey[1000:4000] = 77                                            # one row of 3000+ entries
    ey[ey == 5] = 6                                               # an empty row
    want = oracle.csr_node2node(N, ex, ey, average)
    got = ops.csr_group(N, _t(ey, gpu), _t(ex, gpu), average)
    for g, w in zip(got, want):
        assert np.array_equal(_n(g), w)
    # the same from an interleaved (x, y) array, as GraphStruct::edge_list stores it
    pairs = _t(np.stack([ex, ey], axis=1).reshape(-1), gpu)
    got = ops.csr_group(N, pairs[1:], pairs, average, key_stride=2, payload_stride=2, n=E)
    for g, w in zip(got, want):
        assert np.array_equal(_n(g), w)
    # edge-to-node: payload = edge index
    got = ops.csr_group(N, _t(ey, gpu), _t(np.arange(E, dtype=np.int32), gpu), average)
    for g, w in zip(got, oracle.csr_edge2node(N, ey, average)):
        assert np.array_equal(_n(g), w)
    # subgraph operand with shuffled AddNode order
    B = 37
    perm = rng.permutation(N)
    sid = np.sort(rng.integers(0, B, N))[perm].astype(np.int32); nid = np.arange(N, dtype=np.int32)[perm]
    got = ops.csr_group(B, _t(sid, gpu), _t(nid, gpu), average)
    for g, w in zip(got, oracle.csr_subgraph(B, sid, nid, average)):
        assert np.array_equal(_n(g), w)


def test_device_csr_group_edge_cases_and_scale(gpu, oracle):
    import torch
    from graphnn_amd import ops
    # no pairs; one row; one pair
    rp, ci, v = ops.csr_group(5, torch.zeros(0, dtype=torch.int32, device=gpu), torch.zeros(0, dtype=torch.int32, device=gpu))
    assert np.array_equal(_n(rp), np.zeros(6, np.int32)) and ci.numel() == 0
    rp, ci, v = ops.csr_group(1, _t(np.zeros(700, np.int32), gpu), _t(np.arange(700, dtype=np.int32)[::-1].copy(), gpu), True)
    assert np.array_equal(_n(rp), [0, 700]) and np.array_equal(_n(ci), np.arange(700)[::-1]) and np.all(_n(v) == np.float32(1.0 / 700))
    rp, ci, v = ops.csr_group(9, _t(np.array([8], np.int32), gpu), _t(np.array([3], np.int32), gpu))
    assert np.array_equal(_n(rp), [0] * 9 + [1]) and _n(ci)[0] == 3
    # three radix passes (2^17 rows) and several tiles per pass, against the numpy stable sort
    rng = np.random.default_rng(9)
    rows, n = (1 << 17) + 3, 700_001
    key = rng.integers(0, rows, n).astype(np.int32); pay = rng.integers(0, 1 << 30, n).astype(np.int32)
    rp, ci, v = ops.csr_group(rows, _t(key, gpu), _t(pay, gpu))
    order = np.argsort(key, kind="stable")
    assert np.array_equal(_n(ci), pay[order])
    want_rp = np.zeros(rows + 1, np.int64); np.cumsum(np.bincount(key, minlength=rows), out=want_rp[1:])
    assert np.array_equal(_n(rp), want_rp)
    # a configuration-2 batch: identical to what the host builds
    batch, w, cfg = synth.make_config(2)
    want = batching.node2node_csr(batch.num_nodes, batch.edge_x, batch.edge_y)
    got = ops.csr_group(batch.num_nodes, _t(batch.edge_y, gpu), _t(batch.edge_x, gpu))
    for g, w_ in zip(got, want):
        assert np.array_equal(_n(g), w_)


def _stable_group(rows, key, pay, average=False):
    order = np.argsort(key, kind="stable")
    rp = np.zeros(rows + 1, np.int64); np.cumsum(np.bincount(key, minlength=rows), out=rp[1:])
    lens = np.diff(rp)
    val = (1.0 / np.repeat(lens, lens).astype(np.float64)).astype(np.float32) if average else np.ones(len(key), np.float32)
    return rp, pay[order], val


@pytest.mark.parametrize("case", ["lengths_around_eight", "hub_in_a_window", "one_row_of_all", "largest", "past_the_largest", "many_rows", "ascending",
                                  "ascending_but_one", "long_rows_only", "two_pairs"])
def test_device_csr_group_of_a_small_batch_in_one_launch(gpu, case):
    """up to 65,536 pairs are grouped in one launch of up to 64 workgroups, each with a run of the rows (4 bytes per row of
    the run and 2.35 per pair have to fit 160 KB of LDS): rows of up to 8 entries ordered by a thread, longer rows by a
    wavefront with a bitmap (one bitmap only in the largest cases), keys that already ascend copied through;
    bit-identical to the stable sort"""
    from graphnn_amd import ops
    rng = np.random.default_rng(sum(map(ord, case)))
    if case == "lengths_around_eight":
        lens = rng.integers(0, 19, 3000); lens[:40] = [0, 7, 8, 9, 10, 1, 64, 65] * 5
        rows = len(lens); key = rng.permutation(np.repeat(np.arange(rows), lens)).astype(np.int32)
    elif case == "hub_in_a_window":
        # a batch as GetBatch lays it out: a row's pairs lie close together; one graph has a hub of 900 pairs
        rows = 9000; key = np.sort(rng.integers(0, rows, 30000)).astype(np.int32)
        for i in range(0, 30000, 50):
            key[i:i + 50] = rng.permutation(key[i:i + 50])
        key[12000:12900] = key[12000]
    elif case == "one_row_of_all":
        rows = 5; key = np.full(65536, 3, np.int32)
        key[::1000] = 1                                           # not ascending, so that the row is really ordered
    elif case == "largest":
        rows = 32768; key = rng.integers(0, rows, 65536).astype(np.int32)
    elif case == "past_the_largest":
        rows = 45000; key = rng.integers(0, rows, 65536).astype(np.int32)
    elif case == "many_rows":
        rows = 21000; key = rng.integers(0, rows, 30000).astype(np.int32); key[5000:5400] = 20999
    elif case == "ascending":
        rows = 700; key = np.sort(rng.integers(0, rows, 40000)).astype(np.int32)
    elif case == "ascending_but_one":
        rows = 700; key = np.sort(rng.integers(0, rows, 40000)).astype(np.int32); key[-1] = 0
    elif case == "long_rows_only":
        rows = 256; key = rng.integers(0, rows, 7450).astype(np.int32)
    else:
        rows = 3; key = np.array([2, 0], np.int32)
    n = len(key)
    pay = rng.integers(0, 1 << 30, n).astype(np.int32)
    for average in (False, True):
        rp, ci, v = ops.csr_group(rows, _t(key, gpu), _t(pay, gpu), average)
        want = _stable_group(rows, key, pay, average)
        assert np.array_equal(_n(rp), want[0]), case
        assert np.array_equal(_n(ci), want[1]), case
        assert np.array_equal(_n(v), want[2]), case
    # strided pairs, and a second call on the same stream (the counters and bitmaps start clean every time)
    pairs = _t(np.stack([pay, key], axis=1).reshape(-1), gpu)
    rp, ci, v = ops.csr_group(rows, pairs[1:], pairs, False, key_stride=2, payload_stride=2, n=n)
    want = _stable_group(rows, key, pay)
    assert np.array_equal(_n(rp), want[0]) and np.array_equal(_n(ci), want[1])


@pytest.mark.parametrize("n", [3, 4, 255, 4095, 4096, 4097, 8191, 8193, 16_383, 16_385, 33_001, 65_535])
@pytest.mark.parametrize("rows", [1, 63, 65, 4_097, 50_000, 300_000])
def test_device_csr_group_at_the_edges_of_its_workgroups(gpu, n, rows):
    """the one-launch grouping where its workgroups (512 or 1,024 lanes, 8 rows or more each) and its batches of keys end:
    keys that start at any int (read four at a time only where they are aligned), keys out of range (clamped to the first and
    the last row), runs of equal keys across lanes and wavefronts, rows of 8, 9, 64 and 65 entries; the bits of the stable sort"""
    from graphnn_amd import ops
    rng = np.random.default_rng(n + rows)
    key = rng.integers(0, rows, n)
    key[n // 3:n // 3 + 300] = rng.integers(0, rows)
    at = 0
    for length in (8, 9, 64, 65):                             # rows of about these lengths, scattered
        if n > 1000:
            key[rng.permutation(n)[:length]] = rows * (at + 1) // 5
        at += 1
    for order in ("any", "ascending"):
        if order == "ascending":
            key = np.sort(key)
        raw = key.copy()
        raw[key == 0] -= rng.integers(0, 3, int((key == 0).sum()))
        raw[key == rows - 1] += rng.integers(0, 3, int((key == rows - 1).sum()))
        if rows == 1:
            raw = key + rng.integers(-2, 3, n)
        pay = rng.integers(0, 1 << 30, n).astype(np.int32)
        want = _stable_group(rows, key, pay)
        for shift in (0, 1):
            key_d = _t(np.concatenate([np.zeros(shift, np.int32), raw.astype(np.int32)]), gpu)[shift:]
            got = ops.csr_group(rows, key_d, _t(pay, gpu))
            for g, w in zip(got, want):
                assert np.array_equal(_n(g), w), (order, shift)


@pytest.mark.parametrize("n", [3, 63, 64, 65, 511, 513, 8191, 8193, 16_385, 65_535])
@pytest.mark.parametrize("rows", [1, 65, 4_097, 50_000])
def test_device_csr_group_of_strided_keys(gpu, n, rows):
    """keys two and three ints apart, where a lane takes one pair at a time: runs of equal keys that end with a wavefront and inside
    it, keys out of range, ascending ones; alone, and with the other member of the pair as the key of a second grouping, of the same
    stride and of its own (one of the two strided); the bits of the stable sort"""
    from graphnn_amd import ops
    rng = np.random.default_rng(n + rows)
    key, other = rng.integers(0, rows, n), rng.integers(0, rows, n)
    key[n // 3:n // 3 + 300] = rng.integers(0, rows)
    for order in ("any", "ascending"):
        if order == "ascending":
            key = np.sort(key)
        raw = key.copy()
        raw[key == 0] -= rng.integers(0, 3, int((key == 0).sum()))
        raw[key == rows - 1] += rng.integers(0, 3, int((key == rows - 1).sum()))
        want, turned = _stable_group(rows, key, raw), _stable_group(rows, key, other)
        for stride in (2, 3):
            held = np.full((n, stride), -7, np.int32)
            held[:, stride - 1] = raw
            held_d = _t(held.reshape(-1), gpu)[stride - 1:]
            for g, w in zip(ops.csr_group(rows, held_d, held_d, False, stride, stride, n), want):
                assert np.array_equal(_n(g), w), (order, stride)
            back = _stable_group(rows, other, raw)
            for x_stride in (1, stride):
                x = np.full((n, x_stride), -7, np.int32)
                x[:, 0] = other
                got = ops.csr_group_both(rows, _t(x.reshape(-1), gpu), held_d, x_stride, stride, n)
                for g, w in zip(got[0] + got[1], turned + back):
                    assert np.array_equal(_n(g), w), (order, stride, x_stride)


@pytest.mark.parametrize("rows", [1, 7, 8, 9, 16, 17, 511, 512, 513])
@pytest.mark.parametrize("per", [3, 9, 30, 64, 100])
def test_device_csr_group_of_few_rows(gpu, rows, per):
    """runs of eight rows and more per workgroup: one run and several, the last one short, rows that a thread, a wavefront by rank and
    a bitmap put in order, in one run; the bits of the stable sort"""
    from graphnn_amd import ops
    rng = np.random.default_rng(rows + per)
    lens = rng.integers(0, 2 * per + 1, rows)
    lens[rows // 2] = 64
    key = rng.permutation(np.repeat(np.arange(rows), lens)).astype(np.int32)
    pay = rng.integers(0, 1 << 30, key.size).astype(np.int32)
    for g, w in zip(ops.csr_group(rows, _t(key, gpu), _t(pay, gpu)), _stable_group(rows, key, pay)):
        assert np.array_equal(_n(g), w)


@pytest.mark.parametrize("n", [65_536, 67_584, 67_585, 8_192 * 2_048, 8_192 * 2_048 + 1])
def test_device_csr_group_at_the_edges_of_its_scans(gpu, n):
    """the sort's counters in whole segments of 1,024 and in a part of one more, and either side of the 2,048 segments that a
    workgroup adds up by itself; the bits of the stable sort"""
    from graphnn_amd import ops
    import torch
    rows = 50_000
    gen = torch.Generator(device=gpu).manual_seed(n)
    key = torch.randint(0, rows, (n,), dtype=torch.int32, device=gpu, generator=gen)
    pay = torch.randint(0, 1 << 30, (n,), dtype=torch.int32, device=gpu, generator=gen)
    row_ptr, col_idx, val = ops.csr_group(rows, key, pay)
    kept, order = torch.sort(key, stable=True)
    ends = torch.searchsorted(kept, torch.arange(rows + 1, dtype=torch.int32, device=gpu))
    assert torch.equal(row_ptr.long(), ends)
    assert torch.equal(col_idx, pay[order])
    assert bool((val == 1).all())


@pytest.mark.parametrize("C,mean", [(5, 24), (48, 24), (100, 24), (100, 63), (100, 70), (128, 64), (200, 24), (200, 63), (256, 70)])
def test_readout_has_the_same_bits_whatever_the_batch(gpu, C, mean):
    """a workgroup per graph with three rows in flight and with eight: the first graphs of a batch past the line between them, as
    batches on either side of it"""
    from graphnn_amd import ops
    import torch
    rng = np.random.default_rng(C + mean)
    most, H, Q = 1_700, 33, 3
    sizes = rng.integers(0, 2 * mean + 1, most)
    rp = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    col = np.concatenate([rp[i] + rng.permutation(n) for i, n in enumerate(sizes)]).astype(np.int32)
    val = rng.random(col.size).astype(np.float32)
    gen = torch.Generator(device=gpu).manual_seed(C)
    h = torch.randn(col.size, C, device=gpu, generator=gen)
    W1 = torch.randn(C, H, device=gpu, generator=gen)
    W2 = torch.randn(H, Q, device=gpu, generator=gen)
    want = ops.s2v_readout(_t(rp, gpu), _t(col, gpu), _t(val, gpu), h, W1, W2, most)
    pool64 = np.add.reduceat(np.concatenate([h.cpu().numpy().astype(np.float64)[col] * val[:, None], np.zeros((1, C))]), rp[:-1])
    pool64[sizes == 0] = 0
    # a sum of n products: n + 1 roundings of terms whose magnitudes add up to no more than the absolute sum
    mag = np.add.reduceat(np.concatenate([np.abs(h.cpu().numpy().astype(np.float64)[col]) * val[:, None], np.zeros((1, C))]), rp[:-1])
    assert np.all(np.abs(_n(want[0]) - pool64) <= (sizes[:, None] + 1) * 2.0 ** -24 * mag + 2.0 ** -126)
    for B in (1, 37, 1_024, 1_025, 1_536, 1_537):
        e = int(rp[B])
        got = ops.s2v_readout(_t(rp[:B + 1].copy(), gpu), _t(col[:e].copy(), gpu), _t(val[:e].copy(), gpu), h[:e], W1, W2, B)
        for g, w in zip(got, want):
            assert torch.equal(g, w[:B]), B


@pytest.mark.parametrize("B", [40, 600])
@pytest.mark.parametrize("H,Q", [(1, 1), (3, 2), (32, 4), (64, 5), (17, 8), (33, 9), (5, 16), (64, 17), (130, 3)])
def test_one_launch_readout_of_any_number_of_classes(gpu, B, H, Q):
    """the end of the one-launch forward, graph by graph (sixteen, eight or four lanes add up a logit up to 4, 8, 16 classes, a wavefront
    beyond) and packed (a lane per class), graphs of 1 to 60 nodes so that the pooling ends inside its runs of rows: pooled row, hidden
    layer and logits within the roundings of their sums of float64, from the operands the device itself formed; probabilities
    likewise; classes that tie take the first, a NaN in class 0 is kept, one elsewhere never wins"""
    import torch
    from graphnn_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(B + 100 * H + Q)
    C, K, L = 32, 5, 2
    sizes = (torch.arange(B, device=gpu) * 7) % 60 + 1
    off = torch.zeros(B + 1, dtype=torch.int32, device=gpu)
    off[1:] = torch.cumsum(sizes, 0)
    N = int(off[-1])
    graph = torch.repeat_interleave(torch.arange(B, device=gpu), sizes)
    ring = torch.arange(N, device=gpu) + 1
    ring = torch.where(ring == off[1:][graph], off[:-1][graph].long(), ring).int()
    A = (torch.arange(N + 1, device=gpu).int(), ring, torch.ones(N, device=gpu))
    normal = lambda *shape: torch.randn(*shape, generator=gen, device=gpu)
    S = (off, torch.arange(N, device=gpu).int(), torch.rand(N, generator=gen, device=gpu) + 0.5)
    X, Wn, Wc, W1, W2 = normal(N, K), normal(K, C), normal(C, C) * 0.2, normal(C, H), normal(H, Q)
    bufs = ops.s2v_forward_batched(A, S, X, Wn, Wc, W1, W2, L, int(sizes.max()))
    h, w = bufs.h_final.double(), S[2].double()
    zero = torch.zeros(B, C, dtype=torch.float64, device=gpu)
    pool = zero.index_add(0, graph, h * w[:, None])
    eps = 2.0 ** -24
    def close(got, want, terms, roundings):
        assert bool(((got.double() - want).abs() <= roundings * eps * terms).all())
    close(bufs.pool, pool, zero.index_add(0, graph, (h * w[:, None]).abs()), 64)
    hidden = (bufs.pool.double() @ W1.double()).clamp(min=0)
    close(bufs.hidden, hidden, bufs.pool.double().abs() @ W1.double().abs(), C + 4)
    close(bufs.logits, bufs.hidden.double() @ W2.double(), bufs.hidden.double().abs() @ W2.double().abs(), H + 4)
    # e^x of a rounded x is off by the rounding of x, and what lies below the smallest normal float may be zero
    want = torch.softmax(bufs.logits.double(), 1)
    close(bufs.probs, want, want + 2.0 ** -126 / eps, 2 * Q + 16 + 4 * float(bufs.logits.abs().max()))
    assert torch.equal(bufs.pred.long(), bufs.logits.argmax(1))
    for bad in {0, Q - 1}:
        W2_bad = torch.zeros(H, Q, device=gpu)
        tied = ops.s2v_forward_batched(A, S, X, Wn, Wc, W1, W2_bad, L, int(sizes.max()))
        assert not bool(tied.pred.any()) and bool((tied.probs == tied.probs[:, :1]).all())
        W2_bad[:, bad] = float("nan")
        got = ops.s2v_forward_batched(A, S, X, Wn, Wc, W1, W2_bad, L, int(sizes.max()))
        assert bool(torch.isnan(got.logits[:, bad]).all()) and not bool(got.pred.any())


@pytest.mark.parametrize("B", [512, 513, 575, 577, 640, 4096, 4161, 70_001])
@pytest.mark.parametrize("sizes", ["ones", "tiny", "full", "mixed"])
def test_packed_batches_of_any_number_of_segments(gpu, B, sizes):
    """the bins of a packed batch: segments of 64 graphs, the last one short; a whole segment in one bin (graphs of one node), bins of
    one graph each (128 nodes), a bin per few graphs and graphs without nodes: node outputs with the bits of the forward that
    takes graph by graph (it keeps all levels), graph outputs of the right graphs within the roundings of their sums of float64"""
    import torch
    from graphnn_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(B)
    n = {"ones": torch.ones(B, device=gpu).long(), "tiny": torch.randint(1, 4, (B,), generator=gen, device=gpu),
         "full": torch.full((B,), 128, device=gpu), "mixed": torch.randint(0, 12, (B,), generator=gen, device=gpu)}[sizes]
    n[640:] = n[640:].clamp(max=12)
    if sizes == "mixed":
        n[::97] = 100
    C, K, H, Q, L = 16, 4, 8, 3, 2
    off = torch.zeros(B + 1, dtype=torch.int32, device=gpu)
    off[1:] = torch.cumsum(n, 0)
    N = int(off[-1])
    graph = torch.repeat_interleave(torch.arange(B, device=gpu), n)
    ring = torch.arange(N, device=gpu) + 1
    ring = torch.where(ring == off[1:][graph], off[:-1][graph].long(), ring).int()
    A = (torch.arange(N + 1, device=gpu).int(), ring, torch.ones(N, device=gpu))
    S = (off, torch.arange(N, device=gpu).int(), torch.ones(N, device=gpu))
    normal = lambda *shape: torch.randn(*shape, generator=gen, device=gpu)
    X, Wn, Wc, W1, W2 = normal(N, K), normal(K, C), normal(C, C) * 0.3, normal(C, H), normal(H, Q)
    got = ops.s2v_forward_batched(A, S, X, Wn, Wc, W1, W2, L, int(n.max()))
    one_by_one, h = ops.s2v_forward_batched_train(A, S, X, Wn, Wc, W1, W2, L, int(n.max()))
    assert torch.equal(got.msg, one_by_one.msg) and torch.equal(got.h_final, h[L])
    zero = torch.zeros(B, C, dtype=torch.float64, device=gpu)
    pool = zero.index_add(0, graph, h[L].double())               # embeddings are not negative: the sum is that of its terms' magnitudes
    assert bool(((got.pool.double() - pool).abs() <= 130 * 2.0 ** -24 * pool).all())
    want = (got.pool.double() @ W1.double()).clamp(min=0)
    assert bool(((got.hidden.double() - want).abs() <= (C + 4) * 2.0 ** -24 * (got.pool.double() @ W1.double().abs())).all())
    want = got.hidden.double() @ W2.double()
    assert bool(((got.logits.double() - want).abs() <= (H + 4) * 2.0 ** -24 * (got.hidden.double() @ W2.double().abs())).all())
    assert int(got.status.item()) == 0


@pytest.mark.parametrize("average", [False, True])
def test_device_csr_of_consecutive_rows(gpu, oracle, average):
    """the pooling operand of a batch whose nodes were added subgraph after subgraph, from the subgraph offsets alone:
    bit-identical to what the host builder makes of the (subgraph, node) records, graphs without nodes and a graph of
    3,000 nodes among them"""
    from graphnn_amd import ops
    rng = np.random.default_rng(5)
    sizes = rng.integers(0, 60, 700); sizes[[0, 1, 350, 699]] = 0; sizes[77] = 3000
    sid = np.repeat(np.arange(sizes.size), sizes).astype(np.int32)
    nid = np.arange(sid.size, dtype=np.int32)
    want = oracle.csr_subgraph(sizes.size, sid, nid, average)
    ci, v = ops.csr_consecutive_rows(_t(want[0], gpu), average)
    assert np.array_equal(_n(ci), want[1]) and np.array_equal(_n(v), want[2])
    # the same from the offsets in host memory, in one launch; and a batch without nodes
    got = ops.csr_consecutive_rows_host(want[0], gpu, average)
    for g, w_ in zip(got, want):
        assert np.array_equal(_n(g), w_)
    rp, ci, v = ops.csr_consecutive_rows_host(np.zeros(6, np.int32), gpu, average)
    assert not _n(rp).any() and ci.numel() == 0


@pytest.mark.parametrize("rows,n", [(7450, 16382), (300, 40_000), (50_000, 70_000), (9, 1), (5, 0)])
def test_device_csr_group_both_ways(gpu, rows, n):
    """an edge list grouped by head and by tail at once (a matrix and its transpose, entries in edge order): the one-launch
    grouping with two jobs, the radix route past it; both equal the stable sorts, and the two are transposes of each other"""
    import scipy.sparse as sp
    from graphnn_amd import ops
    rng = np.random.default_rng(rows + n)
    x = rng.integers(0, rows, n).astype(np.int32); y = rng.integers(0, rows, n).astype(np.int32)
    if n > 1000:
        y[100:700] = 3                                            # a long row on one side, short ones on the other
    pairs = _t(np.stack([x, y], axis=1).reshape(-1), gpu)
    if n:
        a, at = ops.csr_group_both(rows, pairs, pairs[1:], 2, 2, n=n)
    else:
        empty = _t(np.zeros(0, np.int32), gpu)
        a, at = ops.csr_group_both(rows, empty, empty)
    for got, want in ((a, _stable_group(rows, y, x)), (at, _stable_group(rows, x, y))):
        for g, w in zip(got, want):
            assert np.array_equal(_n(g), w)
    if n:
        A = sp.csr_matrix((_n(a[2]), _n(a[1]), _n(a[0])), shape=(rows, rows))
        AT = sp.csr_matrix((_n(at[2]), _n(at[1]), _n(at[0])), shape=(rows, rows))
        assert (A.T != AT).nnz == 0


@pytest.mark.parametrize("m,k,nnz", [(411, 233, 3000), (5000, 7000, 120_000), (3, 70_000, 32_768), (1, 1, 1), (900, 20_000, 65_536),
                                     (32_768, 32_768, 65_537)])
def test_device_csr_transpose(gpu, oracle, m, k, nnz):
    """one tile, many tiles, few long rows of A, a single entry, the largest one-launch case, one entry past it"""
    from graphnn_amd import ops
    rng = np.random.default_rng(10 + m)
    csr = _random_csr(rng, m, k, nnz)
    t_rp, t_ci, t_v = ops.csr_transpose(*_csr_t(csr, gpu), m, k)
    import scipy.sparse as sp
    A = sp.csr_matrix((csr[2], csr[1], csr[0]), shape=(m, k))
    # entry order inside a row of A^T: by row of A, then by position in that row (stable)
    rows_of = np.repeat(np.arange(m), np.diff(csr[0]))
    order = np.argsort(csr[1], kind="stable")
    assert np.array_equal(_n(t_ci), rows_of[order]) and np.array_equal(_n(t_v), csr[2][order])
    want_rp = np.zeros(k + 1, np.int64); np.cumsum(np.bincount(csr[1], minlength=k), out=want_rp[1:])
    assert np.array_equal(_n(t_rp), want_rp)
    # A^T B through the forward SpMM equals the transposed product of the reference path
    B = rng.standard_normal((m, 24)).astype(np.float32)
    got = _n(ops.spmm(t_rp, t_ci, t_v, _t(B, gpu), k))
    assert max_rel(got, oracle.spmm_T(*csr, B, m, k)) < PARITY_TOL
    assert np.allclose(got, (A.T @ B), atol=1e-4)


def test_uploads_in_one_batch(gpu):
    """gnnhip_memcpy_h2d_batch: the three arrays of a CSR matrix in one launch, an empty piece among them; pieces that
    are not whole words, or too many, or too large for the staging buffer, go one by one; the host buffers are free
    as soon as the call returns"""
    import ctypes
    import torch
    from graphnn_amd import ops
    rng = np.random.default_rng(12)
    def send(arrays):
        outs = [torch.full((max(a.nbytes, 1),), 255, dtype=torch.uint8, device=gpu) for a in arrays]
        n = len(arrays)
        P = ctypes.c_void_p * n
        ops.check(ops._lib().gnnhip_memcpy_h2d_batch(n, P(*[o.data_ptr() for o in outs]), P(*[a.ctypes.data for a in arrays]),
                                                     (ctypes.c_size_t * n)(*[a.nbytes for a in arrays]), None))
        for a in arrays:
            a[...] = 0                                            # the call has read them
        return [o.cpu().numpy()[:max(len(w), 0)] for o, w in zip(outs, wants)]
    cases = [[rng.integers(0, 1 << 30, 16382).astype(np.int32), rng.standard_normal(16382).astype(np.float32),
              rng.integers(0, 9, 7451).astype(np.int32)],
             [np.zeros(0, np.int32), rng.integers(0, 99, 5).astype(np.int32)],
             [rng.integers(0, 255, 7).astype(np.uint8), rng.integers(0, 99, 33).astype(np.int32)],
             [rng.integers(0, 99, 3).astype(np.int32) for _ in range(11)],
             [rng.integers(0, 99, 700_000).astype(np.int32), rng.integers(0, 99, 4).astype(np.int32)]]
    for arrays in cases:
        wants = [a.tobytes() for a in arrays]
        got = send(arrays)
        for g, w in zip(got, wants):
            assert g.tobytes()[:len(w)] == w


def test_scalars_read_behind_one_wait(gpu):
    """gnnhip_memcpy_d2h_batch: the first elements of several device tensors (a loss, an accuracy, an int), queued
    behind the kernels that wrote them, arrive together; pieces too large for the pinned landing buffer are read one by one"""
    import ctypes
    import torch
    from graphnn_amd import ops
    a = torch.full((1,), 2.5, device=gpu); b = torch.full((3,), -7.0, device=gpu); c = torch.full((1,), 41, dtype=torch.int32, device=gpu)
    a.mul_(2.0)                                                   # still in the queue when the read is issued
    got = ops.read_scalars([a, b, c])
    assert got[0] == 5.0 and got[1] == -7.0 and got[2] == 41
    assert ops.read_scalars([]) == []
    big = torch.arange(3000, dtype=torch.float32, device=gpu)     # 12 KB: past the landing buffer
    host = np.zeros(3000, np.float32); one = np.zeros(1, np.float32)
    P = ctypes.c_void_p * 2
    ops.check(ops._lib().gnnhip_memcpy_d2h_batch(2, P(host.ctypes.data, one.ctypes.data), P(big.data_ptr(), a.data_ptr()),
                                                 (ctypes.c_size_t * 2)(12000, 4), None))
    assert np.array_equal(host, np.arange(3000, dtype=np.float32)) and one[0] == 5.0


@pytest.mark.parametrize("shape,density", [((7450, 38), "one_hot"), ((7450, 38), 0.5), ((100, 7), "one_hot"), ((300_000, 64), "one_hot"),
                                           ((16384,), 0.0), ((16385,), 1.0 / 17), ((40_000, 3), 1.0 / 15), ((5_000_000,), 0.001)])
def test_sparse_upload_rebuilds_the_same_bits(gpu, shape, density):
    """host-to-device copy that sends only the non-zero 32-bit words when they are at most one in sixteen (and the
    plain copy otherwise, or below 16,384 words): the device buffer has the host's bits either way: negative zero
    and denormals are non-zero words, the last word and the words around tile boundaries are hit, the destination
    held other data before, and the host array may be overwritten at once"""
    import torch
    from graphnn_amd import ops
    rng = np.random.default_rng(abs(hash((shape, str(density)))) % (2 ** 32))
    n = int(np.prod(shape))
    if density == "one_hot":
        a = np.zeros(shape, np.float32)
        a[np.arange(shape[0]), rng.integers(0, shape[1], shape[0])] = 1.0
    else:
        a = np.where(rng.random(n) < density, rng.standard_normal(n), 0.0).astype(np.float32).reshape(shape)
    flat = a.reshape(-1)
    if n > 20_000 and density != 0.5:
        flat[-1] = -0.0                                       # a non-zero word, at the very end
        flat[4095] = np.float32(1e-42); flat[4096] = 3.0       # a denormal and the first word of the second tile
    want = flat.view(np.uint32).copy()
    out = torch.full(shape, 7.0, dtype=torch.float32, device=gpu)
    ops.upload_sparse32(a, out=out)
    flat[:] = 5.0                                             # the host buffer has been read by now
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy().reshape(-1).view(np.uint32), want)
    # int32 data takes the same route
    b = np.where(rng.random(50_000) < 0.02, rng.integers(-9, 9, 50_000), 0).astype(np.int32)
    assert np.array_equal(ops.upload_sparse32(b).cpu().numpy(), b)


def test_bindings_make_tensors_as_torch_does(gpu):
    """device, type and layout of torch.empty's tensors, in inference mode and under deterministic algorithms (which fill
    them) too"""
    import torch
    from graphnn_amd import ops
    def check(t, like):
        assert t.device == like.device and t.dtype == like.dtype and t.shape == like.shape and t.stride() == like.stride()
        assert t.requires_grad == like.requires_grad and t.is_inference() == like.is_inference()
    where = torch.empty(1, device=gpu)
    with torch.inference_mode():
        check(ops._empty(where, "f", 3, 5), torch.empty(3, 5, device=gpu))
    i, f = ops._empty(where, "iF", 7, 2, 3)
    check(i, torch.empty(7, dtype=torch.int32, device=gpu))
    check(f, torch.empty(2, 3, device=gpu))
    for sizes in ((-2,), (3, -1)):
        with pytest.raises(RuntimeError):
            ops._empty(where, "f", *sizes)
    torch.use_deterministic_algorithms(True)
    try:
        assert bool(torch.isnan(ops._empty(where, "f", 1000)).all())
    finally:
        torch.use_deterministic_algorithms(False)


def _small_graphs(gpu, sizes, mean_entries, gen, unit=False):
    """(A, S, N): graphs of the given sizes, entries drawn inside their graph, rows of 0 to 2 mean_entries entries (one number, or one per graph)"""
    import torch
    n = torch.as_tensor(sizes, device=gpu)
    off = torch.zeros(n.numel() + 1, dtype=torch.long, device=gpu)
    off[1:] = torch.cumsum(n, 0)
    N = int(off[-1])
    graph = torch.repeat_interleave(torch.arange(n.numel(), device=gpu), n)
    mean = torch.as_tensor(mean_entries, device=gpu).expand(n.numel())[graph]
    deg = (torch.rand(N, generator=gen, device=gpu) * (2 * mean + 1)).long().minimum(2 * mean)
    rp = torch.zeros(N + 1, dtype=torch.int32, device=gpu)
    rp[1:] = torch.cumsum(deg, 0)
    row = torch.repeat_interleave(torch.arange(N, device=gpu), deg)
    ci = off[graph[row]] + (torch.rand(row.numel(), generator=gen, device=gpu) * n[graph[row]]).long().minimum(n[graph[row]] - 1)
    val = torch.ones(row.numel(), device=gpu) if unit else torch.rand(row.numel(), generator=gen, device=gpu) / mean[row].clamp(min=1)
    S = (off.int(), torch.arange(N, device=gpu).int(), torch.rand(N, generator=gen, device=gpu) + 0.5)
    return (rp, ci.int(), val), S, N


def _forward_one_by_one(A, S, X, Wn, Wc, W1, W2, L):
    """the same forward from the stages' own entries (a level at a time)"""
    from graphnn_amd import ops
    msg, h = ops.s2v_input(X, Wn)
    for _ in range(L):
        h = ops.s2v_level(*A, h, Wc, msg)
    return (msg, h) + tuple(ops.s2v_readout(*S, h, W1, W2, S[0].numel() - 1))


def _fill(bufs):
    for name in ("msg", "h_a", "h_b", "pool", "hidden", "logits", "probs"):
        getattr(bufs, name).fill_(float("nan"))


def _in_one_launch(bufs):
    """which route a forward of two levels and more took over buffers that _fill had filled: level by level both embeddings are written whole, in one
    launch the other one holds the bins, which end before its last row"""
    import torch
    other = bufs.h_b if bufs.which.value == 0 else bufs.h_a
    return bool(torch.isnan(other[-1]).all())


def _tried(gpu, sizes, mean_entries, K, C, L):
    """whether a forward over a batch of these sizes, with nothing against it, runs in one launch: the host then tries its likes"""
    import torch
    from graphnn_amd import ops
    A, S, N = _small_graphs(gpu, sizes, mean_entries, torch.Generator(device=gpu).manual_seed(1))
    bufs = ops.ForwardBuffers(N, S[0].numel() - 1, C, 8, 3, gpu)
    _fill(bufs)
    zero = lambda *shape: torch.zeros(*shape, device=gpu)
    ops.s2v_forward(A, S, zero(N, K), zero(K, C), zero(C, C), zero(C, 8), zero(8, 3), L, bufs=bufs)
    return _in_one_launch(bufs)


def _check_forward(gpu, A, S, N, K, C, L, gen, exact, taken):
    """taken: whether the levels run in one launch"""
    import torch
    from graphnn_amd import ops
    H, Q = 8, 3
    B = S[0].numel() - 1
    normal = lambda *shape: torch.randn(*shape, generator=gen, device=gpu)
    X = torch.zeros(N, K, device=gpu)
    X[torch.arange(N, device=gpu), torch.randint(0, K, (N,), generator=gen, device=gpu)] = 1.0
    w = (normal(K, C), normal(C, C) * (0.8 / C ** 0.5), normal(C, H), normal(H, Q))
    bufs = ops.ForwardBuffers(N, B, C, H, Q, gpu)
    _fill(bufs)
    ops.s2v_forward(A, S, X, *w, L, bufs=bufs)
    assert _in_one_launch(bufs) == taken
    got = (bufs.msg, bufs.h_final, bufs.pool, bufs.hidden, bufs.logits, bufs.probs, bufs.pred)
    want = _forward_one_by_one(A, S, X, *w, L)
    assert torch.equal(got[0], want[0])                      # one-hot features: rows of the weights
    for g, e in list(zip(got, want))[:exact]:
        assert torch.equal(g, e)
    # float64 and the sum of the terms' magnitudes, level by level: every level adds the rounding of its two sums
    rp, ci, val = A
    row = torch.repeat_interleave(torch.arange(N, device=gpu), (rp[1:] - rp[:-1]).long())
    msg = X.double() @ w[0].double()
    h, terms = msg.clamp(min=0), msg.abs()
    for _ in range(L):
        zero = torch.zeros(N, C, dtype=torch.float64, device=gpu)
        h = (zero.index_add(0, row, h[ci.long()] * val.double()[:, None]) @ w[1].double() + msg).clamp(min=0)
        terms = zero.index_add(0, row, terms[ci.long()] * val.double()[:, None].abs()) @ w[1].double().abs() + msg.abs()
    longest = int((rp[1:] - rp[:-1]).max()) if row.numel() else 0
    bound = L * (longest + C + 2) * 2.0 ** -24
    assert bool(((got[1].double() - h).abs() <= bound * terms).all())
    pool = torch.zeros(B, C, dtype=torch.float64, device=gpu)
    graph = torch.repeat_interleave(torch.arange(B, device=gpu), (S[0][1:] - S[0][:-1]).long(), output_size=S[1].numel())
    pool.index_add_(0, graph, got[1].double()[S[1].long()] * S[2].double()[:, None])
    # no negative terms; a rounding for each and for its weight, of the longest row of S (one that names a whole batch is summed in pieces)
    members = min(int((S[0][1:] - S[0][:-1]).max()), 4200)
    assert bool(((got[2].double() - pool).abs() <= (members + 2) * 2.0 ** -24 * pool.abs() + 1e-30).all())
    # the readout from its own pooled rows: a rounding per term, and expf's two units in the last place, the sum and the quotient
    hidden, hidden_terms = got[2].double() @ w[2].double(), got[2].double().abs() @ w[2].double().abs()
    assert bool(((got[3].double() - hidden.clamp(min=0)).abs() <= (C + 1) * 2.0 ** -24 * hidden_terms).all())
    logits, logit_terms = got[3].double() @ w[3].double(), got[3].double().abs() @ w[3].double().abs()
    assert bool(((got[4].double() - logits).abs() <= (H + 1) * 2.0 ** -24 * logit_terms).all())
    assert bool(((got[5].double() - torch.softmax(got[4].double(), 1)).abs() <= 16 * 2.0 ** -24).all())
    assert torch.equal(got[6].long(), got[4].argmax(1))


def _enough(n, C, L, pooled=False):
    """the sizes repeated until the batch is one that the forward tries to take in one launch, with pooled: that adds up the pooled rows too"""
    least = (12e6 if C in (16, 64) else 6e6 if 32 < C < 64 else 4e6) * (1 if np.sum(n) <= 64 * np.size(n) else 6 if L == 2 else 3)
    need = max(32769, least / ((L - 1) * C), (12e6 if C > 64 else 4e6) / C if pooled else 0)
    return np.tile(np.asarray(n, np.int64), int(np.ceil(need / np.sum(n))))


@pytest.mark.parametrize("C", [16, 17, 31, 32, 33, 48, 50, 64, 65, 80, 95, 100, 112])
@pytest.mark.parametrize("sizes", ["molecules", "ones", "full", "with_empty", "dense"])
def test_forward_over_a_large_batch_of_small_graphs(gpu, C, sizes):
    """batches whose levels run in one launch: bins of one graph of 128 nodes, of 64 graphs of one node, graphs without nodes, bins of
    more entries than are kept in LDS among others, a last tile of one row; feature columns around the steps of the input stage, hidden sizes around
    the padded ones.  The embeddings of hidden 16 and 32 have the bits of the stages called one by one; all else is held to the rounding of
    fp32 sums"""
    import torch
    gen = torch.Generator(device=gpu).manual_seed(C)
    for K, L, seed in ((2, 2, 0), (3, 4, 1), (17, 3, 2), (33, 4, 3), (64, 2, 4)):
        rng = np.random.default_rng(100 * C + seed)
        n = {"molecules": rng.integers(10, 111, 1100), "ones": np.ones(33_001, np.int64), "full": np.tile([128, 10], 300),
             "with_empty": np.where(rng.random(4000) < 0.3, 0, rng.integers(1, 40, 4000)),
             "dense": np.where(np.arange(800) % 4, rng.integers(5, 30, 800), rng.integers(120, 129, 800))}[sizes]
        n = _enough(n, C, L, pooled=seed % 2 == 0)
        if sizes == "with_empty":
            n[640:768] = 0                                       # two segments without nodes
            n[-1] = 0
        A, S, N = _small_graphs(gpu, n, np.where(n >= 120, 11, 2) if sizes == "dense" else 2, gen)
        _check_forward(gpu, A, S, N, K, C, L, gen, 2 if C in (16, 32) else 0, True)


@pytest.mark.parametrize("C", [16, 30, 32, 46, 64, 77, 100])
@pytest.mark.parametrize("kind", ["crossing", "crossing_dense", "large_graph", "uncovered", "offset", "overlapping", "long_row", "foreign_member",
                                  "permuted_members"])
def test_forward_over_a_batch_that_is_none(gpu, C, kind):
    """what the one launch must refuse on the device: one entry that leaves its bin (kept in LDS, or read from memory), a graph of 129
    nodes, rows of S that leave out nodes, begin past node 0, name nodes twice or those of other graphs: embeddings and pooled rows
    have the bits of the stages called one by one"""
    import torch
    gen = torch.Generator(device=gpu).manual_seed(7)
    rng = np.random.default_rng(C)
    dense = kind == "crossing_dense"                             # every fourth graph, the last one among them, fills a bin with more entries than are kept in LDS
    n = np.where(np.arange(800) % 4 < 3, rng.integers(5, 30, 800), rng.integers(120, 129, 800)) if dense else rng.permutation(rng.integers(10, 111, 1100))
    n = _enough(n, C, 3, pooled=kind in ("foreign_member", "permuted_members", "large_graph"))
    assert _tried(gpu, n, np.where(n >= 120, 11, 2) if dense else 2, 9, C, 3)
    if kind == "large_graph":
        n[700] = 129
    A, S, N = _small_graphs(gpu, n, np.where(n >= 120, 11, 2) if dense else 2, gen)
    rp, ci, val = A
    if kind.startswith("crossing"):
        first = int(torch.nonzero(rp[1:] > rp[:-1])[-1])         # the last row with entries points to node 0
        ci[int(rp[first])] = 0
        assert not dense or int(rp[-1] - rp[int(S[0][-2])]) > 1024
    elif kind == "long_row":                                     # a row of 5,000 entries that stay inside: the one launch takes it
        first = int(S[0][3])
        width = int(S[0][4]) - first
        at = int(rp[first])
        extra = first + torch.arange(5000, device=gpu) % width
        ci = torch.cat([ci[:at], extra.int(), ci[at:]])
        val = torch.cat([val[:at], torch.rand(5000, generator=gen, device=gpu) / 5000, val[at:]])
        rp = rp.clone(); rp[first + 1:] += 5000
    elif kind == "uncovered":
        S = (S[0][:-1].contiguous(), S[1], S[2])                 # the last graph's nodes belong to none
        S = (S[0], S[1][:int(S[0][-1])].contiguous(), S[2][:int(S[0][-1])].contiguous())
    elif kind == "offset":
        S = (S[0][1:] - S[0][1], S[1][int(S[0][1]):].contiguous(), S[2][int(S[0][1]):].contiguous())
    elif kind == "overlapping":                                  # the last row names all nodes of the batch again
        S = (torch.cat([S[0], S[0][-1:] + N]), torch.cat([S[1], S[1]]), torch.cat([S[2], S[2]]))
    elif kind == "foreign_member":                               # the last graph's row names a node of the first in its own one's place
        S[1][-1] = 0
    elif kind == "permuted_members":                             # the nodes of a row in another order, one of them twice: the one launch takes it
        first, last = int(S[0][5]), int(S[0][6])
        S[1][first:last] = S[1][first:last].flip(0)
        S[1][first] = first + 1
    taken = kind in ("long_row", "permuted_members")
    # hidden 16 has its pooled rows from the readout, whoever the members are
    _check_forward(gpu, (rp, ci, val), S, N, 9, C, 3, gen, 0 if taken else 3, taken or (kind == "foreign_member" and C == 16))


@pytest.mark.parametrize("C", [16, 31, 64, 90])
@pytest.mark.parametrize("planned", [False, True])
def test_forward_over_a_batch_that_is_none_with_long_rows(gpu, C, planned):
    """refused on the device (its last graph has 129 nodes) with rows of 64, 65, 2,048, 2,049 and 9,000 entries, which the launch of the bins counts for
    all levels, or a kept plan: embeddings and pooled rows have the bits of the stages called one by one, twice over, and after a batch of
    as many entries without long rows on the same arrays"""
    import torch
    from graphnn_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(C)
    n = _enough(np.random.default_rng(C).integers(10, 111, 1100), C, 4, pooled=True)
    assert _tried(gpu, n, 3, 9, C, 4)
    n[-1] = 129
    (rp, ci, val), S, N = _small_graphs(gpu, n, 3, gen)
    deg = (rp[1:] - rp[:-1]).long()
    long = [64, 65, 2048, 2049, 9000]
    rows = torch.arange(5, device=gpu) * (N // 5) + 7
    deg[rows] = torch.tensor(long, device=gpu)
    rp2 = torch.zeros_like(rp)
    rp2[1:] = torch.cumsum(deg, 0)
    E = int(rp2[-1])
    graph = torch.repeat_interleave(torch.arange(n.size, device=gpu), torch.from_numpy(n).to(gpu))
    row = torch.repeat_interleave(torch.arange(N, device=gpu), deg)
    off, size = S[0].long()[graph[row]], torch.from_numpy(n).to(gpu)[graph[row]]
    ci = (off + (torch.rand(E, generator=gen, device=gpu) * size).long().minimum(size - 1)).int()
    val = torch.rand(E, generator=gen, device=gpu) / deg[row]
    H, Q, K, B = 8, 3, 9, n.size
    normal = lambda *shape: torch.randn(*shape, generator=gen, device=gpu)
    X = torch.zeros(N, K, device=gpu)
    X[torch.arange(N, device=gpu), torch.randint(0, K, (N,), generator=gen, device=gpu)] = 1.0
    w = (normal(K, C), normal(C, C) * (0.8 / C ** 0.5), normal(C, H), normal(H, Q))
    even = torch.linspace(0, E, N + 1, device=gpu).round().int()               # the same entries in rows of as many each
    for shape in (rp2, rp2, even, rp2):
        A = (shape, ci, val)
        want = _forward_one_by_one(A, S, X, *w, 4)
        bufs = ops.ForwardBuffers(N, B, C, H, Q, gpu)
        _fill(bufs)
        if planned:
            with ops.CsrPlan(*A, N, N) as plan:
                ops.s2v_forward_planned(plan, S, X, *w, 4, bufs=bufs)
        else:
            ops.s2v_forward(A, S, X, *w, 4, bufs=bufs)
        assert not _in_one_launch(bufs)
        for got, e in zip((bufs.msg, bufs.h_final, bufs.pool), want):
            assert torch.equal(got, e)


@pytest.mark.parametrize("C", [32, 64, 100])
def test_large_batch_forward_replays_from_a_captured_graph(gpu, C):
    """captured over a batch that the levels' one launch takes, then replayed over matrices changed in place: whether it takes them is
    found out by every replay, and each has the bits of the same eager call"""
    import torch
    from graphnn_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(C)
    A, S, N = _small_graphs(gpu, _enough(np.random.default_rng(C).integers(10, 111, 1100), C, 3, pooled=True), 2, gen)
    B, K, H, Q = S[0].numel() - 1, 9, 8, 3
    normal = lambda *shape: torch.randn(*shape, generator=gen, device=gpu)
    X, w = normal(N, K), (normal(K, C), normal(C, C) * (0.8 / C ** 0.5), normal(C, H), normal(H, Q))
    bufs, eager = ops.ForwardBuffers(N, B, C, H, Q, gpu), ops.ForwardBuffers(N, B, C, H, Q, gpu)
    last = int(A[0][int(torch.nonzero(A[0][1:] > A[0][:-1])[-1])])          # an entry of the last graph
    inside = int(A[1][last])
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        ops.s2v_forward(A, S, X, *w, 3, bufs=bufs)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        ops.s2v_forward(A, S, X, *w, 3, bufs=bufs)
    torch.cuda.synchronize()
    outputs = lambda b: [getattr(b, n) for n in ("msg", "h_final", "pool", "hidden", "logits", "probs", "pred")]
    for column in (inside, 0, 0, inside, inside):
        A[1][last] = column
        _fill(eager)
        for t in outputs(bufs):
            t.fill_(-1)
        ops.s2v_forward(A, S, X, *w, 3, bufs=eager)
        torch.cuda.synchronize()
        assert _in_one_launch(eager) == (column == inside)
        graph.replay()
        torch.cuda.synchronize()
        for got, want in zip(outputs(bufs), outputs(eager)):
            assert torch.equal(got, want), column


@pytest.mark.parametrize("C,K,N", [(20, 3, 20_000), (31, 40, 13_000), (40, 7, 24_000), (63, 64, 17_000), (65, 2, 8_000), (66, 64, 6_000), (96, 16, 4_097),
                                   (96, 17, 16_400), (97, 16, 6_000), (100, 17, 12_000), (112, 5, 16_384), (112, 1, 16_385)])
@pytest.mark.parametrize("crossing", [False, True])
def test_forward_over_a_few_small_graphs_of_odd_hidden_sizes(gpu, C, K, N, crossing):
    """some thousand nodes, which the levels' one launch takes where it is their input stage too, and its refusal, behind which the
    level-by-level launches have tiles of 16 or 32 rows"""
    import torch
    gen = torch.Generator(device=gpu).manual_seed(N)
    n = np.random.default_rng(C).integers(1, 60, N)
    n = n[:int(np.searchsorted(np.cumsum(n), N))]
    n = np.append(n, N - int(n.sum()))
    A, S, N = _small_graphs(gpu, n, 2, gen)
    if crossing:
        A[1][int(A[0][int(torch.nonzero(A[0][1:] > A[0][:-1])[-1])])] = 0
    _check_forward(gpu, A, S, N, K, C, 5, gen, 3 if crossing else 0, not crossing)


@pytest.mark.parametrize("C", [64, 100])
def test_forward_over_small_graphs_with_large_and_tiny_values(gpu, C):
    """products in bf16 pieces over a large batch of small graphs: rows of 2^38 and more and columns of W likewise (scaled down before they
    are split) beside ordinary ones, values near the smallest floats, infinities and NaNs in a row, which stay in the columns and graphs
    they belong to"""
    import torch
    from graphnn_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(5)
    A, S, N = _small_graphs(gpu, _enough(np.full(700, 60), C, 2), 2, gen)
    rp, ci, val = A
    row = torch.repeat_interleave(torch.arange(N, device=gpu), (rp[1:] - rp[:-1]).long())
    B, K = S[0].numel() - 1, 8
    w1, w2 = torch.zeros(C, 4, device=gpu), torch.zeros(4, 2, device=gpu)
    for scale in (1.0, 1e-36, 1e10):
        X = torch.rand(N, K, generator=gen, device=gpu)
        Wn = torch.rand(K, C, generator=gen, device=gpu) * scale
        Wc = torch.randn(C, C, generator=gen, device=gpu) * 0.1
        Wc[:, 5] *= 2.0 ** 40
        Wc[5, 5] = 0.0                                           # or the second level overflows
        X[1000:1100] *= 2.0 ** 40
        bufs = ops.ForwardBuffers(N, B, C, 4, 2, gpu)
        _fill(bufs)
        ops.s2v_forward(A, S, X, Wn, Wc, w1, w2, 2, bufs=bufs)
        assert _in_one_launch(bufs)
        h = bufs.msg.clamp(min=0)
        h1 = ops.s2v_level(*A, h, Wc, bufs.msg)
        want, zero = bufs.msg.double(), torch.zeros(N, C, dtype=torch.float64, device=gpu)
        sums = zero.index_add(0, row, h1[ci.long()].double() * val.double()[:, None])
        want = (sums @ Wc.double() + bufs.msg.double()).clamp(min=0)
        terms = sums @ Wc.double().abs() + bufs.msg.double().abs()
        # h1 comes from the FP32 matrix cores here: C + 2 roundings of its terms, which the second level multiplies
        h1_terms = zero.index_add(0, row, h[ci.long()].double() * val.double()[:, None]) @ Wc.double().abs() + bufs.msg.double().abs()
        terms = terms + zero.index_add(0, row, h1_terms[ci.long()] * val.double()[:, None]) @ Wc.double().abs()
        bad = (bufs.h_final.double() - want).abs() > 2 * (C + 8) * 2.0 ** -24 * terms + 2.0 ** -140
        assert bool(torch.isfinite(want).all()) and not bool(bad.any()), scale
    # an infinity and a NaN in the features of one node each: nothing outside their graphs changes
    X = torch.rand(N, K, generator=gen, device=gpu)
    Wn, Wc = torch.rand(K, C, generator=gen, device=gpu), torch.randn(C, C, generator=gen, device=gpu) * 0.1
    clean = ops.s2v_forward(A, S, X, Wn, Wc, w1, w2, 2).h_final.clone()
    X[60 * 10 + 3, 2], X[60 * 20 + 4, 0] = float("inf"), float("nan")
    got = ops.s2v_forward(A, S, X, Wn, Wc, w1, w2, 2).h_final
    one_by_one = _forward_one_by_one(A, S, X, Wn, Wc, w1, w2, 2)[1]
    touched = torch.zeros(N, dtype=torch.bool, device=gpu)
    touched[600:660] = touched[1200:1260] = True
    assert torch.equal(got[~touched], clean[~touched])
    assert torch.equal(torch.isnan(got), torch.isnan(one_by_one)) and torch.equal(torch.isinf(got), torch.isinf(one_by_one))


@pytest.mark.parametrize("C", [4, 7, 16, 33, 64, 65, 100, 128, 129, 200, 252, 255, 256])
def test_levels_over_few_rows_have_the_bits_of_many(gpu, C):
    """a level, its backward and the input stage over up to 4,096 rows (a workgroup per 16 rows and share of the columns) against the same
    rows inside a matrix of more (another kernel): 1 to 17 rows, the last rows where the columns are shared out and where they are not,
    rows of 0, 1, 4, 5, 8, 9, 300 and 3,000 entries, a bias, a gate and a running sum"""
    import torch
    from graphnn_amd import ops
    if C in (16, 64, 128, 256):                                # these sizes have kernels of their own: as widths of the input stage only
        return _few_rows_input(gpu, C)
    gen = torch.Generator(device=gpu).manual_seed(C)
    rand = lambda *shape: torch.randn(*shape, generator=gen, device=gpu)
    big = 4113
    W, bias = rand(C, C) * 0.2, rand(C)
    for N in (1, 16, 17, 272, 2048, 2049, 4096):
        # columns of the first N rows lie below N, so both matrices mean the same for these rows
        deg = torch.randint(0, 10, (big,), generator=gen, device=gpu)
        deg[torch.randperm(min(N, 40), generator=gen, device=gpu)[:2]] = 300
        deg[N // 2] = 3000
        rp = torch.zeros(big + 1, dtype=torch.int32, device=gpu)
        rp[1:] = torch.cumsum(deg, 0)
        ci = torch.randint(0, N, (int(rp[-1]),), generator=gen, device=gpu).int()
        val = rand(int(rp[-1]))
        x, msg, gate, acc = rand(big, C), rand(big, C), rand(big, C), rand(big, C)
        E = int(rp[N])
        few = (rp[:N + 1].contiguous(), ci[:E].contiguous(), val[:E].contiguous())
        part = lambda t: t[:N].contiguous()
        for b in (None, bias):
            assert torch.equal(ops.s2v_level(*few, part(x), W, part(msg), b), ops.s2v_level(rp, ci, val, x, W, msg, b)[:N]), (N, b is None)
        a_few, a_big = part(acc), acc.clone()
        u, g = ops.s2v_level_backward(*few, part(x), W, gate_h=part(gate), acc=a_few)
        u2, g2 = ops.s2v_level_backward(rp, ci, val, x, W, gate_h=gate, acc=a_big)
        assert torch.equal(u, u2[:N]) and torch.equal(g, g2[:N]) and torch.equal(a_few, a_big[:N]), N
        u, g = ops.s2v_level_backward(*few, part(x), W)
        assert torch.equal(g, ops.s2v_level_backward(rp, ci, val, x, W)[1][:N]), N
    _few_rows_input(gpu, C)


@pytest.mark.parametrize("C", [4, 7, 20, 33, 63])
@pytest.mark.parametrize("N", [1, 16, 17, 272, 2049])
def test_narrow_levels_over_few_rows_with_many_entries(gpu, C, N):
    """up to 64 columns, few rows of more entries on average than columns, or than sixteen, take the kernel of many rows: the last average on one side
    and the first on the other, against the same rows inside a matrix of more, a row of half of all entries among them"""
    import torch
    from graphnn_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(C)
    rand = lambda *shape: torch.randn(*shape, generator=gen, device=gpu)
    big, line = 4113, min(C, 16)
    W = rand(C, C) * 0.2
    for E in (line * N, line * N + 1, 40 * N):
        deg = torch.bincount(torch.randint(0, N, (E - E // 2,), generator=gen, device=gpu), minlength=N)
        deg[N // 2] += E // 2
        rp = torch.zeros(big + 1, dtype=torch.int32, device=gpu)
        rp[1:N + 1] = torch.cumsum(deg, 0)
        rp[N + 1:] = E + torch.cumsum(torch.randint(0, 10, (big - N,), generator=gen, device=gpu), 0)
        ci = torch.randint(0, N, (int(rp[-1]),), generator=gen, device=gpu).int()
        val, x, msg, acc = rand(int(rp[-1])), rand(big, C), rand(big, C), rand(big, C)
        few = (rp[:N + 1].contiguous(), ci[:E].contiguous(), val[:E].contiguous())
        part = lambda t: t[:N].contiguous()
        assert torch.equal(ops.s2v_level(*few, part(x), W, part(msg)), ops.s2v_level(rp, ci, val, x, W, msg)[:N]), E
        a_few, a_big = part(acc), acc.clone()
        u, g = ops.s2v_level_backward(*few, part(x), W, gate_h=part(msg), acc=a_few)
        u2, g2 = ops.s2v_level_backward(rp, ci, val, x, W, gate_h=msg, acc=a_big)
        assert torch.equal(u, u2[:N]) and torch.equal(g, g2[:N]) and torch.equal(a_few, a_big[:N]), E


def _few_rows_input(gpu, C):
    """the input stage of few rows, feature columns narrower and wider than its steps: within the rounding of its sums"""
    import torch
    from graphnn_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(C + 1)
    for N, K in ((1, 4), (15, 5), (33, 17), (300, 64), (4096, 100)):
        X, Wn = torch.randn(N, K, generator=gen, device=gpu), torch.randn(K, C, generator=gen, device=gpu)
        msg, h = ops.s2v_input(X, Wn)
        bound = (K + 2) * 2.0 ** -24 * (X.double().abs() @ Wn.double().abs())
        assert bool(((msg.double() - X.double() @ Wn.double()).abs() <= bound).all()) and torch.equal(h, msg.clamp(min=0)), (N, K)


@pytest.mark.parametrize("N", [1, 40, 2048])
def test_level_of_hidden_256_over_few_rows(gpu, oracle, N):
    """the FP32 level of hidden 256 takes the kernel of few rows: against the oracle, with a bias and without"""
    from graphnn_amd import ops
    rng = np.random.default_rng(N)
    C = 256
    csr = _random_csr(rng, N, N, 3 * N)
    h_in = np.maximum(rng.standard_normal((N, C)), 0).astype(np.float32)
    W = (rng.standard_normal((C, C)) * 0.1).astype(np.float32)
    msg, bias = rng.standard_normal((N, C)).astype(np.float32), rng.standard_normal(C).astype(np.float32)
    for b in (None, bias):
        want, w64 = _level_want(oracle, *csr, h_in, W, msg, b)
        got = _n(ops.s2v_level(*_csr_t(csr, gpu), _t(h_in, gpu), _t(W, gpu), _t(msg, gpu), None if b is None else _t(b, gpu)))
        assert_parity("level", got, want, w64)
        assert_condition("level", got, w64(), w64.cond())


@pytest.mark.parametrize("N", [1, 15, 16, 33, 1024, 1025, 2048])
def test_wide_levels_in_pieces_over_few_rows_have_the_bits_of_many(gpu, N):
    """hidden 256, up to 2,048 rows (workgroups share the columns of 16 rows) against the same rows inside a matrix of more (another
    kernel): a level of a forward and a backward level, rows of 0 to 300 entries, rows and columns of W that are scaled down before they
    are split"""
    import torch
    from graphnn_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(N)
    rand = lambda *shape: torch.randn(*shape, generator=gen, device=gpu)
    C, K, big = 256, 8, 2100
    deg = torch.randint(0, 10, (big,), generator=gen, device=gpu)
    deg[torch.arange(0, N, 97)] = torch.tensor([64, 65, 8, 300], device=gpu).repeat(6)[:len(range(0, N, 97))]
    rp = torch.zeros(big + 1, dtype=torch.int32, device=gpu)
    rp[1:] = torch.cumsum(deg, 0)
    ci = torch.randint(0, N, (int(rp[-1]),), generator=gen, device=gpu).int()
    val = rand(int(rp[-1]))
    E = int(rp[N])
    few = (rp[:N + 1].contiguous(), ci[:E].contiguous(), val[:E].contiguous())
    part = lambda t: t[:N].contiguous()
    W = rand(C, C) * 0.1
    for large in (False, True):
        X = torch.zeros(big, K, device=gpu)
        X[torch.arange(big, device=gpu), torch.randint(0, K, (big,), generator=gen, device=gpu)] = 1.0
        dz, gate, acc = rand(big, C), rand(big, C), rand(big, C)
        if large:
            W[:, 17] *= 2.0 ** 40
            W[3, :] *= 2.0 ** 39
            X[N // 3] *= 2.0 ** 39
            dz[N // 2] *= 2.0 ** 41
        a_few, a_big = part(acc), acc.clone()
        u, g = ops.s2v_level_backward(*few, part(dz), W, gate_h=part(gate), acc=a_few)
        u2, g2 = ops.s2v_level_backward(rp, ci, val, dz, W, gate_h=gate, acc=a_big)
        assert torch.equal(u, u2[:N]) and torch.equal(g, g2[:N]) and torch.equal(a_few, a_big[:N])
        assert torch.equal(ops.s2v_level_backward(*few, part(dz), W)[1], ops.s2v_level_backward(rp, ci, val, dz, W)[1][:N])
        Wn, w1, w2 = rand(K, C), torch.zeros(C, 4, device=gpu), torch.zeros(4, 2, device=gpu)
        whole = lambda n: (torch.tensor([0, n], device=gpu).int(), torch.arange(n, device=gpu).int(), torch.ones(n, device=gpu))
        for L in (1, 2):                                       # the first level reads ReLU(msg)
            got = ops.s2v_forward(few, whole(N), part(X), Wn, W, w1, w2, L)
            want = ops.s2v_forward((rp, ci, val), whole(big), X, Wn, W, w1, w2, L)
            assert torch.equal(got.h_final, want.h_final[:N]), (L, large)


@pytest.mark.parametrize("C,K", [(64, 16), (64, 13), (64, 4), (64, 1), (64, 17), (32, 16), (32, 7), (16, 8), (16, 9)])
@pytest.mark.parametrize("N", [32785, 196607, 196609])
def test_forward_of_a_power_law_graph_forms_msg_again(gpu, C, K, N):
    """levels of a graph of more than twelve entries per row and 196,608 rows or more whose contraction forms msg from up to sixteen feature columns
    instead of reading it (fewer rows, 17 columns and hidden 16 are the other side of that): features that are no one-hot rows, against the
    levels called one by one on the msg that the forward gives; rows without entries, of one piece and of many, a last tile of one row"""
    import torch
    from graphnn_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(C + K)
    L = 3
    deg = torch.randint(0, 45, (N,), generator=gen, device=gpu)
    deg[::3] = 0
    deg[torch.arange(5, N, 1000)] = 900
    rp = torch.zeros(N + 1, dtype=torch.int32, device=gpu)
    rp[1:] = torch.cumsum(deg, 0)
    E = int(rp[-1])
    assert E >= 12 * N
    ci = torch.randint(0, N, (E,), generator=gen, device=gpu).int()
    row = torch.repeat_interleave(torch.arange(N, device=gpu), deg)
    val = (torch.rand(E, generator=gen, device=gpu) / deg[row]).contiguous()
    normal = lambda *shape: torch.randn(*shape, generator=gen, device=gpu)
    X, Wn, Wc, w1, w2 = normal(N, K), normal(K, C), normal(C, C) * (0.8 / C ** 0.5), torch.zeros(C, 4, device=gpu), torch.zeros(4, 2, device=gpu)
    S = (torch.tensor([0, N], device=gpu).int(), torch.arange(N, device=gpu).int(), torch.ones(N, device=gpu))
    got = ops.s2v_forward((rp, ci, val), S, X, Wn, Wc, w1, w2, L)
    with ops.CsrPlan(rp, ci, val, N, N) as plan:
        planned = ops.s2v_forward_planned(plan, S, X, Wn, Wc, w1, w2, L)
    assert torch.equal(planned.h_final, got.h_final) and torch.equal(planned.msg, got.msg)
    h = got.msg.clamp(min=0)
    terms = X.double().abs() @ Wn.double().abs()
    err = (K + 1) * 2.0 ** -24 * terms                         # the two sums that make msg
    zero = torch.zeros(N, C, dtype=torch.float64, device=gpu)
    agg = lambda t: zero.index_add(0, row, t[ci.long()] * val.double()[:, None])
    for _ in range(L):
        h = ops.s2v_level(rp, ci, val, h, Wc, got.msg)
        terms, err = agg(terms) @ Wc.double().abs() + X.double().abs() @ Wn.double().abs(), agg(err) @ Wc.double().abs() + (K + 1) * 2.0 ** -24 * (X.double().abs() @ Wn.double().abs())
    if C == 64:
        assert torch.equal(got.h_final, h)                     # the input stage adds in the same order
    else:                                                      # and every level rounds its own sums from there on
        assert bool(((got.h_final.double() - h.double()).abs() <= err + L * (C + 900) * 2.0 ** -24 * terms).all())


@pytest.mark.parametrize("C,N,Ks", [(256, 1, (49, 64)), (256, 15, (64,)), (256, 65, (53, 64)), (256, 3001, (49, 50, 61, 64)), (256, 32_768, (49, 64)),
                                    (256, 32_769, (49, 50, 61, 64)), (256, 33_085, (53, 64)), (256, 270_001, (17, 40, 64)),
                                    (64, 1_048_577, (1, 5, 16, 19, 32, 33)), (128, 530_049, (1, 3, 16, 20, 64))])
@pytest.mark.parametrize("with_h0", [False, True])
def test_input_stage_of_wide_and_large_calls(gpu, C, N, Ks, with_h0):
    """msg alone in bf16 pieces (hidden 256, more than 48 feature columns, more than 32,768 rows), whole rows per store and fewer workgroups (more than 256 MB of
    outputs): sizes around a tile of 64 rows, the last rows of the last tile, and nothing written behind them"""
    import torch
    from graphnn_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(C + N)
    for K in Ks:
        X, W = torch.randn(N, K, generator=gen, device=gpu), torch.randn(K, C, generator=gen, device=gpu)
        out = [torch.full((N + 1, C), float("nan"), device=gpu) for _ in range(1 + with_h0)]
        ops._bound().s2v_input_f32(N, K, C, X, W, out[0], out[1] if with_h0 else None)
        at = torch.cat([torch.arange(0, min(N, 300)), torch.randint(0, N, (300,)), torch.arange(max(N - 300, 0), N)]).to(gpu)
        want, terms = X[at].double() @ W.double(), X[at].double().abs() @ W.double().abs()
        # a rounding per term and two of the split operands' own sums
        assert bool(((out[0][at].double() - want).abs() <= (K + 4) * 2.0 ** -24 * terms).all()), K
        assert bool(torch.isfinite(out[0][:N]).all()) and all(bool(torch.isnan(o[N]).all()) for o in out)
        if with_h0:
            assert torch.equal(out[1][:N], out[0][:N].clamp(min=0))


def test_input_stage_in_pieces_with_large_and_tiny_values(gpu):
    """rows and columns of 2^38 and more (scaled down) beside ordinary and tiny ones, one-hot rows to the bit, infinities and NaN in
    their rows only"""
    import torch
    from graphnn_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(3)
    N, K, C = 33_000, 64, 256
    msg = torch.empty(N, C, device=gpu)
    run = lambda X, W: (ops._bound().s2v_input_f32(N, K, C, X, W, msg, None), msg.clone())[1]
    X, W = torch.randn(N, K, generator=gen, device=gpu), torch.randn(K, C, generator=gen, device=gpu)
    for scale in (1.0, 1e-36, 1e8):
        Xs, Ws = X.clone(), W * scale
        Xs[100:200] *= 2.0 ** 40
        Ws[:, 7] *= 2.0 ** 45
        want, terms = Xs.double() @ Ws.double(), Xs.double().abs() @ Ws.double().abs()
        assert bool(torch.isfinite(want).all()) and bool(((run(Xs, Ws).double() - want).abs() <= (K + 4) * 2.0 ** -24 * terms + 2.0 ** -148).all()), scale
    one_hot = torch.zeros(N, K, device=gpu)
    label = torch.randint(0, K, (N,), generator=gen, device=gpu)
    one_hot[torch.arange(N, device=gpu), label] = 1.0
    assert torch.equal(run(one_hot, W), W[label])
    clean = run(X, W)
    X[5, 3], X[17, 60] = float("inf"), float("nan")
    got = run(X, W)
    rest = torch.ones(N, dtype=torch.bool, device=gpu)
    rest[5] = rest[17] = False
    assert torch.equal(got[rest], clean[rest])
    assert torch.equal(got[5], torch.sign(W[3]) * float("inf")) and bool(torch.isnan(got[17]).all())


@pytest.mark.parametrize("C", [128, 256])
@pytest.mark.parametrize("B,nodes", [(2047, 20), (2048, 20), (2063, 128), (2064, 129), (4096, 3), (4097, 300), (10_240, 9), (10_241, 9), (16_385, 5)])
def test_readout_of_wide_hidden_sizes_by_tiles_of_graphs(gpu, C, B, nodes):
    """batches around the sizes from which a workgroup takes 16 graphs, and from which it has eight wavefronts for them instead of sixteen: a last
    tile of one graph and of all, graphs of 0, 1, 8, 9, 64, 65 and 200 nodes among the others, nodes in another order than the rows"""
    import torch
    from graphnn_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(B + C)
    rng = np.random.default_rng(B)
    n = np.full(B, nodes, np.int64)
    n[rng.permutation(B)[:70]] = np.tile([0, 1, 8, 9, 64, 65, 200], 10)
    n[-1] = max(n[-1], 1)
    off = np.zeros(B + 1, np.int32)
    np.cumsum(n, out=off[1:])
    N, H, Q = int(off[-1]), 33, 3
    S = (torch.from_numpy(off).to(gpu), torch.randperm(N, generator=gen, device=gpu).int(), torch.rand(N, generator=gen, device=gpu) + 0.5)
    normal = lambda *shape: torch.randn(*shape, generator=gen, device=gpu)
    h, W1, W2 = normal(N, C), normal(C, H), normal(H, Q)
    pool, hidden, logits, probs, pred = ops.s2v_readout(*S, h, W1, W2, B)
    rows = h[S[1].long()].double() * S[2].double()[:, None]
    graph = torch.repeat_interleave(torch.arange(B, device=gpu), torch.from_numpy(n).to(gpu), output_size=N)
    zero = torch.zeros(B, C, dtype=torch.float64, device=gpu)
    want, terms = zero.index_add(0, graph, rows), zero.index_add(0, graph, rows.abs())
    assert bool(((pool.double() - want).abs() <= (max(nodes, 200) + 1) * 2.0 ** -24 * terms).all())          # a rounding per term
    # each layer from the one before it as the call gave it
    want, terms = (pool.double() @ W1.double()).clamp(min=0), pool.double().abs() @ W1.double().abs()
    assert bool(((hidden.double() - want).abs() <= (C + 1) * 2.0 ** -24 * terms).all())
    want, terms = hidden.double() @ W2.double(), hidden.double().abs() @ W2.double().abs()
    assert bool(((logits.double() - want).abs() <= (H + 1) * 2.0 ** -24 * terms).all())
    assert bool(((probs.double() - torch.softmax(logits.double(), 1)).abs() <= 16 * 2.0 ** -24).all())
    assert torch.equal(pred.long(), logits.argmax(1))


@pytest.mark.parametrize("where", ["h_a", "h_b", "hidden", "pool"])
@pytest.mark.parametrize("kind,C,K", [("batch", 64, 64), ("batch", 32, 32), ("batch", 100, 16), ("graph", 64, 16), ("graph", 32, 8)])
def test_forward_over_features_that_lie_in_an_output(gpu, kind, C, K, where):
    """features in a buffer that the forward writes after it has formed msg (the embeddings of the call before, fed back in): the same outputs
    as with features of their own, over a batch of small graphs and over a power-law graph"""
    import torch
    from graphnn_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(C + K)
    if kind == "batch":
        A, S, N = _small_graphs(gpu, _enough(np.random.default_rng(C).integers(10, 111, 1100), C, 3, pooled=True), 2, gen)
    else:
        N = 200_003
        deg = torch.randint(0, 30, (N,), generator=gen, device=gpu)
        rp = torch.zeros(N + 1, dtype=torch.int32, device=gpu)
        rp[1:] = torch.cumsum(deg, 0)
        E = int(rp[-1])
        A = (rp, torch.randint(0, N, (E,), generator=gen, device=gpu).int(), torch.rand(E, generator=gen, device=gpu) / 15)
        S = (torch.tensor([0, N // 3, N], device=gpu).int(), torch.arange(N, device=gpu).int(), torch.ones(N, device=gpu))
    B, H, Q = S[0].numel() - 1, 8, 3
    normal = lambda *shape: torch.randn(*shape, generator=gen, device=gpu)
    X, w = normal(N, K), (normal(K, C), normal(C, C) * (0.8 / C ** 0.5), normal(C, H), normal(H, Q))
    names = ("msg", "h_final", "pool", "hidden", "logits", "probs", "pred")
    apart, bufs = ops.ForwardBuffers(N, B, C, H, Q, gpu), ops.ForwardBuffers(N, B, C, H, Q, gpu)
    ops.s2v_forward(A, S, X, *w, 3, bufs=apart)
    room = torch.empty(max(N * K, N * C), device=gpu)            # the features, with the output at their start
    room[:N * K] = X.reshape(-1)
    rows, width = {"h_a": (N, C), "h_b": (N, C), "hidden": (B, H), "pool": (B, C)}[where]
    setattr(bufs, where, room[:rows * width].view(rows, width))
    ops.s2v_forward(A, S, room[:N * K].view(N, K), *w, 3, bufs=bufs)
    for name in names:
        got, want = getattr(bufs, name), getattr(apart, name)
        if got.dtype == torch.float32:                           # another route may form them, in another order of the sums
            assert float((got - want).norm()) <= 1e-5 * float(want.norm()), name
        else:
            assert float((got != want).float().mean()) <= 1e-3, name


@pytest.mark.parametrize("C", [20, 64, 100, 130, 200, 252, 256])
@pytest.mark.parametrize("N", [1, 33, 300, 4096, 5000])
def test_input_stage_in_place(gpu, C, N):
    """as many feature columns as hidden units, msg or h0 over the features: every row is read before it is written, whoever forms its columns"""
    import torch
    from graphnn_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(C + N)
    X, W = torch.randn(N, C, generator=gen, device=gpu), torch.randn(C, C, generator=gen, device=gpu)
    msg, h = ops.s2v_input(X, W)
    run = ops._bound().s2v_input_f32
    for in_msg in (True, False):
        a, b = X.clone(), torch.empty_like(X)
        run(N, C, C, a, W, a if in_msg else b, b if in_msg else a)
        assert torch.equal(a if in_msg else b, msg) and torch.equal(b if in_msg else a, h), in_msg
    a = X.clone()
    run(N, C, C, a, W, a, None)
    b = torch.empty_like(X)
    run(N, C, C, X, W, b, None)                                  # (wide hidden sizes: another kernel where h0 is not asked for)
    assert torch.equal(a, b)


@pytest.mark.parametrize("C", [32, 64])
@pytest.mark.parametrize("refused", [False, True])
def test_forward_with_msg_over_the_features(gpu, C, refused):
    """a forward whose msg is to lie where its features are, over a batch of small graphs that one launch takes, and over one that it refuses"""
    import torch
    from graphnn_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(C)
    A, S, N = _small_graphs(gpu, _enough(np.random.default_rng(C).integers(10, 111, 1100), C, 3, pooled=True), 2, gen)
    if refused:
        A[1][int(A[0][int(torch.nonzero(A[0][1:] > A[0][:-1])[-1])])] = 0
    B, H, Q = S[0].numel() - 1, 8, 3
    normal = lambda *shape: torch.randn(*shape, generator=gen, device=gpu)
    X, w = normal(N, C), (normal(C, C) / C ** 0.5, normal(C, C) * (0.8 / C ** 0.5), normal(C, H), normal(H, Q))
    want, bufs = ops.s2v_forward(A, S, X, *w, 3), ops.ForwardBuffers(N, B, C, H, Q, gpu)
    bufs.msg = X
    ops.s2v_forward(A, S, X, *w, 3, bufs=bufs)
    for name in ("msg", "h_final", "pool", "hidden", "logits", "probs"):
        e = getattr(want, name)
        assert float((getattr(bufs, name) - e).norm()) <= 1e-5 * float(e.norm()), name


@pytest.mark.parametrize("C", [20, 64, 100])
@pytest.mark.parametrize("late", ["pool", "hidden"])
@pytest.mark.parametrize("where", ["msg", "h_b", "a_val"])
def test_forward_whose_late_outputs_lie_in_what_is_done_with(gpu, C, late, where):
    """pooled rows or hidden layer in an array that nothing reads any more when they are written: msg, the embedding that is not the last one, the entries
    of A.  The same outputs as with arrays of their own, over a batch of small graphs that one launch would take otherwise"""
    import torch
    from graphnn_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(C)
    n = _enough(np.random.default_rng(C).integers(10, 111, 1100), C, 3, pooled=True)
    assert _tried(gpu, n, 2, 9, C, 3)
    A, S, N = _small_graphs(gpu, n, 2, gen)
    B, H, Q = S[0].numel() - 1, 8, 3
    normal = lambda *shape: torch.randn(*shape, generator=gen, device=gpu)
    X, w = normal(N, 9), (normal(9, C), normal(C, C) * (0.8 / C ** 0.5), normal(C, H), normal(H, Q))
    want, bufs = ops.s2v_forward(A, S, X, *w, 3), ops.ForwardBuffers(N, B, C, H, Q, gpu)
    rows, width = {"hidden": (B, H), "pool": (B, C)}[late]
    room = A[2] if where == "a_val" else getattr(bufs, where).view(-1)
    assert room.numel() >= rows * width
    setattr(bufs, late, room[:rows * width].view(rows, width))
    ops.s2v_forward(A, S, X, *w, 3, bufs=bufs)
    for name in ("h_final", "pool", "hidden", "logits", "probs"):
        e = getattr(want, name)
        assert float((getattr(bufs, name) - e).norm()) <= 1e-5 * float(e.norm()), name
    assert float((bufs.pred != want.pred).float().mean()) <= 1e-3


@pytest.mark.parametrize("C,K,L,nodes,mean,taken", [(64, 38, 4, 31_000, 29, False), (64, 38, 5, 32_000, 29, True), (64, 38, 4, 60_000, 39, False), (64, 38, 5, 60_000, 39, True),
                                                    (64, 9, 3, 68_000, 39, True), (72, 38, 2, 31_000, 39, False), (72, 38, 3, 31_000, 39, True), (100, 38, 3, 31_000, 39, False),
                                                    (100, 38, 4, 31_000, 39, True), (56, 38, 2, 70_000, 39, False), (56, 38, 3, 34_000, 39, True), (64, 38, 2, 150_000, 65, False),
                                                    (64, 38, 4, 150_000, 65, True)])
def test_which_batches_the_forward_tries_to_take_in_one_launch(gpu, C, K, L, nodes, mean, taken):
    """both sides of the lines below which the level-by-level kernels are the faster ones: graphs of half to one and a half times the mean size, or, where
    that is more than half a bin, all of one size"""
    n = np.random.default_rng(nodes).integers(mean // 2, mean + mean // 2 + 1, nodes // mean) if mean < 64 else np.full(nodes // mean, mean)
    assert _tried(gpu, n, 2, K, C, L) == taken


def test_bins_of_a_batch_fill_one_round_of_workgroups(gpu):
    """sizes of molecules, whose bins waste more than half a mean graph: where a round of 512 workgroups can take the batch, its bins are no more than that"""
    import torch
    from graphnn_amd import ops
    n = np.clip((np.random.default_rng(33_000).gamma(2.0, 10.0, 1138) + 9).astype(int), 10, 110)
    A, S, N = _small_graphs(gpu, n, 2, torch.Generator(device=gpu).manual_seed(1))
    bufs = ops.ForwardBuffers(N, n.size, 64, 8, 3, gpu)
    _fill(bufs)
    zero = lambda *shape: torch.zeros(*shape, device=gpu)
    ops.s2v_forward(A, S, zero(N, 9), zero(9, 64), zero(64, 64), zero(64, 8), zero(8, 3), 5, bufs=bufs)
    assert _in_one_launch(bufs)
    other = bufs.h_b if bufs.which.value == 0 else bufs.h_a
    words = other.view(-1)[:2 * ((n.size + 63) // 64)].contiguous().view(torch.int32).cpu().numpy()
    assert sum(bin(int(w) & 0xffffffff).count("1") for w in words) <= 512
