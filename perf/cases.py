"""The work that users of this framework have it do, as cases to be timed.

Four kinds of work, each through the public helpers of graphnn_amd.ops:

  infer   one forward of the structure2vec network over a batch of small graphs (molecules, proteins)
  train   one training iteration on such a batch: the batch's matrices from its edge list, forward with every level kept,
          loss, backward, weight gradients, optimizer step
  spmm    one product of a CSR matrix with a dense matrix
  graph   one forward over a single large power-law graph cut into contiguous subgraphs, with the softmax of node scores
          inside every subgraph
"""
import math

import numpy as np
import torch

from graphnn_amd import ops

LABEL_TYPES_GRAPH = 16      # node label types of the power-law graphs
READOUT_GRAPH = 64          # hidden units of their readout


def listed():
    return [
        # scoring one small batch (MUTAG-like): a service answering single requests; launches and latency count
        {"name": "infer_50", "kind": "infer", "graphs": 50, "sizes": "uniform", "lo": 10, "hi": 28, "edge_factor": 1.1, "types": 7,
         "input": "onehot", "hidden": 64, "units": 32, "classes": 2, "levels": 3},
        # the headline configuration: 256 molecules with NCI109's right-skewed sizes
        {"name": "infer_256", "kind": "infer", "graphs": 256, "sizes": "skewed", "lo": 10, "hi": 110, "edge_factor": 1.1, "types": 38,
         "input": "onehot", "hidden": 64, "units": 32, "classes": 2, "levels": 4},
        # a whole screening library in one call, node tags handed over as integers (no one-hot matrix), narrow network
        {"name": "infer_labels_3001", "kind": "infer", "graphs": 3001, "sizes": "skewed", "lo": 10, "hi": 110, "edge_factor": 1.1, "types": 37,
         "input": "labels", "hidden": 32, "units": 32, "classes": 2, "levels": 4},
        # bulk scoring: 880 thousand nodes in one batch, past what the one-launch forward is for
        {"name": "infer_30000", "kind": "infer", "graphs": 30000, "sizes": "skewed", "lo": 10, "hi": 110, "edge_factor": 1.1, "types": 38,
         "input": "onehot", "hidden": 64, "units": 32, "classes": 2, "levels": 4},
        # the wide network: 10,000 graphs, hidden 256, five levels
        {"name": "infer_wide_10000", "kind": "infer", "graphs": 10000, "sizes": "uniform", "lo": 20, "hi": 40, "edge_factor": 1.1, "types": 64,
         "input": "onehot", "hidden": 256, "units": 128, "classes": 2, "levels": 5},
        # protein graphs (ENZYMES' degree) and an embedding size that nothing is tuned for
        {"name": "infer_odd_1500", "kind": "infer", "graphs": 1500, "sizes": "uniform", "lo": 2, "hi": 63, "edge_factor": 1.9, "types": 3,
         "input": "onehot", "hidden": 100, "units": 50, "classes": 6, "levels": 3},
        # the reference's default training run: ENZYMES, batches of 50, hidden 64, three levels, momentum SGD
        {"name": "train_50", "kind": "train", "graphs": 50, "sizes": "uniform", "lo": 2, "hi": 63, "edge_factor": 1.9, "types": 3,
         "hidden": 64, "units": 64, "classes": 6, "levels": 3, "optimizer": "momentum"},
        # training on the headline configuration's batches with Adam
        {"name": "train_256", "kind": "train", "graphs": 256, "sizes": "skewed", "lo": 10, "hi": 110, "edge_factor": 1.1, "types": 38,
         "hidden": 64, "units": 32, "classes": 2, "levels": 4, "optimizer": "adam"},
        # large-batch training of the wide network
        {"name": "train_wide_10000", "kind": "train", "graphs": 10000, "sizes": "uniform", "lo": 20, "hi": 40, "edge_factor": 1.1, "types": 64,
         "hidden": 256, "units": 128, "classes": 2, "levels": 5, "optimizer": "momentum"},
        # one message-passing product on a graph of uniform degree, far larger than the caches
        {"name": "spmm_1m", "kind": "spmm", "rows": 1000000, "cols": 1000000, "entries": 10000000, "width": 128, "planned": False},
        # one big social-network-like graph kept on the device, batch after batch of features: the matrix's plan is kept too
        {"name": "graph_4m_planned", "kind": "graph", "nodes": 1 << 22, "degree": 16, "hidden": 64, "levels": 3, "subgraphs": 4096, "planned": True},
        # a graph seen once: nothing about its matrix is known before the call
        {"name": "graph_300k", "kind": "graph", "nodes": 300001, "degree": 13, "hidden": 32, "levels": 3, "subgraphs": 301, "planned": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["infer", "infer", "infer", "train", "train", "spmm", "graph"])
    if kind in ("infer", "train"):
        hidden = rng.choice([16, 32, 64, 64, 128, 256, rng.randint(20, 200)])
        # the largest batches shrink with the width of the network, so that none costs more than the listed ones
        most = min(30000, 2560000 // hidden) if kind == "infer" else min(10000, 2560000 // hidden)
        case = {"kind": kind, "graphs": _log_int(rng, 8, most), "types": rng.randint(2, 64), "hidden": hidden,
                "units": rng.choice([16, 32, 64, 128, rng.randint(10, 128)]), "classes": rng.randint(2, 10), "levels": rng.randint(2, 5),
                "edge_factor": round(rng.uniform(1.05, 2.2), 3)}
        if rng.random() < 0.5:
            case.update(sizes="skewed", lo=10, hi=110)
        else:
            lo = rng.randint(2, 25)
            case.update(sizes="uniform", lo=lo, hi=rng.randint(lo + 5, lo + 30))
        if kind == "infer":
            case["input"] = rng.choice(["onehot", "onehot", "labels"])
        else:
            case["optimizer"] = rng.choice(["momentum", "adam"])
        return case
    if kind == "spmm":
        rows, width = _log_int(rng, 5000, 1000000), rng.choice([16, 32, 64, 128, 256, rng.randint(1, 200)])
        degree = rng.uniform(2, 12)
        entries = min(int(rows * degree), 1280000000 // max(width, 128))
        return {"kind": "spmm", "rows": rows, "cols": _log_int(rng, 5000, 1000000), "entries": entries, "width": width, "planned": rng.random() < 0.3}
    nodes, hidden = _log_int(rng, 40000, 3000000), rng.choice([16, 32, 64, rng.randint(20, 100)])
    nodes = min(nodes, 3000000 * 64 // max(hidden, 64))
    return {"kind": "graph", "nodes": nodes, "degree": rng.randint(4, 18), "hidden": hidden, "levels": rng.randint(2, 3),
            "subgraphs": _log_int(rng, 50, max(51, nodes // 500)), "planned": rng.random() < 0.5}


# ---------------------------------------------------------------- inputs
def _graph_sizes(case):
    """nodes per graph, a function of the case alone (quantiles of the size distribution); prepare() shuffles them"""
    B = case["graphs"]
    u = (np.arange(B) + 0.5) / B
    if case["sizes"] == "skewed":
        return (case["lo"] + np.minimum(case["hi"] - case["lo"], np.floor(-20.0 * np.log1p(-u)))).astype(np.int64)
    return (case["lo"] + np.floor(u * (case["hi"] - case["lo"] + 1))).astype(np.int64)


def _edge_count(case):
    """directed edges of a batch, up to the few repeated draws that are dropped"""
    sizes = _graph_sizes(case)
    return int(2 * np.minimum(np.maximum(np.rint(case["edge_factor"] * sizes), sizes - 1), sizes * (sizes - 1) // 2).sum())


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(gen, shape, std):
    return torch.randn(shape, generator=gen, device="cuda") * std


def _batch(case, seed):
    """A batch of connected graphs: a random spanning tree each plus extra edges, every edge in both directions, edges by source
    node and neighbours ascending, as the datasets list them."""
    gen = _generator(seed)
    order = np.random.default_rng(int(seed)).permutation(case["graphs"])
    sizes_host = _graph_sizes(case)[order]
    offsets_host = np.zeros(sizes_host.size + 1, np.int32)
    np.cumsum(sizes_host, out=offsets_host[1:])
    N = int(offsets_host[-1])
    sizes = torch.from_numpy(sizes_host).cuda()
    offsets = torch.from_numpy(offsets_host.astype(np.int64)).cuda()
    graph = torch.repeat_interleave(torch.arange(sizes.numel(), device="cuda"), sizes, output_size=N)
    start, node = offsets[graph], torch.arange(N, device="cuda")
    local = node - start
    parent = start + (torch.rand(N, generator=gen, device="cuda") * local).long().minimum((local - 1).clamp(min=0))
    tree = torch.stack([parent, node])[:, local > 0]
    # extra edges: factor * n of them altogether with the tree, pairs drawn freely, repeats and loops dropped
    extra_host = np.maximum(0, np.rint(case["edge_factor"] * sizes_host).astype(np.int64) - (sizes_host - 1))
    n_extra = int(extra_host.sum())
    eg = torch.repeat_interleave(torch.arange(sizes.numel(), device="cuda"), torch.from_numpy(extra_host).cuda(), output_size=n_extra)
    pick = lambda: offsets[eg] + (torch.rand(n_extra, generator=gen, device="cuda") * sizes[eg]).long().minimum(sizes[eg] - 1)
    a, b = pick(), pick()
    extra = torch.stack([torch.minimum(a, b), torch.maximum(a, b)])[:, a != b]
    both = torch.cat([tree, extra], 1)
    key = torch.unique(torch.cat([both[0] * N + both[1], both[1] * N + both[0]]))
    x, y = key // N, key % N
    row_ptr = torch.zeros(N + 1, dtype=torch.int32, device="cuda")
    row_ptr[1:] = torch.cumsum(torch.bincount(x, minlength=N), 0)
    labels = torch.randint(0, case["types"], (N,), generator=gen, device="cuda")
    onehot = torch.zeros(N, case["types"], device="cuda")
    onehot[node, labels] = 1.0
    classes = torch.randint(0, case["classes"], (sizes.numel(),), generator=gen, device="cuda")
    return {"gen": gen, "N": N, "offsets_host": offsets_host, "largest": int(sizes_host.max()), "x": x.int(), "y": y.int(),
            "A": (row_ptr, y.int(), torch.ones(y.numel(), device="cuda")),
            "S": (offsets.int(), node.int(), torch.ones(N, device="cuda")), "labels": labels.int(), "X": onehot,
            "Y": (torch.arange(sizes.numel() + 1, device="cuda").int(), classes.int(), torch.ones(sizes.numel(), device="cuda"))}


def _prepare_batch(case, seed):
    s = _batch(case, seed)
    s["case"] = case
    gen, C, H, Q = s["gen"], case["hidden"], case["units"], case["classes"]
    train = case["kind"] == "train"
    # inference with grown weights (0.1 at hidden 64, the same gain per level at other widths), training from the reference's start
    std = 0.01 if train else 0.8 / math.sqrt(C)
    s["W"] = [_normal(gen, (case["types"], C), std if train else 0.1), _normal(gen, (C, C), std), _normal(gen, (C, H), std), _normal(gen, (H, Q), std)]
    # the one-launch forward where the framework's own host layer takes it: batches of up to 120,000 nodes
    s["one_launch"] = C in (16, 32, 64, 128) and s["N"] <= 120000
    N, B, dev = s["N"], case["graphs"], s["X"].device
    if not train:
        s["bufs"] = (ops.BatchedBuffers if s["one_launch"] else ops.ForwardBuffers)(N, B, C, H, Q, dev)
        return s
    s["grads"] = [torch.zeros_like(w) for w in s["W"]]
    s["moments"] = [[torch.zeros_like(w) for w in s["W"]] for _ in range(2)]
    s["step"] = 0
    L = case["levels"]
    s["us"] = torch.empty((L, N, C), device=dev)
    s["dmsg"] = torch.empty((N, C), device=dev)
    s["g2"] = torch.empty((N, C), device=dev)
    if s["one_launch"]:
        s["bufs"] = ops.BatchedBuffers(N, B, C, H, Q, dev)
    else:
        s["hs"] = torch.empty((L + 1, N, C), device=dev)
    return s


def _prepare_spmm(case, seed):
    gen = _generator(seed)
    m, k, nnz = case["rows"], case["cols"], case["entries"]
    rows = torch.randint(0, m, (nnz,), generator=gen, device="cuda")
    key = torch.sort(rows * k + torch.randint(0, k, (nnz,), generator=gen, device="cuda"))[0]
    row_ptr = torch.zeros(m + 1, dtype=torch.int32, device="cuda")
    row_ptr[1:] = torch.cumsum(torch.bincount(key // k, minlength=m), 0)
    s = {"case": case, "A": (row_ptr, (key % k).int(), torch.ones(nnz, device="cuda")),
         "B": torch.randn(k, case["width"], generator=gen, device="cuda"), "out": torch.empty(m, case["width"], device="cuda")}
    if case["planned"]:
        s["plan"] = ops.CsrPlan(*s["A"], m, k)
    return s


def _rmat(gen, nodes, entries):
    """row_ptr, col_idx of an R-MAT graph (0.57, 0.19, 0.19, 0.05), columns ascending inside a row, repeats kept"""
    scale = max(1, (nodes - 1).bit_length())
    keys = []
    for lo in range(0, entries, 1 << 24):
        n = min(1 << 24, entries - lo)
        r = torch.zeros(n, dtype=torch.int64, device="cuda")
        c = torch.zeros(n, dtype=torch.int64, device="cuda")
        for _ in range(scale):
            u = torch.rand(n, generator=gen, device="cuda")
            r = (r << 1) | (u >= 0.76)
            c = (c << 1) | (((u >= 0.57) & (u < 0.76)) | (u >= 0.95))
        keys.append(((r * nodes) >> scale) * nodes + ((c * nodes) >> scale))
    key = torch.sort(torch.cat(keys))[0]
    row_ptr = torch.zeros(nodes + 1, dtype=torch.int32, device="cuda")
    row_ptr[1:] = torch.cumsum(torch.bincount(key // nodes, minlength=nodes), 0)
    return row_ptr, (key % nodes).int()


def _segment_bounds(case):
    per = case["nodes"] // case["subgraphs"]
    bounds = np.arange(case["subgraphs"] + 1, dtype=np.int64) * per
    bounds[-1] = case["nodes"]
    return bounds


def _prepare_graph(case, seed):
    gen = _generator(seed)
    N, C, B, K, H = case["nodes"], case["hidden"], case["subgraphs"], LABEL_TYPES_GRAPH, READOUT_GRAPH
    row_ptr, col_idx = _rmat(gen, N, N * case["degree"])
    # a mean over the neighbours: power-law sums would grow with the degree level after level
    val = torch.repeat_interleave(1.0 / (row_ptr[1:] - row_ptr[:-1]).clamp(min=1).float(), (row_ptr[1:] - row_ptr[:-1]).long(), output_size=col_idx.numel())
    X = torch.zeros(N, K, device="cuda")
    X[torch.arange(N, device="cuda"), torch.randint(0, K, (N,), generator=gen, device="cuda")] = 1.0
    std = 0.8 / math.sqrt(C)
    bounds = torch.from_numpy(_segment_bounds(case)).cuda()
    s = {"case": case, "A": (row_ptr, col_idx, val), "S": (bounds.int(), torch.arange(N, device="cuda").int(), torch.ones(N, device="cuda")),
         "X": X, "W": [_normal(gen, (K, C), 0.1), _normal(gen, (C, C), std), _normal(gen, (C, H), std), _normal(gen, (H, 2), 0.1)],
         "w_score": _normal(gen, (C, 1), 0.1), "lens": (bounds[1:] - bounds[:-1]).int(),
         "bufs": ops.ForwardBuffers(N, B, C, H, 2, X.device), "score": torch.empty(N, 1, device="cuda")}
    if case["planned"]:
        s["plan"] = ops.CsrPlan(row_ptr, col_idx, val, N, N)
    return s


def prepare(case, seed):
    return {"infer": _prepare_batch, "train": _prepare_batch, "spmm": _prepare_spmm, "graph": _prepare_graph}[case["kind"]](case, seed)


# ---------------------------------------------------------------- one pass
def _forward_outputs(bufs):
    return {"msg": bufs.msg, "h": bufs.h_final, "pool": bufs.pool, "hidden": bufs.hidden, "logits": bufs.logits, "probs": bufs.probs, "pred": bufs.pred}


def _run_infer(s):
    case, bufs = s["case"], s["bufs"]
    Wn, Wc, W1, W2 = s["W"]
    L = case["levels"]
    if s["one_launch"]:
        if case["input"] == "labels":
            ops.s2v_forward_batched_labels(s["A"], s["S"], s["labels"], Wn, Wc, W1, W2, L, s["largest"], bufs=bufs)
        else:
            ops.s2v_forward_batched(s["A"], s["S"], s["X"], Wn, Wc, W1, W2, L, s["largest"], bufs=bufs)
    elif case["input"] == "labels":
        msg, h = ops.s2v_input_labels(s["labels"], Wn)
        for l in range(L):
            h = ops.s2v_level(*s["A"], h, Wc, msg, out=(bufs.h_a, bufs.h_b)[l & 1])
        pool, hidden, logits, probs, pred = ops.s2v_readout(*s["S"], h, W1, W2, case["graphs"])
        return {"msg": msg, "h": h, "pool": pool, "hidden": hidden, "logits": logits, "probs": probs, "pred": pred}
    else:
        ops.s2v_forward(s["A"], s["S"], s["X"], Wn, Wc, W1, W2, L, bufs=bufs)
    return _forward_outputs(bufs)


def _run_train(s):
    case = s["case"]
    Wn, Wc, W1, W2 = s["W"]
    gWn, gWc, gW1, gW2 = s["grads"]
    N, B, C, L = s["N"], case["graphs"], case["hidden"], case["levels"]
    us, dmsg, g2 = s["us"], s["dmsg"], s["g2"]
    # the batch's matrices: A and its transpose from the edge list, S from the graphs' node offsets
    A, At = ops.csr_group_both(N, s["x"], s["y"])
    S = ops.csr_consecutive_rows_host(s["offsets_host"], s["X"].device)
    # forward, every level kept
    if s["one_launch"]:
        bufs, hs = ops.s2v_forward_batched_train(A, S, s["X"], Wn, Wc, W1, W2, L, s["largest"], bufs=s["bufs"])
        pool, hidden, logits = bufs.pool, bufs.hidden, bufs.logits
    else:
        hs = s["hs"]
        msg, hs[0] = ops.s2v_input(s["X"], Wn)
        for l in range(L):
            ops.s2v_level(*A, hs[l], Wc, msg, out=hs[l + 1])
        pool, hidden, logits, _, _ = ops.s2v_readout(*S, hs[L], W1, W2, B)
    loss, _, probs, loss_rows, hit = ops.loss_acc(logits, *s["Y"], want_rows=True)
    # backward: readout, levels from the top (each past the gate of the level below, summed into the msg gradient), weights
    dlogits, du, g = ops.readout_backward(S, probs, s["Y"], 1.0 / B, hidden, W1, W2, N)
    ops.grad_gate(hs[L], g, g, dmsg)
    for l in range(L, 0, -1):
        ops.s2v_level_backward(*At, g, Wc, u=us[l - 1], g_prev=g2, gate_h=hs[l - 1], acc=dmsg)
        g, g2 = g2, g
    ops.gemm_tn_batch([(hs[:L].reshape(L * N, C), us.reshape(L * N, C), gWc), (s["X"], dmsg, gWn), (pool, du, gW1), (hidden, dlogits, gW2)])
    s["step"] += 1
    m, v = s["moments"]
    if case["optimizer"] == "adam":
        ops.adam_batch(s["W"], s["grads"], m, v, 1e-4, 1e-4, 5.0, 0.9, 0.999, 1e-8, s["step"])
    else:
        ops.momentum_sgd_batch(s["W"], s["grads"], m, 1e-4, 0.9, 1e-4)
    return {"loss": loss, "probs": probs, "loss_rows": loss_rows, "hit": hit, "weights": s["W"], "moments": s["moments"]}


def _run_spmm(s):
    if s["case"]["planned"]:
        return s["plan"].spmm(s["B"], out=s["out"])
    return ops.spmm(*s["A"], s["B"], s["case"]["rows"], out=s["out"])


def _run_graph(s):
    Wn, Wc, W1, W2 = s["W"]
    bufs, L = s["bufs"], s["case"]["levels"]
    if s["case"]["planned"]:
        ops.s2v_forward_planned(s["plan"], s["S"], s["X"], Wn, Wc, W1, W2, L, bufs=bufs)
    else:
        ops.s2v_forward(s["A"], s["S"], s["X"], Wn, Wc, W1, W2, L, bufs=bufs)
    ops.gemm(bufs.h_final, s["w_score"], out=s["score"])
    ops.jagged_softmax(s["score"], s["lens"])
    return dict(_forward_outputs(bufs), score=s["score"])


def run(state):
    return {"infer": _run_infer, "train": _run_train, "spmm": _run_spmm, "graph": _run_graph}[state["case"]["kind"]](state)


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    if case["kind"] == "spmm":
        m, k, nnz, n = case["rows"], case["cols"], case["entries"], case["width"]
        return {"bytes": 4 * (m + 1) + 8 * nnz + 4 * k * n + 4 * m * n, "flops": 2 * nnz * n}
    if case["kind"] == "graph":
        N, E, B, K, H, Q = case["nodes"], case["nodes"] * case["degree"], case["subgraphs"], LABEL_TYPES_GRAPH, READOUT_GRAPH, 2
    else:
        N, E = int(_graph_sizes(case).sum()), _edge_count(case)
        B, K, H, Q = case["graphs"], case["types"], case["units"], case["classes"]
    C, L = case["hidden"], case["levels"]
    weights = K * C + C * C + C * H + H * Q
    sparse = 4 * (N + 1) + 8 * E + 4 * (B + 1) + 8 * N
    features = 4 * N if case.get("input") == "labels" else 4 * N * K
    forward = (0 if case.get("input") == "labels" else 2 * N * K * C) + L * (2 * E * C + 2 * N * C * C + 2 * N * C) + 2 * N * C + 2 * B * (C * H + H * Q)
    per_graph = 4 * B * (C + H + 2 * Q + 1)
    if case["kind"] == "train":
        # edges, features and labels in; weights and optimizer state in and out; loss and probabilities out
        states = 2 if case["optimizer"] == "adam" else 1
        backward = 2 * B * 2 * (C * H + H * Q) + L * (2 * E * C + 4 * N * C * C) + 2 * N * K * C
        return {"bytes": 8 * E + 4 * (B + 1) + features + 8 * B + 8 * weights * (1 + states) + 4 * B * (Q + 2), "flops": forward + backward}
    score = (2 * N * C, 4 * N) if case["kind"] == "graph" else (0, 0)
    return {"bytes": sparse + features + 4 * weights + 8 * N * C + per_graph + score[1], "flops": forward + score[0]}


def tolerance(case):
    # 32-bit sums in another order.  Gradients pass ReLU gates that rounding may flip, and cancel over the batch: ten times that.
    # Whole values: predictions and hits, which near ties decide.
    if case["kind"] == "train":
        return {"rel": 1e-4, "differ": 1e-3}
    return {"rel": 1e-5, "differ": 1e-3}
