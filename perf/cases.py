"""The work a user of this framework has it do, as cases that can be timed and whose results can be compared.

``listed`` names a dozen of them, ``draw`` makes more of the same ranges, ``prepare`` builds what a program holds before
the call (the graph in its formats, the operators the decider picks, features, weights), ``run`` is one pass through the
public entry points, ``work`` counts what a pass cannot do without and ``tolerance`` says how far another correct
implementation may be off.

The graphs are the families of ``synth.py``, drawn on the GPU so that a preparation takes a fraction of a second, with
exactly ``edges`` undirected edges where enough distinct ones were drawn.
"""
import functools
import math

import numpy as np
import torch

from paramspmm_ae_amd import GNN
from paramspmm_ae_amd._capi import bw_stripe
from paramspmm_ae_amd.decider import SpMMDecider
from paramspmm_ae_amd.gnn_conv import AGNNConv
from paramspmm_ae_amd.graph_input import graph_input
from paramspmm_ae_amd.PCSR import pcsr_spmm
import ParamSDDMM
import ParamSpMM

FEATURES, CLASSES = 32, 16  # input width and class count of the training configurations


# ---- cases ------------------------------------------------------------------------------------------------------
def listed():
    return [
        # one product on a citation-graph-sized matrix, as in full-batch inference on a small dataset: launch latency
        # and the host path
        {"name": "spmm small", "kind": "spmm", "graph": "chung_lu", "nodes": 19717, "edges": 44325, "max_degree": 171, "width": 16, "dtype": "float32"},
        # class scores of a mid-sized graph: an odd node count and a width that no vector load divides
        {"name": "spmm ragged", "kind": "spmm", "graph": "chung_lu", "nodes": 200003, "edges": 1400000, "max_degree": 3000, "width": 47, "dtype": "float32"},
        # the headline sweep's matrix at its middle width
        {"name": "spmm rmat", "kind": "spmm", "graph": "rmat", "nodes": 1 << 20, "edges": 8400000, "max_degree": 0, "width": 128, "dtype": "float32"},
        # several right-hand sides of a mesh operator in double precision, the other type the operators dispatch
        {"name": "spmm mesh f64", "kind": "spmm", "graph": "mesh", "nodes": 1449 * 1451, "edges": 0, "max_degree": 0, "width": 32, "dtype": "float64"},
        # the large skewed graph: 125 million stored entries, hub rows of 17 thousand
        {"name": "spmm large", "kind": "spmm", "graph": "chung_lu", "nodes": 2450000, "edges": 61300000, "max_degree": 17000, "width": 128, "dtype": "float32"},
        # edge scores <X_i, X_j> of an attention layer
        {"name": "sddmm rmat", "kind": "sddmm", "graph": "rmat", "nodes": 1 << 20, "edges": 8400000, "max_degree": 0, "width": 64, "dtype": "float32"},
        # scores, softmax over each row's entries and their aggregation: the attention layer with a softmax, H [n, 32]
        {"name": "attention rmat", "kind": "attention", "graph": "rmat", "nodes": 1 << 20, "edges": 8400000, "max_degree": 0, "width": 32, "dtype": "float32"},
        # a hidden attention layer (no softmax, as in AGNN), forward and backward, on a graph in no particular order
        {"name": "agnn layer shuffled", "kind": "agnn_layer", "graph": "sbm_shuffled", "nodes": 1000000, "edges": 10000000, "max_degree": 0, "width": 32, "dtype": "float32"},
        # training step of a five-layer network on a small dataset: host work and launches count
        {"name": "gcn step small", "kind": "train", "net": "GCN", "graph": "chung_lu", "nodes": 19717, "edges": 44325, "max_degree": 171, "width": 16, "dtype": "float32"},
        # the same on a million nodes in community order, narrow and wide hidden layers
        {"name": "gcn step 1M", "kind": "train", "net": "GCN", "graph": "sbm", "nodes": 1000000, "edges": 10000000, "max_degree": 0, "width": 16, "dtype": "float32"},
        {"name": "gin step 1M wide", "kind": "train", "net": "GIN", "graph": "sbm", "nodes": 1000000, "edges": 10000000, "max_degree": 0, "width": 128, "dtype": "float32"},
        # a CSR matrix from host arrays to every format the operators run on
        {"name": "load rmat", "kind": "load", "graph": "rmat", "nodes": 1 << 20, "edges": 8400000, "max_degree": 0, "width": 0, "dtype": "float32"},
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    """Node counts over two decades, mean degrees 3 to 50, every family; widths 1 to 256 for the plain operators, 16 to
    128 for the layers (the widths of the driver's decider dictionary)."""
    kind = rng.choice(["spmm", "spmm", "spmm", "sddmm", "attention", "agnn_layer", "train", "train", "load"])
    graph = rng.choice(["chung_lu", "rmat", "sbm", "sbm_shuffled", "mesh"])
    nodes = int(_log_uniform(rng, 8000, 1500000))
    if graph == "sbm" or graph == "sbm_shuffled":
        nodes = nodes // 100 * 100
    if graph == "rmat":
        nodes = 1 << rng.randrange(13, 21)
    edges = int(nodes * _log_uniform(rng, 1.5, 25))
    if graph.startswith("sbm"):
        edges = int(nodes * rng.uniform(3, 14))
    edges = min(edges, 12000000)
    max_degree = int(_log_uniform(rng, 4, 150) * 2 * edges / nodes) if graph == "chung_lu" else 0
    case = {"kind": kind, "graph": graph, "nodes": nodes, "edges": 0 if graph == "mesh" else edges, "max_degree": min(max_degree, nodes // 8), "dtype": "float32"}
    if kind == "spmm":
        case["width"] = int(_log_uniform(rng, 8, 256.99)) if rng.random() < 0.8 else rng.randrange(1, 257)
        if rng.random() < 0.2:
            case["dtype"] = "float64"
            case["width"] = min(case["width"], 128)
    elif kind == "sddmm" or kind == "attention":
        case["width"] = int(_log_uniform(rng, 8, 128.99))
    elif kind == "load":
        case["width"] = 0
    else:
        case["width"] = 16 * rng.randrange(1, max(2, min(8, 60000000 // (16 * nodes)) + 1))
        if kind == "train":
            case["net"] = rng.choice(["GCN", "GIN"])
    return case


# ---- graphs -----------------------------------------------------------------------------------------------------
def _mesh_sides(nodes):
    nx = int(math.isqrt(nodes))
    while nodes % nx and nodes // nx < 2 * nx:
        nx -= 1
    return (nx, nodes // nx)


def _entries(case):
    """(rows, stored entries) of a case's matrix: both directions of every edge and the diagonal."""
    if case["graph"] == "mesh":
        nx, ny = _mesh_sides(case["nodes"])
        return nx * ny, 2 * (nx * (ny - 1) + ny * (nx - 1)) + nx * ny
    return case["nodes"], 2 * case["edges"] + case["nodes"]


def _endpoints(case, gen):
    """Endpoint pairs, a quarter more than asked for: some will be loops and duplicates."""
    n, m = case["nodes"], int(case["edges"] * 1.25) + 64
    dev = torch.device("cuda")
    if case["graph"] == "rmat":
        u = torch.zeros(m, dtype=torch.int64, device=dev)
        v = torch.zeros(m, dtype=torch.int64, device=dev)
        for _ in range(n.bit_length() - 1):
            r = torch.rand(m, device=dev, generator=gen)
            u = u * 2 + (r >= 0.76)
            v = v * 2 + (((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
        return u, v
    if case["graph"] == "chung_lu":
        alpha = 1.0 / 1.1  # degree exponent 2.1
        k = torch.arange(n, dtype=torch.float64, device=dev)
        lo, hi = 1e-3, float(n)
        for _ in range(40):  # offset that gives the hub its expected degree
            mid = (lo + hi) / 2
            w = (k + mid) ** -alpha
            lo, hi = (mid, hi) if (w[0] / w.sum() * 2 * case["edges"]).item() > case["max_degree"] else (lo, mid)
        cdf = torch.cumsum((k + (lo + hi) / 2) ** -alpha, 0)
        cdf /= cdf[-1].clone()
        perm = torch.randperm(n, device=dev, generator=gen)
        return tuple(perm[torch.searchsorted(cdf, torch.rand(m, dtype=torch.float64, device=dev, generator=gen)).clamp_(max=n - 1)] for _ in range(2))
    # block model: communities of 100 consecutive nodes, one edge in eleven leaves its community
    out = m // 11
    u = torch.randint(0, n, (m,), device=dev, generator=gen)
    v = u // 100 * 100 + torch.randint(0, 100, (m,), device=dev, generator=gen)
    v[:out] = torch.randint(0, n, (out,), device=dev, generator=gen)
    if case["graph"] == "sbm_shuffled":
        perm = torch.randperm(n, device=dev, generator=gen)
        u, v = perm[u], perm[v.clamp_(max=n - 1)]
    return u, v.clamp_(max=n - 1)


def _csr(case, gen, relabel=None):
    """Host CSR arrays: D^-1/2 (A + I) D^-1/2, for GIN the pattern with 1.5 on the diagonal.  ``relabel``: the vertices
    are numbered anew, in pairs rotated by a random step and at random swapped -- another matrix with as many 2x1 blocks
    and row segments."""
    dev = torch.device("cuda")
    if case["graph"] == "mesh":
        nx, ny = _mesh_sides(case["nodes"])
        n = nx * ny
        idx = torch.arange(n, device=dev).view(ny, nx)
        lo = torch.cat([idx[:, :-1].reshape(-1), idx[:-1, :].reshape(-1)])
        hi = torch.cat([idx[:, 1:].reshape(-1), idx[1:, :].reshape(-1)])
    else:
        n = case["nodes"]
        u, v = _endpoints(case, gen)
        keep = u != v
        u, v = u[keep], v[keep]
        key = torch.unique(torch.minimum(u, v) * n + torch.maximum(u, v))
        if key.numel() > case["edges"]:
            key = key[torch.randperm(key.numel(), device=dev, generator=gen)[: case["edges"]]]
        lo, hi = key // n, key % n
    if relabel is not None:
        even = n // 2 * 2
        swap = torch.randint(0, 2, (n // 2,), device=dev, generator=relabel).repeat_interleave(2)
        new = (torch.arange(even, device=dev) ^ swap).roll(2 * torch.randint(0, n // 2, (1,), device=dev, generator=relabel).item())
        new = torch.cat([new, torch.arange(even, n, device=dev)])
        lo, hi = new[lo], new[hi]
    diag = torch.arange(n, device=dev)
    key = torch.sort(torch.cat([lo * n + hi, hi * n + lo, diag * n + diag])).values
    row, col = key // n, key % n
    count = torch.bincount(row, minlength=n)
    if case.get("net") == "GIN":
        val = torch.where(row == col, 1.5, 1.0).float()
    else:
        scale = count.double().pow(-0.5)
        val = (scale[col] * scale[row]).float()
    rowPtr = torch.zeros(n + 1, dtype=torch.int32, device=dev)
    rowPtr[1:] = torch.cumsum(count, 0).int()
    return rowPtr.cpu().numpy(), col.int().cpu().numpy(), val.cpu().numpy()


# ---- preparation ------------------------------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _decider(dims):
    decider = SpMMDecider()
    decider.gen_model_dict(list(dims))
    return decider


def _load(arrays, if_mask=False):
    graph = graph_input("case", "")
    graph.verbose = False
    return graph.load_from_csr(*arrays, if_mask=if_mask)


def _operator(graph, width):
    if_split, vec_size, CF, blkWarpNum = _decider((width,)).config_PCSR(graph, width)
    return pcsr_spmm(graph=graph, vec_size=vec_size, if_split=if_split, CF=CF, blkWarpNum=blkWarpNum)


def _randn(rows, width, gen, dtype=torch.float32):
    return torch.randn(rows, width, device="cuda", generator=gen, dtype=dtype)


def _unit_rows(rows, width, gen):
    return torch.nn.functional.normalize(_randn(rows, width, gen), dim=1).contiguous()


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind, width = case["kind"], case["width"]
    if kind == "load":
        # one graph under numberings drawn from the seed: the formats' arrays keep their lengths, which depend on the matrix
        return {"kind": kind, "arrays": _csr(case, torch.Generator(device="cuda").manual_seed(1), relabel=gen)}
    arrays = _csr(case, gen)
    n = arrays[0].size - 1
    rows = (n + 1) // 2 * 2  # even, so that 2x1 blocks fit
    state = {"kind": kind}
    graph = _load(arrays, if_mask=kind == "agnn_layer")
    if kind == "spmm":
        state["op"] = _operator(graph, width)
        state["X"] = _randn(rows, width, gen, getattr(torch, case["dtype"]))
        state["val"] = state["op"].val.double() if case["dtype"] == "float64" else None
    elif kind == "sddmm":
        state["op"] = _operator(graph, width)
        state["X"] = _unit_rows(rows, width, gen)
    elif kind == "attention":
        # the edge values live in CSR order: one of the two CSR layouts, with the decider's CF and workgroup size
        if_split, _, CF, bw = _decider((32,)).config_PCSR(graph, 32)
        c = graph.csr_data
        state.update(split=bool(if_split), n=n, CF=CF, bw=bw | bw_stripe(c.xcd_stripe(bool(if_split))),
                     rowPtr=c.on_device("rowPtr_split" if if_split else "rowPtr", "cuda"), colIdx=c.on_device("colIdx", "cuda"),
                     val=c.on_device("val", "cuda"), target=c.on_device("target_row", "cuda") if if_split else None,
                     X=_unit_rows(n, width, gen), Y=_unit_rows(n, width, gen), H=_randn(n, 32, gen))
    elif kind == "agnn_layer":
        state["ops"] = GNN.configure_operators(_decider((width,)), graph, [width])
        torch.manual_seed(seed)
        state["layer"] = AGNNConv(width, width).cuda()
        state["colIdx"] = graph.csr_data.on_device("colIdx", "cuda").unsqueeze(-1)
        state["X"] = _unit_rows(rows, width, gen).requires_grad_()
        state["dY"] = _randn(rows, width, gen)
    else:
        dims = sorted({width, CLASSES, FEATURES})
        ops = GNN.configure_operators(_decider(tuple(dims)), graph, dims)
        torch.manual_seed(seed)
        state["model"] = GNN.build_model(case["net"], graph, ops, width, FEATURES, CLASSES)
        state["labels"] = torch.randint(0, CLASSES, graph.y.shape, device="cuda", generator=gen)
    return state


# ---- one pass ---------------------------------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    if kind == "spmm":
        op = state["op"]
        return op.GIN_spmm(state["X"]) if state["val"] is None else op.AGNN_spmm(state["val"], state["X"])
    if kind == "sddmm":
        return state["op"].AGNN_sddmm(state["X"])
    if kind == "attention":
        s = state
        if s["split"]:
            e, m = ParamSDDMM.csr_split_sddmm_scaled_rowmax(s["X"], s["Y"], s["rowPtr"], s["colIdx"], s["val"], s["target"], s["n"], s["bw"])
            return ParamSpMM.csr_split_spmm_softmax(s["H"], s["rowPtr"], s["colIdx"], e, m, s["target"], s["CF"], s["bw"])
        e, m = ParamSDDMM.csr_sddmm_scaled_rowmax(s["X"], s["Y"], s["rowPtr"], s["colIdx"], s["val"], s["bw"])
        return ParamSpMM.csr_spmm_softmax(s["H"], s["rowPtr"], s["colIdx"], e, m, s["CF"], s["bw"])
    if kind == "agnn_layer":
        X, layer = state["X"], state["layer"]
        X.grad = layer.weights.grad = layer.attention_w.grad = None
        out = layer(X, state["ops"], state["colIdx"], relu_input=True)
        out.backward(state["dY"])
        return out.detach(), X.grad, layer.weights.grad, layer.attention_w.grad
    if kind == "train":
        # forward, loss and gradients; the update that follows is PyTorch's own Adam
        model = state["model"]
        for p in model.parameters():
            p.grad = None
        loss = GNN.loss_of_step(model, state["labels"])
        loss.backward()
        return [loss.detach()] + [p.grad for p in model.parameters()]
    graph = _load(state["arrays"])
    c, b = graph.csr_data, graph.bcsr_data
    return [c.rowPtr_split, c.target_row, b.rowPtr, b.colIdx, b.val, b.rowPtr_split, b.target_row, graph.get_info()]


# ---- what a pass cannot do without ------------------------------------------------------------------------------
def work(case):
    n, nnz = _entries(case)
    kind, w = case["kind"], case["width"]
    size = 8 if case["dtype"] == "float64" else 4
    matrix = 4 * (n + 1) + 4 * nnz  # row pointers and columns
    dense = size * n * w
    if kind == "spmm":
        return {"bytes": matrix + size * nnz + 2 * dense, "flops": 2 * nnz * w}
    if kind == "sddmm":
        return {"bytes": matrix + 4 * nnz + dense, "flops": 2 * nnz * w}
    if kind == "attention":  # the scores need not leave the chip
        return {"bytes": matrix + 4 * nnz + 2 * dense + 2 * 4 * n * 32, "flops": 2 * nnz * (w + 32)}
    if kind == "agnn_layer":
        # X and the matrix read once each way; out, dX written; the incoming gradient read; the two sparse sums each way
        # and the three dense products
        return {"bytes": 2 * matrix + 5 * dense, "flops": 8 * nnz * w + 6 * n * w * w}
    if kind == "train":
        # per layer: the matrix with its values each way, the input and output of both passes once (the first layer's
        # input needs no gradient); sparse products of the narrower width both ways, three dense products
        total = {"bytes": 8 * n, "flops": 0}
        widths = [FEATURES, w, w, w, w, CLASSES]
        for i, (a, b) in enumerate(zip(widths, widths[1:])):
            total["bytes"] += 2 * (matrix + 4 * nnz) + 4 * n * (2 * a + 2 * b if i else a + 2 * b)
            total["flops"] += (4 if i else 2) * nnz * min(a, b) + (6 if i else 4) * n * a * b
        return total
    # load: the CSR arrays read; 2x1 blocks (about as many as entries) and the two row splits written
    return {"bytes": 2 * matrix + 12 * nnz + 12 * n, "flops": 0}


def tolerance(case):
    if case["kind"] == "load":
        return {"rel": 1e-6, "differ": 0.0}  # whole numbers alike; the statistics are means and deviations of 32-bit sums
    if case["dtype"] == "float64":
        return {"rel": 1e-13}
    if case["kind"] == "train":
        # an activation that rounds to the other side of zero drops or adds a term of the gradient
        return {"rel": 1e-4}
    return {"rel": 1e-5}
