"""Performance cases of the walk engine: the calls a user's program makes, over their real range.

Kinds of case (field "kind"):
  walk      Walk.run on a graph that the program keeps, then X_hops, as the host array of
            Walk.frontier or as the device tile matrix of Walk.export.
  batch     WalkBatch.run of uneven queries over several graphs, then every query's X_hops.
  square    C = A * A by tile products (symbolic and numeric pass); with "min_bits" the numeric
            pass that sends dense tile pairs to the matrix cores.
  pruned    one hop X_{k+1} = X_k * A of a product walk, sized by the cost model.
  ingest    host edge arrays to the device tile matrix of A^T.
  two_hop   pair enumeration of an edge list, to host arrays.
  predict   the cost model's forward pass on host feature rows.
  train     two optimiser steps of the cost model on host samples, and its new weights.

Graphs are R-MAT (edge factor 16, (a, b, c, d) = (0.57, 0.19, 0.19, 0.05)); n_vertices need not
be a power of two (ids are then taken modulo n_vertices); one graph of a batch is Erdos-Renyi.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import matrixgraph_amd as M
from matrixgraph_amd import learned as LN
from matrixgraph_amd import workloads as WL

ABCD = (0.57, 0.19, 0.19, 0.05)
EDGE_FACTOR = 16
COMMUNITY_SIZE = 1024
COMMUNITY_P = 0.3
LR = 2e-3
HIDDEN = 64

_CTX = []


def context():
    """One context for the process, as a single-threaded program has it."""
    if not _CTX:
        _CTX.append(M.Context(0))
    return _CTX[0]


# --- the cases -----------------------------------------------------------------


def listed():
    return [
        # Interactive lookup: who is reached from one vertex in three steps (launch latency).
        {"name": "walk_one_source", "kind": "walk", "graph": 1, "n_vertices": 1 << 16, "sources": 1,
         "hops": 3, "result": "frontier"},
        # An ordinary query of the uneven mix (sizes log-uniform in 1..4096), ragged graph.
        {"name": "walk_300_sources", "kind": "walk", "graph": 2, "n_vertices": 200003, "sources": 300,
         "hops": 5, "result": "export"},
        # A large query below the full panel, on the mix's largest graph.
        {"name": "walk_1500_sources", "kind": "walk", "graph": 3, "n_vertices": 1 << 20, "sources": 1500,
         "hops": 6, "result": "export"},
        # The headline walk: 4096 sources, 4 hops, scale 22.
        {"name": "walk_4096_sources", "kind": "walk", "graph": 4, "n_vertices": 1 << 22, "sources": 4096,
         "hops": 4, "result": "export"},
        # A service's queries of several users in one captured launch sequence.
        {"name": "batch_16_queries", "kind": "batch", "graph": 5, "scale": 16, "graphs": 3, "queries": 16},
        # PPRQuery's product of a small graph with itself.
        {"name": "square_scale_14", "kind": "square", "graph": 6, "n_vertices": 1 << 14, "communities": 0,
         "min_bits": 0},
        # The same of a graph with planted dense communities, dense tile pairs on the matrix cores.
        {"name": "square_communities", "kind": "square", "graph": 7, "n_vertices": 1 << 16, "communities": 16,
         "min_bits": 128},
        # One hop of a product walk with pruned frontiers, output sized by the cost model.
        {"name": "pruned_hop", "kind": "pruned", "graph": 8, "n_vertices": 1 << 18, "sources": 1000},
        # Loading a user's graph: host edge list to device tiles, ragged size.
        {"name": "ingest_300k_vertices", "kind": "ingest", "graph": 9, "n_vertices": 300007},
        # Two-hop pairs of a small graph, as the enumerating walk gives them.
        {"name": "two_hop_scale_13", "kind": "two_hop", "graph": 10, "n_vertices": 1 << 13},
        # Scheduler predictions for the chunks of a large batch.
        {"name": "predict_200k_rows", "kind": "predict", "rows": 200003},
        # Fine-tuning the cost model on freshly logged samples.
        {"name": "train_8k_rows", "kind": "train", "rows": 8000, "batch": 4096},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["walk", "walk", "walk", "batch", "square", "pruned", "ingest", "two_hop", "predict", "train"])
    if kind == "predict":
        return {"kind": kind, "rows": _log_uniform(rng, 100, 1 << 20)}
    if kind == "train":
        batch = rng.choice([512, 1024, 4096, 16384])
        return {"kind": kind, "rows": rng.randint(batch + 1, 2 * batch), "batch": batch}
    case = {"kind": kind, "graph": rng.randint(100, 1 << 20)}
    if kind == "walk":
        n = _log_uniform(rng, 1 << 12, 1 << 20)
        sources = min(n // 4, _log_uniform(rng, 1, 4096))
        return dict(case, n_vertices=n, sources=sources, hops=rng.randint(1, 6),
                    result=rng.choice(["frontier", "export"]) if n * sources <= 1 << 26 else "export")
    if kind == "batch":
        return dict(case, scale=rng.randint(13, 17), graphs=rng.randint(1, 4), queries=rng.randint(2, 16))
    if kind == "square":
        dense = rng.choice([False, True])
        n = _log_uniform(rng, 1 << 13 if dense else 1 << 10, 1 << 16)
        return dict(case, n_vertices=n, communities=rng.randint(1, n // (4 * COMMUNITY_SIZE)) if dense else 0,
                    min_bits=rng.choice([64, 128, 512]) if dense else 0)
    if kind == "pruned":
        return dict(case, n_vertices=_log_uniform(rng, 1 << 13, 1 << 18), sources=_log_uniform(rng, 1, 2048))
    if kind == "ingest":
        return dict(case, n_vertices=_log_uniform(rng, 1 << 10, 1 << 19))
    return dict(case, n_vertices=_log_uniform(rng, 1 << 8, 1 << 13))


# --- inputs --------------------------------------------------------------------
# A case's graph is fixed by its "graph" number. The seed names its vertices: ids rotate within
# every block of 64, so that another seed's inputs and results differ while tile sets, pair
# counts and work stay those of the case.


def _rename(ids, n, seed):
    """ids (int64, on the GPU) with the names that `seed` gives; a last partial block keeps its own."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    turn = torch.randint(0, M.TILE, (-(-n // M.TILE),), generator=g, device="cuda")
    if n % M.TILE:
        turn[-1] = 0
    return (ids & ~(M.TILE - 1)) | ((ids + turn[ids >> 6]) & (M.TILE - 1))


def _host_ids(ids):
    return ids.to(torch.int32).cpu().numpy().view(np.uint32)


def _graph(n, graph, kind="rmat", communities=0):
    """(src, dst) of the case's graph before renaming: duplicates kept, self-loops removed."""
    g = torch.Generator(device="cuda").manual_seed(graph)
    if kind == "er":
        src, dst = (torch.randint(0, n, (32 * n,), generator=g, device="cuda") for _ in range(2))
    else:
        src = torch.zeros(EDGE_FACTOR * n, dtype=torch.int64, device="cuda")
        dst = torch.zeros_like(src)
        a, b, c, _ = ABCD
        for _ in range(max(1, (n - 1).bit_length())):
            r = torch.rand(src.shape, generator=g, device="cuda")
            src = 2 * src + (r >= a + b)
            dst = 2 * dst + (((r >= a) & (r < a + b)) | (r >= a + b + c))
        src, dst = src % n, dst % n
    parts = [(src, dst)]
    for k in range(communities):
        inside = torch.rand(COMMUNITY_SIZE, COMMUNITY_SIZE, generator=g, device="cuda") < COMMUNITY_P
        u, v = inside.nonzero(as_tuple=True)
        first = k * (n // communities // M.TILE * M.TILE)
        parts.append((u + first, v + first))
    src, dst = (torch.cat(p) for p in zip(*parts))
    keep = src != dst
    return src[keep], dst[keep]


def _upload(n, edges, seed):
    src, dst = (_host_ids(_rename(v, n, seed)) for v in edges)
    return M.EdgeList.upload(context(), n, src, dst)


def _sources(n, edges, count, graph, seed):
    """Distinct source vertices: a lookup of a few names vertices that have edges, a large query
    samples the whole vertex range."""
    if count > 64:
        ids = torch.from_numpy(M.sample_sources(n, count, graph).astype(np.int64)).cuda()
    else:
        g = torch.Generator(device="cuda").manual_seed(graph)
        with_edges = torch.unique(edges[0])
        ids = with_edges[torch.randperm(len(with_edges), generator=g, device="cuda")[:count]]
    return _host_ids(_rename(ids, n, seed))


def _features(rows, seed):
    rng = np.random.default_rng(seed)
    x = rng.uniform(0.0, 1.2, (rows, LN.N_FEATURES)).astype(np.float32)
    t = np.stack([0.5 * x[:, 0] + 0.2 * x[:, 1] * x[:, 4], np.clip(x[:, 3] - 0.1 * x[:, 5], 0, 1)], 1)
    return x, (t + rng.normal(0, 0.02, t.shape)).astype(np.float32)


def _weights(n_in, n_out, seed, bias=0.0):
    """FP32 masters of an n_in -> 64 -> 64 -> n_out network in the library's layout."""
    rng = np.random.default_rng(seed + 1)
    he = lambda rows, fan: rng.uniform(-1, 1, rows * fan) * math.sqrt(6.0 / fan)  # noqa: E731
    parts = [he(HIDDEN, n_in), np.zeros(HIDDEN), he(HIDDEN, HIDDEN), np.zeros(HIDDEN),
             he(n_out, HIDDEN) * (0.02 if bias else 1.0), np.full(n_out, bias)]
    return np.concatenate(parts).astype(np.float32)


def _model(n_in, n_out, seed, bias=0.0):
    mlp = M.MLP(context(), n_in, n_out, seed=1)
    mlp.set_params(_weights(n_in, n_out, seed, bias))
    return mlp


def prepare(case, seed):
    ctx, kind = context(), case["kind"]
    state = {"kind": kind, "case": dict(case)}
    if kind in ("predict", "train"):
        state["x"], state["t"] = _features(case["rows"], seed)
        state["model"] = _model(LN.N_FEATURES, LN.N_TARGETS, seed)
        return state
    if kind == "batch":
        specs = [WL.GraphSpec("er" if i == 2 else "rmat", case["scale"] + i % 3, case["graph"] + i)
                 for i in range(case["graphs"])]
        graphs, queries = [], WL.batch_queries(specs, case["queries"], case["graph"])
        for s in specs:
            el = _upload(s.n_vertices, _graph(s.n_vertices, s.seed, s.kind), seed)
            graphs.append(el.to_tiled_matrix(transpose=True))
            el.close()
        for q in queries:
            ids = torch.from_numpy(q.sources.astype(np.int64)).cuda()
            q.sources = _host_ids(_rename(ids, specs[q.graph].n_vertices, seed))
        state["batch"] = M.WalkBatch(ctx, graphs, queries)
        return state
    n = case["n_vertices"]
    edges = _graph(n, case["graph"], communities=case.get("communities", 0))
    if kind == "ingest":
        state["src"], state["dst"] = (_host_ids(_rename(v, n, seed)) for v in edges)
        return state
    el = _upload(n, edges, seed)
    if kind == "two_hop":
        state["edges"] = el
        return state
    at = el.to_tiled_matrix(transpose=True)
    if kind == "walk":
        state["walk"] = M.Walk(ctx, at, case["sources"], case["hops"])
        state["sources"] = _sources(n, edges, case["sources"], case["graph"], seed)
    elif kind == "square":
        state["a"], state["at"] = el.to_tiled_matrix(transpose=False), at
    else:
        at.prepare_operand()
        x0 = WL.sources_matrix(ctx, n, _sources(n, edges, case["sources"], case["graph"], seed))
        state["x"], state["at"] = M.multiply_pruned(ctx, x0, at)[0], at
        state["model"] = _model(M.ROW_FEATURES, LN.ROW_TARGETS, seed, bias=0.6)
    el.close()
    return state


# --- one pass --------------------------------------------------------------------


class _Array:
    """A device array of a tile matrix, which it keeps alive, for torch.as_tensor."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": typestr, "version": 2}


def _tensors(m):
    """The four arrays of a device tile matrix, without a copy."""
    strips, tiles, _ = m.metadata()
    names, shapes = ("offset", "row", "col", "data"), ((strips + 1,), (tiles,), (tiles,), (tiles, M.TILE))
    out = {}
    for name, shape, ptr in zip(names, shapes, m.device_arrays()):
        kind = "<i8" if name == "data" else "<i4"
        out[name] = (torch.as_tensor(_Array(m, ptr, shape, kind), device="cuda") if shape[0]
                     else torch.zeros(shape, dtype=torch.int64 if name == "data" else torch.int32, device="cuda"))
    return out


def run(state):
    ctx, kind, case = context(), state["kind"], state["case"]
    if kind == "walk":
        w = state["walk"]
        w.run(state["sources"], case["hops"])
        return w.frontier(case["hops"]).view(np.int64) if case["result"] == "frontier" else _tensors(w.export(case["hops"]))
    if kind == "batch":
        b = state["batch"]
        b.run()
        return [_tensors(b.query_export(q)) for q in range(case["queries"])]
    if kind == "square":
        c, _ = M.multiply_symbolic(ctx, state["a"], state["at"])
        if case["min_bits"]:
            M.multiply_numeric_dense(ctx, state["a"], state["at"], c, case["min_bits"])
        else:
            M.multiply_numeric(ctx, state["a"], state["at"], c)
        return _tensors(c)
    if kind == "pruned":
        c, _, predicted = M.multiply_pruned_model(ctx, state["x"], state["at"], state["model"])
        return dict(_tensors(c), predicted=predicted)
    if kind == "ingest":
        el = M.EdgeList.upload(ctx, case["n_vertices"], state["src"], state["dst"])
        at = el.to_tiled_matrix(transpose=True)
        el.close()
        return _tensors(at)
    if kind == "two_hop":
        pairs = state["edges"].two_hop()
        src, dst = pairs.download()
        pairs.close()
        return [src.view(np.int32), dst.view(np.int32)]
    if kind == "predict":
        return state["model"].forward(state["x"])
    loss = state["model"].train(state["x"], state["t"], epochs=1, batch=case["batch"], lr=LR)
    return {"loss": loss, "weights": state["model"].params()[0]}


# --- what a pass cannot do without -------------------------------------------------


def _rmat_tiles(n):
    """Expected edges and occupied 64 x 64 tiles of an R-MAT graph on about n vertices: a tile
    is a path of log2(n / 64) quadrant choices, so the sum runs over the choices' counts."""
    edges, levels = float(EDGE_FACTOR * n), max(0, round(math.log2(max(64, n) / 64)))
    tiles = 0.0
    for i in range(levels + 1):
        for j in range(levels - i + 1):
            for k in range(levels - i - j + 1):
                rest = levels - i - j - k
                ways = math.comb(levels, i) * math.comb(levels - i, j) * math.comb(levels - i - j, k)
                p = ABCD[0] ** i * ABCD[1] ** j * ABCD[2] ** k * ABCD[3] ** rest
                tiles += ways * -math.expm1(-edges * p)
    return edges, tiles


def _words(sources):
    return -(-sources // 64)


def _mlp_flops(rows, n_in, n_out):
    return 2.0 * rows * (n_in * HIDDEN + HIDDEN * HIDDEN + HIDDEN * n_out)


def work(case):
    """Bytes: inputs read and outputs written once. A walk reads each edge (4 bytes) once a hop
    and X_k, and writes X_{k+1}; a product reads the tiles (520 bytes with their index) of its
    operands and writes those of C. Operations: one per word ORed, tile word pair tested or
    multiply and add."""
    kind = case["kind"]
    n = case.get("n_vertices", 0)
    if kind == "walk":
        edges, _ = _rmat_tiles(n)
        w = _words(case["sources"])
        return {"bytes": case["hops"] * (4 * edges + 16.0 * n * w) + 16.0 * n * w, "flops": case["hops"] * edges * w}
    if kind == "batch":
        # Mean query: 490 sources (8 words), 3.5 hops; the hops of one graph share its edges.
        n = 1 << case["scale"]
        edges = EDGE_FACTOR * 2.0 * n
        per_query = 3.5 * 16.0 * 2 * n * 8
        return {"bytes": case["graphs"] * 6 * 4 * edges + case["queries"] * per_query,
                "flops": case["queries"] * 3.5 * edges * 8}
    if kind == "square":
        strips = -(-n // 64)
        _, tiles = _rmat_tiles(n)
        tiles += case["communities"] * (COMMUNITY_SIZE // 64) ** 2
        return {"bytes": 520.0 * (2 * tiles + strips * strips), "flops": 64.0 * tiles * tiles / max(1, strips)}
    if kind == "pruned":
        strips, rows = -(-n // 64), _words(case["sources"])
        _, tiles = _rmat_tiles(n)
        return {"bytes": 520.0 * (rows * strips + tiles), "flops": 64.0 * rows * tiles}
    if kind == "ingest":
        edges, tiles = _rmat_tiles(n)
        return {"bytes": 8 * edges + 520.0 * tiles, "flops": 0}
    if kind == "two_hop":
        edges, _ = _rmat_tiles(n)
        pairs = min(0.2 * n * n, 64.0 * edges)
        return {"bytes": 8 * edges + 8 * pairs, "flops": 16.0 * edges}
    n_in, n_out = LN.N_FEATURES, LN.N_TARGETS
    rows = case["rows"]
    if kind == "predict":
        return {"bytes": 4.0 * rows * (n_in + n_out), "flops": _mlp_flops(rows, n_in, n_out)}
    return {"bytes": 4.0 * rows * (n_in + n_out), "flops": 4 * _mlp_flops(rows, n_in, n_out)}


# --- 64-bit values -------------------------------------------------------------------


def _split(w, n_in, n_out):
    """The six parameter arrays of a flat parameter vector."""
    sizes = [(HIDDEN, n_in), (HIDDEN,), (HIDDEN, HIDDEN), (HIDDEN,), (n_out, HIDDEN), (n_out,)]
    out, at = [], 0
    for s in sizes:
        count = math.prod(s)
        out.append(w[at:at + count].reshape(s))
        at += count
    return out


def _bf16(w):
    """The BF16 weights (rounded to nearest even from FP32 masters) in 64 bits."""
    return w.to(torch.float32).to(torch.bfloat16).to(torch.float64)


def _network(w, n_in, n_out, x):
    w1, b1, w2, b2, w3, b3 = _split(w, n_in, n_out)
    h1 = torch.relu(x @ w1.T + b1)
    return torch.relu(h1 @ w2.T + b2) @ w3.T + b3


def _exact_train(case, seed):
    """Adam on the mean squared error over the batches in order, then the loss over all rows."""
    x, t = (torch.from_numpy(v).cuda().double() for v in _features(case["rows"], seed))
    dims = (LN.N_FEATURES, LN.N_TARGETS)
    w = torch.from_numpy(_weights(*dims, seed)).cuda().double()
    m, v = torch.zeros_like(w), torch.zeros_like(w)
    f = np.float32
    b1, b2, lr, eps = (float(f(c)) for c in (0.9, 0.999, LR, 1e-8))
    for step, at in enumerate(range(0, case["rows"], case["batch"]), 1):
        q = _bf16(w).requires_grad_(True)
        y = _network(q, *dims, x[at:at + case["batch"]])
        (g,) = torch.autograd.grad((y - t[at:at + case["batch"]]).square().mean(), q)
        m = b1 * m + float(f(1) - f(0.9)) * g
        v = b2 * v + float(f(1) - f(0.999)) * g * g
        c1, c2 = float(f(1) - f(0.9) ** f(step)), float(f(1) - f(0.999) ** f(step))
        w = w - lr * (m / c1) / ((v / c2).sqrt() + eps)
    loss = (_network(_bf16(w), *dims, x) - t).square().mean()
    return {"loss": float(loss), "weights": w.cpu().numpy()}


def _exact_prediction(case, seed):
    """Per row of C: structural tiles times the model's clamped output on the row's features."""
    state = prepare(case, seed)
    x, at = state["x"].download(), state["at"].download()
    n = x.n_strips

    def counts(m):
        return torch.from_numpy(np.bitwise_count(m.data).sum(1).astype(np.float64)).cuda()

    ab, bb = counts(x), counts(at)
    ar, ac, br, bc = (torch.from_numpy(v.astype(np.int64)).cuda() for v in (x.row_idx, x.col_idx, at.row_idx, at.col_idx))
    rows = int(x.row_idx.max()) + 1 if len(x.row_idx) else 1
    pa = torch.zeros(rows, n, device="cuda")
    pa[ar, ac] = 1
    pb = torch.zeros(n, n, device="cuda")
    pb[bc, br] = 1
    z = torch.zeros(n, dtype=torch.float64, device="cuda")
    cnt = z.clone()
    cnt[:rows] = ((pa @ pb) > 0).sum(1).double()
    b_tiles, b_bits = z.index_add(0, bc, torch.ones_like(bb)), z.index_add(0, bc, bb)
    tp, bbits = z.index_add(0, ar, b_tiles[ac]), z.index_add(0, ar, b_bits[ac])
    nt, abits = z.index_add(0, ar, torch.ones_like(ab)), z.index_add(0, ar, ab)
    mean = lambda s, c: torch.where(c > 0, s / c.clamp(min=1), z)  # noqa: E731
    f = torch.stack([cnt.log1p() / 16, tp.log1p() / 20, nt.log1p() / 16, abits.log1p() / 20, bbits.log1p() / 24,
                     mean(abits, nt).log1p() / 8, mean(bbits, tp).log1p() / 8, cnt / n], 1)
    dims = (M.ROW_FEATURES, LN.ROW_TARGETS)
    w = _bf16(torch.from_numpy(_weights(*dims, seed, 0.6)).cuda())
    return (cnt * _network(w, *dims, f)[:, 0].clamp(0, 1)).cpu().numpy()


def exact(case, seed):
    """The floating outputs in 64 bits; Boolean results and tile indices are whole numbers."""
    if case["kind"] == "predict":
        x = torch.from_numpy(_features(case["rows"], seed)[0]).cuda().double()
        dims = (LN.N_FEATURES, LN.N_TARGETS)
        return _network(_bf16(torch.from_numpy(_weights(*dims, seed)).cuda()), *dims, x).cpu().numpy()
    if case["kind"] == "train":
        return _exact_train(case, seed)
    if case["kind"] == "pruned":
        return {"predicted": _exact_prediction(case, seed), "offset": None, "row": None, "col": None, "data": None}
    return None
