"""The graph work that is measured: each case is one call of a public entry
point on one graph (or one batch of graphs), as a program keeps it on the GPU.

The listed cases are the workloads of this repository's benchmark and tests at
their own sizes: BFS on a small Erdos-Renyi graph through the drop-in entry,
the six kernels on R-MAT 22 / R-MAT 20, PageRank on the 2048 x 2048 grid, the
edge-based SSSP style, a BFS of thousands of narrow levels, and a batch of
uneven graphs.  `draw` spreads the same kinds of graphs over their whole range of
sizes, degrees and shapes.

A case's graph comes from `family`:
  er       Erdos-Renyi, `n` vertices, average degree `degree`
  rmat     R-MAT (0.57, 0.19, 0.19, 0.05), `n` vertices (samples beyond n are
           dropped when n is no power of two), average degree `degree`
  grid     `side` x `side` mesh, a share `long` of the vertices with one
           long-range edge
  chunglu  Chung-Lu power law, `n`, `degree`, exponent `gamma`
  batch    `graphs` of them, half er and half rmat, vertices log-uniform in
           [2^10, 2^hi], average degree in [4, 32]
"""
import ctypes
import math

import numpy as np
import torch

from indigo2suite_amd import batched, device, graph

PR_EPS = 1e-6      # PageRank: L1 change of the last iteration
PR_MAX_ITER = 100


def listed():
    return [
        # the smallest call: one BFS of a small graph through the drop-in
        # entry, levels back in host memory; latency and launches count
        {"name": "bfs_er16k_entry", "algo": "bfs", "family": "er", "n": 16384, "degree": 8.0, "entry": True},
        # the benchmark's graph: power law, 128 M directed edges
        {"name": "bfs_rmat22", "algo": "bfs", "family": "rmat", "n": 1 << 22, "degree": 32.0},
        {"name": "sssp_rmat22", "algo": "sssp", "family": "rmat", "n": 1 << 22, "degree": 32.0},
        {"name": "cc_rmat22", "algo": "cc", "family": "rmat", "n": 1 << 22, "degree": 32.0},
        {"name": "mis_rmat22", "algo": "mis", "family": "rmat", "n": 1 << 22, "degree": 32.0},
        # a mesh or road-like graph: thousands of narrow levels
        {"name": "bfs_grid1024", "algo": "bfs", "family": "grid", "side": 1024, "long": 0.0},
        # the edge-based, data-driven SSSP style with the caller's sp[]
        {"name": "sssp_edge_rmat20", "algo": "sssp", "family": "rmat", "n": 1 << 20, "degree": 32.0,
         "style": "e_data_push_thread"},
        # PageRank and triangle counting: a power law, and a graph of short
        # rows of much the same length
        {"name": "pr_rmat20", "algo": "pr", "family": "rmat", "n": 1 << 20, "degree": 32.0},
        {"name": "pr_grid2048", "algo": "pr", "family": "grid", "side": 2048, "long": 0.05},
        {"name": "tc_rmat20", "algo": "tc", "family": "rmat", "n": 1 << 20, "degree": 32.0},
        {"name": "tc_er2m", "algo": "tc", "family": "er", "n": 1 << 21, "degree": 16.0},
        # many uneven graphs in one persistent launch: BFS, CC and MIS of each
        {"name": "batch128", "algo": "batch", "family": "batch", "graphs": 128, "hi": 17, "block": 1024},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    algo = rng.choice(["bfs", "sssp", "sssp", "cc", "mis", "pr", "tc", "batch"])
    if algo == "batch":
        return {"algo": algo, "family": "batch", "graphs": _log_int(rng, 8, 128), "hi": rng.randint(12, 16),
                "block": rng.choice([256, 512, 1024])}
    # (a mesh holds next to no triangles: no case of its own for counting them)
    family = rng.choice(["er", "rmat", "chunglu"] if algo == "tc" else ["er", "rmat", "rmat", "grid", "chunglu"])
    case = {"algo": algo, "family": family}
    if algo == "sssp" and rng.random() < 0.5:
        case["style"] = "e_data_push_thread"
    if algo in ("bfs", "cc", "mis") and rng.random() < 0.3:
        case["entry"] = True
    if family == "grid":
        # a narrow grid's SSSP and BFS cost grows with its diameter
        case["side"] = _log_int(rng, 32, 512 if algo == "sssp" else 1024)
        case["long"] = rng.choice([0.0, 0.05])
        return case
    big = (1 << 19) if algo == "tc" or "style" in case else (1 << 21)
    case["n"] = _log_int(rng, 1 << (12 if algo == "tc" else 10), big)
    if rng.random() < 0.3:
        case["n"] = 1 << (case["n"].bit_length() - 1)  # powers of two as well as ragged sizes
    case["degree"] = round(rng.uniform(8.0 if algo == "tc" else 4.0, 32.0), 2)
    if family == "chunglu":
        case["gamma"] = round(rng.uniform(2.3, 3.0), 2)
    return case


class _Out:
    """A torch tensor handed to the library as its output buffer."""

    def __init__(self, count, dtype):
        self.t = torch.empty(count, dtype=dtype, device="cuda")
        self.ptr = ctypes.c_void_p(self.t.data_ptr())
        self.nbytes = self.t.numel() * self.t.element_size()

    def free(self):
        pass  # the tensor's own


def _graph(case, seed):
    gs = seed % 1000003 + 1
    if case["family"] == "er":
        return graph.erdos_renyi(case["n"], case["degree"], seed=gs)
    if case["family"] == "rmat":
        n = case["n"]
        scale = max(1, (n - 1).bit_length())
        return graph.rmat(scale, case["degree"] / 2.0, seed=gs, n_limit=n if n < (1 << scale) else 0)
    if case["family"] == "grid":
        return graph.grid2d(case["side"], case["long"], seed=gs)
    return graph.chung_lu(case["n"], case["degree"], case["gamma"], seed=gs)


def _batch(case, seed):
    # the batched workload's recipe: the sizes are the batch's, the edges the seed's
    gs = []
    for i in range(case["graphs"]):
        sizes = np.random.default_rng(1000 + i)
        n = int(round(2.0 ** sizes.uniform(10, case["hi"])))
        part = {"family": "er" if i < case["graphs"] // 2 else "rmat", "n": n, "degree": float(sizes.uniform(4.0, 32.0))}
        gs.append(_graph(part, 1000 * seed + i))
    return gs


def _source(g, case, seed):
    # R-MAT and power laws from the hub, as the benchmark does; elsewhere any
    # vertex that has a neighbour
    if case["family"] in ("rmat", "chunglu"):
        return g.max_degree_vertex()
    has = np.flatnonzero(np.diff(g.nindex) > 0)
    return int(has[np.random.default_rng(seed).integers(has.size)]) if has.size else 0


def prepare(case, seed):
    if case["algo"] == "batch":
        db = batched.DeviceBatch(_batch(case, seed))
        db.graphs = None  # the program keeps the device copy
        for k in list(db.outs):
            db.outs[k].free()
            db.outs[k] = _Out(db.total_nodes, torch.int32)
        return {"case": case, "db": db}
    g = _graph(case, seed)
    src = 0
    if case["algo"] in ("bfs", "sssp"):
        src = _source(g, case, seed)
    if case["algo"] == "sssp":
        g = g.with_weights(1, 255, seed=seed % 1000003 + 1)
    dg = device.DeviceGraph(g)
    dg.host = None  # the program keeps the device copy
    state = {"case": case, "dg": dg, "src": src, "sp": None}
    if case.get("style"):
        state["sp"] = device.build_sp(dg)
    if case["algo"] == "pr":
        device.set_pr_params(PR_EPS, PR_MAX_ITER)
        state["out"] = _Out(g.nodes, torch.float32)
    elif case["algo"] == "tc":
        state["out"] = _Out(1, torch.int64)
    elif not case.get("entry"):
        state["out"] = _Out(g.nodes, torch.int32)
    return state


def run(state):
    case = state["case"]
    algo = case["algo"]
    if algo == "batch":
        db = state["db"]
        db.run(7, case["block"], use_graph=True)
        return {k: v.t for k, v in db.outs.items()}
    dg = state["dg"]
    if case.get("entry"):
        # the drop-in entries: result in host memory
        if algo == "bfs":
            return device.bfs_vertex(state["src"], dg)[0]
        if algo == "cc":
            return device.cc_vertex(dg)[0]
        return list(device.mis_vertex(dg)[:2])
    info = device.run_device(algo, dg, state["out"], case.get("style"), state["src"],
                             state["sp"].ptr if state["sp"] is not None else None)
    if algo == "pr":
        return {"scores": state["out"].t, "iterations": info.iterations}
    return state["out"].t


def _sizes(case):
    """Expected vertices and directed edges."""
    if case["family"] == "grid":
        n = case["side"] ** 2
        return n, 4 * n - 4 * case["side"] + 2 * case["long"] * n
    if case["family"] == "batch":
        lo, hi = 1 << 10, 1 << case["hi"]
        n = case["graphs"] * (hi - lo) / math.log(hi / lo)
        return n, 18.0 * n
    return case["n"], case["degree"] * case["n"] * (0.95 if case["family"] == "rmat" else 1.0)


def work(case):
    # each input read once (offsets, ids, weights), each output written once;
    # PageRank reads its graph and scores once an iteration, for as many
    # iterations as the two families take to this residual
    n, m = _sizes(case)
    algo = case["algo"]
    if algo == "sssp":
        b = 8 * m + 8 * n
    elif algo == "pr":
        iters = 47 if case["family"] == "grid" else 16
        b = iters * (4 * m + 16 * n)
    elif algo == "tc":
        b = 4 * m + 4 * n + 8
    elif algo == "batch":
        b = 3 * (4 * m + 8 * n)  # three algorithms, one pass over each graph for each
    else:
        b = 4 * m + 8 * n
    return {"bytes": float(b), "flops": 0.0}


def exact(case, seed):
    """PageRank in float64 to the same residual; every other result is a whole number."""
    if case["algo"] != "pr":
        return None
    g = _graph(case, seed)
    n = g.nodes
    nindex = torch.from_numpy(g.nindex.astype(np.int64)).cuda()
    nlist = torch.from_numpy(g.nlist).cuda().long()
    deg = nindex[1:] - nindex[:-1]
    rows = torch.repeat_interleave(torch.arange(n, device="cuda"), deg)
    score = torch.full((n,), 1.0 / n, dtype=torch.float64, device="cuda")
    base = (1.0 - 0.85) / n
    iters = 0
    while iters < PR_MAX_ITER:
        contrib = torch.where(deg > 0, score / deg.clamp(min=1), torch.zeros_like(score))
        total = torch.zeros(n, dtype=torch.float64, device="cuda").index_add_(0, rows, contrib[nlist])
        new = base + 0.85 * total
        change = float((new - score).abs().sum())
        score = new
        iters += 1
        if change < PR_EPS:
            break
    return {"scores": score, "iterations": None}
