"""PageRank's balanced style on both sides of its renumbering rule: graphs
whose 16384 vertices of highest degree take at least a quarter of the edges
(worked on in degree order) and graphs where they do not, ragged sizes,
isolated vertices, rows of one and of several chunks, and iteration limits
around the first batch of iterations, after which kernels without work are
left out.  Scores within 1e-5 relative of the FP64 oracle at the same
iteration count (the bound of every style), iteration counts equal to the
thread-per-vertex style's, which works on the graph as given."""
import numpy as np
import pytest

import oracle as O
from indigo2suite_amd import graph as G

pytestmark = pytest.mark.gpu

RTOL = 1e-5


def _star(n, hubs):
    """`hubs` centres, every other vertex joined to one of them and its successor; the last 100 isolated"""
    v = np.arange(hubs, n - 100, dtype=np.int32)
    return G.from_edges(n, np.r_[v, v[:-1]], np.r_[(v % hubs).astype(np.int32), v[1:]], f"star{n}_{hubs}")


CASES = {
    "below_size": lambda: G.rmat(15, 16, seed=2, n_limit=32767),
    "at_size": lambda: G.rmat(15, 16, seed=2),
    "ragged": lambda: G.rmat(17, 12, seed=3, n_limit=70001),
    "one_hub": lambda: _star(40000, 1),
    "many_hubs": lambda: _star(60011, 300),
    "flat": lambda: G.erdos_renyi(200003, 9.0, seed=4),
    "mesh": lambda: G.grid2d(200, 0.05, seed=5),
    "edgeless": lambda: G.Graph(np.zeros(40001, np.int32), np.zeros(0, np.int32), None, "edgeless"),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_scores_and_iterations(gpu, name):
    g = CASES[name]()
    try:
        with gpu.DeviceGraph(g) as dg:
            for eps, limit in ((1e-6, 100), (0.0, 1), (0.0, 4), (0.0, 5), (0.0, 13)):
                gpu.set_pr_params(eps, limit)
                r = gpu.run("pr", dg, "pull_balanced_kahan")
                t = gpu.run("pr", dg, "pull_thread_kahan")
                assert r.iterations == t.iterations, (name, eps, limit)
                ref, _, _ = O.pr_fp64(g, eps, limit, fixed_iters=r.iterations)
                assert np.max(np.abs(r.out - ref) / ref) <= RTOL, (name, eps, limit)
    finally:
        gpu.set_pr_params(1e-4, 100)
