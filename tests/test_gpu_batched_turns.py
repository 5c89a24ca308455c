"""The batched BFS where it turns: frontiers at and around a 24th of the
vertices and an edge a vertex, levels after which no vertex with an edge is
left, graphs too small for either, meshes and paths that stay top-down and
power laws that do not.  Levels, components and sets against the oracle."""
import numpy as np
import pytest

import oracle as O
from indigo2suite_amd import batched, graph as G

pytestmark = pytest.mark.gpu


def _path(n):
    v = np.arange(n - 1, dtype=np.int32)
    return G.from_edges(n, v, v + 1, f"path{n}")


def _star(n, tail=0):
    """vertex 0 joined to n - 1 others, the last of which starts a path of `tail` more"""
    v = np.arange(1, n, dtype=np.int32)
    t = np.arange(n - 1, n - 1 + tail, dtype=np.int32)
    return G.from_edges(n + tail, np.r_[np.zeros(n - 1, np.int32), t], np.r_[v, t + 1], f"star{n}_{tail}")


def _levels(width, depth):
    """vertex 0, then `depth` levels of `width` vertices, each joined to the next level's same and next place"""
    ids = 1 + np.arange(width * depth, dtype=np.int32).reshape(depth, width)
    a = [np.zeros(width, np.int32)] + [np.r_[ids[k], ids[k]] for k in range(depth - 1)]
    b = [ids[0]] + [np.r_[ids[k + 1], np.roll(ids[k + 1], 1)] for k in range(depth - 1)]
    return G.from_edges(1 + width * depth, np.concatenate(a), np.concatenate(b), f"levels{width}_{depth}")


GRAPHS = [
    _path(2), _path(23), _path(24), _path(1500), _star(2), _star(24), _star(5000), _star(3000, 40),
    G.grid2d(64, 0.0, seed=1), G.grid2d(80, 0.05, seed=2),
    *[_levels(w, d) for w in (40, 41, 42, 43) for d in (23, 24, 25)],
    G.erdos_renyi(3000, 3.0, seed=3), G.erdos_renyi(3000, 40.0, seed=4), G.rmat(12, 16, seed=5),
    G.Graph(np.zeros(2, np.int32), np.zeros(0, np.int32), None, "single"),
    G.Graph(np.zeros(31, np.int32), np.zeros(0, np.int32), None, "edgeless"),
]


@pytest.mark.parametrize("block", [256, 512, 1024])
def test_against_the_oracle(gpu, block):
    with batched.DeviceBatch(GRAPHS) as db:
        db.run(7, block, use_graph=False)
        got = {k: db.results(k) for k in ("bfs", "cc", "mis")}
    for i, g in enumerate(GRAPHS):
        assert np.array_equal(got["bfs"][i], O.bfs_serial(g, 0)), g.name
        assert np.array_equal(got["cc"][i], O.cc_omp_pull(g)[0]), g.name
        assert np.array_equal(got["mis"][i], O.mis_greedy(g).astype(np.int32)), g.name
