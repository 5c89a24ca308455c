"""Batched BFS, CC and MIS on graphs at the edges of their kernels: one vertex,
isolated vertices, self loops left out, stars (rows longer than the 1024 edges
that one wave walks, inside and outside the sampled component), paths (many
levels), complete graphs (long rows in every MIS round), rows of 32 and 33
edges, sizes around the workgroup's, and a disconnected source.  Results equal
the oracle's."""
import numpy as np
import pytest

import oracle as O
from indigo2suite_amd import batched as BT
from indigo2suite_amd import graph as G

pytestmark = pytest.mark.gpu


def _star(n, centre=0):
    leaves = np.delete(np.arange(n), centre).astype(np.int32)
    return G.from_edges(n, np.full(n - 1, centre, np.int32), leaves, f"star{n}")


def _stars(k, leaves):
    c = np.repeat(np.arange(k), leaves) * (leaves + 1)
    v = c + np.tile(np.arange(1, leaves + 1), k)
    return G.from_edges(k * (leaves + 1), c.astype(np.int32), v.astype(np.int32), f"stars{k}x{leaves}")


def _complete(n):
    a, b = np.triu_indices(n, 1)
    return G.from_edges(n, a.astype(np.int32), b.astype(np.int32), f"K{n}")


def _path(n):
    return G.from_edges(n, np.arange(n - 1, dtype=np.int32), np.arange(1, n, dtype=np.int32), f"path{n}")


def _graphs():
    gs = [G.Graph(np.zeros(2, np.int32), np.zeros(0, np.int32), None, "one"),
          G.Graph(np.zeros(301, np.int32), np.zeros(0, np.int32), None, "isolated"),
          _star(3000), _star(1500, 1499), _stars(5, 1100), _stars(40, 33), _stars(40, 32), _path(1300),
          _complete(33), _complete(34), _complete(300)]
    for n in (255, 256, 257, 1023, 1024, 1025, 4097):
        gs.append(G.erdos_renyi(n, 6.0, seed=n))
    gs.append(G.rmat(14, 24, seed=3, n_limit=12001))
    gs.append(G.rmat(13, 3, seed=4))          # many small components, vertex 0 in the large one
    gs.append(G.grid2d(70, 0.0, seed=5))
    gs.append(G.from_edges(5000, np.arange(1, 4999, dtype=np.int32), np.arange(2, 5000, dtype=np.int32), "off_source"))
    gs.append(G.chung_lu(9000, 12.0, 2.2, seed=6))
    return gs


@pytest.fixture(scope="module")
def batch(gpu):
    gs = _graphs()
    refs = {"bfs": [O.bfs_serial(g, 0) for g in gs], "cc": [O.cc_omp_pull(g)[0] for g in gs],
            "mis": [O.mis_greedy(g).astype(np.int32) for g in gs]}
    with BT.DeviceBatch(gs) as db:
        yield gs, db, refs


@pytest.mark.parametrize("block", [256, 512, 1024])
def test_shapes(gpu, batch, block):
    gs, db, refs = batch
    for use_graph in (False, True):
        db.run(7, block, use_graph)
        for algo in ("bfs", "cc", "mis"):
            for g, out, ref in zip(gs, db.results(algo), refs[algo]):
                assert np.array_equal(out, ref), (algo, g.name, block)
