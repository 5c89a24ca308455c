"""Default SSSP where narrow rounds (run by the workgroup that ends a round)
meet wide ones: frontiers of 4096 edges and one more, hubs that end a narrow
run, more rounds than one launch runs, weights of zero and up to 2^20,
vertices lowered several times in a round, sources without neighbours.
Distances equal the serial oracle's (sssp_edge_omp.h:105-130)."""
import numpy as np
import pytest

import oracle as O
from indigo2suite_amd import graph as G

pytestmark = pytest.mark.gpu


def _edges(n, pairs, name):
    a = np.concatenate([np.asarray(p[0], np.int32) for p in pairs])
    b = np.concatenate([np.asarray(p[1], np.int32) for p in pairs])
    return G.from_edges(n, a, b, name)


def _path(n):
    return _edges(n, [(np.arange(n - 1), np.arange(1, n))], f"path{n}")


def _hubs(leaves):
    """path of 40, a hub with `leaves` leaves, the leaves joined to a second hub, a path of 700"""
    hub, first = 40, 41
    hub2 = first + leaves
    leaf = np.arange(first, first + leaves)
    tail = np.arange(hub2, hub2 + 700)
    return _edges(hub2 + 702, [(np.arange(40), np.arange(1, 41)), (np.full(leaves, hub), leaf),
                               (leaf, np.full(leaves, hub2)), (tail, tail + 1)], f"hubs{leaves}")


def _layers(width, depth):
    """consecutive layers joined completely: every vertex is lowered by many edges in one round"""
    pairs = []
    for d in range(depth - 1):
        a = np.repeat(np.arange(d * width, (d + 1) * width), width)
        b = np.tile(np.arange((d + 1) * width, (d + 2) * width), width)
        pairs.append((a, b))
    return _edges(width * depth, pairs, f"layers{width}x{depth}")


CASES = {
    "path": (lambda: _path(3001), [0, 1500, 3000], (1, 255)),
    "path_zero": (lambda: _path(700), [0], (0, 0)),
    "grid": (lambda: G.grid2d(60, 0.0, seed=1), [0, 1800], (1, 255)),
    "grid_zero": (lambda: G.grid2d(60, 0.0, seed=1), [0], (0, 3)),
    "grid_wide": (lambda: G.grid2d(150, 0.02, seed=2), [7], (1, 255)),
    "grid_heavy": (lambda: G.grid2d(80, 0.02, seed=2), [7], (1, 1 << 20)),
    "hub_below": (lambda: _hubs(4094), [0, 41, 4800], (1, 255)),
    "hub_at": (lambda: _hubs(4095), [0, 40], (1, 255)),
    "hub_above": (lambda: _hubs(4097), [0, 40], (1, 255)),
    "hub_wide": (lambda: _hubs(70000), [0, 70000], (1, 255)),
    "layers": (lambda: _layers(60, 20), [0, 600], (1, 255)),
    "layers_wide": (lambda: _layers(100, 8), [0], (0, 9)),
    "isolated": (lambda: G.from_edges(70, np.array([1, 2], np.int32), np.array([2, 3], np.int32), "iso"), [0, 1, 69],
                 (1, 255)),
    "er": (lambda: G.erdos_renyi(5000, 8.0, seed=3), [1, 2], (1, 255)),
    "rmat": (lambda: G.rmat(14, 16, seed=3), [0, 77], (1, 255)),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_narrow_and_wide_rounds(gpu, name):
    make, sources, (lo, hi) = CASES[name]
    g = make().with_weights(lo, hi, seed=6)
    with gpu.DeviceGraph(g) as dg:
        for src in sources:
            for _ in range(2):  # the second run starts from the first one's bitmaps and queues
                assert np.array_equal(gpu.run("sssp", dg, "v_do_balanced", src).out, O.sssp_serial(g, src)), (name, src)
