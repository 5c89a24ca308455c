"""Default BFS where narrow levels (run by the workgroup that ends a level)
meet wide ones: frontiers of 4096 edges and one more, hubs that end a narrow
run, returns to narrow levels, more levels than one launch runs, sources
without neighbours.  Levels equal the serial oracle's (bfs_vertex_omp.h)."""
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


def _fan(width):
    """a root with `width` chains of 5: levels of exactly 2 * width edges"""
    pairs = [(np.zeros(width, np.int32), 1 + np.arange(width))]
    for k in range(4):
        pairs.append((1 + k * width + np.arange(width), 1 + (k + 1) * width + np.arange(width)))
    return _edges(1 + 5 * width, pairs, f"fan{width}")


CASES = {
    "path": (lambda: _path(3001), [0, 1500, 3000]),
    "grid": (lambda: G.grid2d(301, 0.0, seed=1), [0, 45150]),
    "grid_long": (lambda: G.grid2d(200, 0.02, seed=2), [7]),
    "hub_below": (lambda: _hubs(4094), [0, 41, 4800]),
    "hub_at": (lambda: _hubs(4095), [0, 40]),
    "hub_above": (lambda: _hubs(4097), [0, 40]),
    "hub_wide": (lambda: _hubs(70000), [0, 70000]),
    "fan_at": (lambda: _fan(2048), [0, 5]),
    "fan_above": (lambda: _fan(2049), [0, 5]),
    "isolated": (lambda: G.from_edges(70, np.array([1, 2], np.int32), np.array([2, 3], np.int32), "iso"), [0, 1, 69]),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_narrow_and_wide_levels(gpu, name):
    make, sources = CASES[name]
    g = make()
    with gpu.DeviceGraph(g) as dg:
        for src in sources:
            for _ in range(2):  # the second run starts from the first one's bitmaps and queues
                assert np.array_equal(gpu.run("bfs", dg, "do_hybrid", src).out, O.bfs_serial(g, src)), (name, src)
