"""MIS default style at the edges of its kernel: first neighbours at once (4),
walks of 8 at once up to 32 more, walks by the wave beyond, rows of at most and
above the 1024 edges that a wave excludes by itself, a long run of rounds (a
path whose priorities alternate at random), self loops, isolated vertices.
The set equals the greedy one of the unsigned hash order
(mis_vertex_omp.h:127-132)."""
import numpy as np
import pytest

import oracle as O
from indigo2suite_amd import graph as G

pytestmark = pytest.mark.gpu


def _priority(v):
    x = (np.asarray(v, np.uint64) + np.uint64(712313887)) & np.uint64(0xFFFFFFFF)
    for _ in range(2):
        x = (((x >> np.uint64(16)) ^ x) * np.uint64(0x45D9F3B)) & np.uint64(0xFFFFFFFF)
    return (x >> np.uint64(16)) ^ x


def _star_at(n, top):
    """a star whose centre has the highest (it joins first) or the lowest priority (it is walked to the end)"""
    p = _priority(np.arange(n))
    c = int(np.argmax(p) if top else np.argmin(p))
    leaves = np.delete(np.arange(n), c).astype(np.int32)
    return G.from_edges(n, np.full(n - 1, c, np.int32), leaves, f"star{n}_{top}")


def _complete(n):
    a, b = np.triu_indices(n, 1)
    return G.from_edges(n, a.astype(np.int32), b.astype(np.int32), f"K{n}")


def _loops():
    return G.Graph(np.array([0, 2, 4, 5, 5]), np.array([0, 1, 0, 1, 2]), None, "loops")


CASES = {f"star{n}_{'top' if t else 'low'}": (lambda n=n, t=t: _star_at(n, t))
         for n in (5, 6, 37, 38, 1025, 1026, 70000) for t in (True, False)}
CASES.update({
    "K5": lambda: _complete(5), "K37": lambda: _complete(37), "K1026": lambda: _complete(1026),
    "path": lambda: G.from_edges(5001, np.arange(5000, dtype=np.int32), np.arange(1, 5001, dtype=np.int32), "path"),
    "loops": _loops,
    "rmat": lambda: G.rmat(15, 20, seed=9, n_limit=30001),
    "one": lambda: G.Graph(np.zeros(2, np.int32), np.zeros(0, np.int32), None, "one"),
})


@pytest.mark.parametrize("name", sorted(CASES))
def test_greedy_set(gpu, name):
    g = CASES[name]()
    with gpu.DeviceGraph(g) as dg:
        for _ in range(2):
            assert np.array_equal(gpu.run("mis", dg, "v_resume_pull").out, O.mis_greedy(g).astype(np.int32)), name
