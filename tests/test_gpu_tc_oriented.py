"""Triangle counting by the default style at the edges of its kernels: lists
of 32 and 33 (short and long count), rows that cross the 2048-edge tiles of
the flat passes, runs of empty rows, ranks around 16 bits and
beyond the bitmap (hash set), hubs.
Counts are exact, against the serial oracle (tc_vertex_omp.h)."""
import numpy as np
import pytest

import oracle as O
from indigo2suite_amd import graph as G

pytestmark = pytest.mark.gpu


def _complete(k, extra=0):
    a, b = np.triu_indices(k, 1)
    return G.from_edges(k + extra, a.astype(np.int32), b.astype(np.int32), f"K{k}+{extra}")


def _cliques(sizes, gap):
    src, dst, base = [], [], 0
    for s in sizes:
        a, b = np.triu_indices(s, 1)
        src.append(a + base)
        dst.append(b + base)
        base += s + gap
    return G.from_edges(base, np.concatenate(src).astype(np.int32), np.concatenate(dst).astype(np.int32), "cliques")


CASES = {
    # the out-lists of K_k are 0 .. k - 1 long: both sides of the 32 limit
    "K33": lambda: _complete(33),
    "K34": lambda: _complete(34),
    "K70_isolated": lambda: _complete(70, 5000),      # runs of empty rows at the end
    "cliques_gaps": lambda: _cliques([2, 3, 31, 32, 33, 34, 35, 64, 65, 66, 129], 300),
    "rmat_hub": lambda: G.rmat(13, 48, seed=5),       # hubs of several tiles
    "er_tiles": lambda: G.erdos_renyi(2051, 2.0, seed=3),
    "star_plus": lambda: G.from_edges(6001, np.r_[np.zeros(6000), np.arange(1, 6000)].astype(np.int32),
                                      np.r_[np.arange(1, 6001), np.arange(2, 6001)].astype(np.int32), "wheel"),
    # ranks on both sides of 2^16 - 1, up to which the lists are read as 16 bits
    "around_16bit": lambda: G.erdos_renyi(70000, 90.0, seed=4),
    # more than 2^17 vertices with out-lists above 32: ranks beyond the bitmap
    "beyond_bitmap": lambda: G.erdos_renyi(150000, 90.0, seed=2),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_oriented_count(gpu, name):
    g = CASES[name]()
    with gpu.DeviceGraph(g) as dg:
        r = gpu.run("tc", dg, "oriented_lds")
    assert r.out == O.tc_forward(g), name
