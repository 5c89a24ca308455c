"""Edge worklist styles (BFS, SSSP, CC) at the edges of their appends: list
sizes around the one-item-per-thread limit of the grid, ranges of 256 and 257
edges (written with and without a search), hubs whose neighbours are hubs, and
lists long enough for several items per thread.  Results equal the oracle's."""
import numpy as np
import pytest

import oracle as O
from indigo2suite_amd import graph as G

pytestmark = pytest.mark.gpu


def _hub_of(k, leaves):
    """a root joined to k centres of `leaves` leaves each"""
    c = 1 + np.arange(k)
    centre = np.repeat(c, leaves)
    leaf = 1 + k + np.arange(k * leaves)
    src = np.r_[np.zeros(k, np.int64), centre].astype(np.int32)
    dst = np.r_[c, leaf].astype(np.int32)
    return G.from_edges(1 + k + k * leaves, src, dst, f"hubs{k}x{leaves}")


CASES = {
    "range_256": lambda: _hub_of(70, 255),
    "range_257": lambda: _hub_of(70, 256),
    "range_mixed": lambda: _hub_of(129, 300),
    "alone_limit": lambda: _hub_of(65536, 1),
    "above_alone": lambda: _hub_of(65537, 1),
    "several_items": lambda: G.rmat(16, 24, seed=2, n_limit=50001),   # rounds of more than 524,288 items
    "grid": lambda: G.grid2d(150, 0.02, seed=3),
    "tiny": lambda: G.from_edges(5, np.array([0, 1], np.int32), np.array([1, 2], np.int32), "tiny"),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_edge_worklists(gpu, name):
    g = CASES[name]().with_weights(1, 255, seed=4)
    bfs, sssp, cc = O.bfs_serial(g, 0), O.sssp_serial(g, 0), O.cc_omp_pull(g)[0]
    with gpu.DeviceGraph(g) as dg:
        assert np.array_equal(gpu.run("bfs", dg, "e_data_push_thread", 0).out, bfs)
        assert np.array_equal(gpu.run("sssp", dg, "e_data_push_thread", 0).out, sssp)
        assert np.array_equal(gpu.run("sssp", dg, "e_data_push_rw_thread", 0).out, sssp)
        assert np.array_equal(gpu.run("cc", dg, "e_data_push_thread").out, cc)
