"""Which graphs PageRank's balanced style works on renumbered by degree: those
whose 16384 vertices of highest degree take a quarter of the edges, well above
their share of the vertices, are met by long rows, lie scattered where the
contributions exceed an XCD's L2, and whose edges outnumber the vertices.  The
side is read from the timed launches of the kernel that only renumbered graphs
have; the scores are the thread-per-vertex style's (both within 1e-5 of FP64)
and so are the iterations, the sums of either side being exact to rounding."""
import ctypes

import numpy as np
import pytest

from indigo2suite_amd import graph as G

pytestmark = pytest.mark.gpu


def _star(n, hubs):
    v = np.arange(hubs, n, dtype=np.int32)
    return G.from_edges(n, v, (v % hubs).astype(np.int32), f"star{n}_{hubs}")


def _inside(g, n):
    """g's vertices first, the others of n isolated"""
    return G.Graph(np.r_[g.nindex, np.full(n - g.nodes, g.edges, np.int32)], g.nlist, None, f"{g.name}_in{n}")


CASES = {  # name: (graph, renumbered)
    "rmat": (lambda: G.rmat(16, 16, seed=1), True),
    "chung_lu": (lambda: G.chung_lu(100000, 16.0, 2.5, seed=1), True),
    "rmat_beyond_l2": (lambda: G.rmat(21, 2, seed=1), True),
    "sorted_beyond_l2": (lambda: G.chung_lu(1200000, 12.0, 2.3, seed=1), False),
    "sorted_beyond_l2_short_rows": (lambda: G.chung_lu(1200000, 6.0, 2.3, seed=1), True),
    "mesh_200": (lambda: G.grid2d(200, 0.05, seed=1), False),
    "mesh_250": (lambda: G.grid2d(250, 0.0, seed=1), False),
    "mesh_300": (lambda: G.grid2d(300, 0.05, seed=1), False),
    "random_sparse": (lambda: G.erdos_renyi(40000, 4.0, seed=1), False),
    "random_dense": (lambda: G.erdos_renyi(65536, 64.0, seed=1), False),
    "star": (lambda: _star(300000, 40), False),
    "few_edges": (lambda: _inside(G.rmat(15, 8, seed=1), 1 << 20), False),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_side(gpu, name):
    make, renumbered = CASES[name]
    g = make()
    lib = gpu.lib()
    n = ctypes.c_int()
    try:
        gpu.set_pr_params(1e-6, 100)
        with gpu.DeviceGraph(g) as dg:
            lib.igx_profile_kernel(b"pr_hot_chunks")
            r = gpu.run("pr", dg, "pull_balanced_kahan")
            lib.igx_profile_read(None, ctypes.byref(n))
            lib.igx_profile_kernel(None)
            t = gpu.run("pr", dg, "pull_thread_kahan")
        assert (n.value > 0) == renumbered
        assert abs(r.iterations - t.iterations) <= 1
        if r.iterations == t.iterations:
            assert np.max(np.abs(r.out - t.out) / t.out) <= 2e-5
    finally:
        lib.igx_profile_kernel(None)
        gpu.set_pr_params(1e-4, 100)


def test_no_memory_for_a_copy_that_is_not_made(gpu):
    def free_bytes():
        # the HIP runtime that the library itself is linked to
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert gpu.lib()["hipMemGetInfo"](ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    g = G.erdos_renyi(1 << 20, 16.0, seed=1)
    with gpu.DeviceGraph(g) as dg:
        buf = gpu.DeviceBuffer(4 * g.nodes)
        assert gpu.lib().igx_release_workspace() == 0
        before = free_bytes()
        gpu.run_device("pr", dg, buf, "pull_balanced_kahan")
        after = free_bytes()
        buf.free()
    # contributions, the lists of longer rows and the partial sums take about 28 MB,
    # the copy of the lists alone would take four bytes an edge (67 MB)
    assert before - after < 4 * g.edges
