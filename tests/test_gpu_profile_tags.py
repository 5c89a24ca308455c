"""What the timing tags cover: where a step is shared by several kernels its
tag times them all, so the rest of the run (set-up, the ends of PageRank's
iterations, the lists of longer rows) is the smaller part."""
import ctypes

import pytest

from indigo2suite_amd import graph as G

pytestmark = pytest.mark.gpu

CASES = {
    "bfs": (lambda: G.grid2d(150, 0.0, seed=1), "bfs_do_level"),
    "sssp": (lambda: G.grid2d(100, 0.0, seed=1).with_weights(1, 255, seed=1), "sssp_do_round"),
    "pr": (lambda: G.rmat(20, 16, seed=1), "pr_bal_main"),
}


@pytest.mark.parametrize("algo", sorted(CASES))
def test_share_of_the_run(gpu, algo):
    make, tag = CASES[algo]
    g = make()
    lib = gpu.lib()
    ms, n = ctypes.c_double(), ctypes.c_int()
    try:
        gpu.set_pr_params(1e-6, 100)
        with gpu.DeviceGraph(g) as dg:
            gpu.run(algo, dg)
            lib.igx_profile_kernel(tag.encode())
            r = gpu.run(algo, dg)
            lib.igx_profile_read(ctypes.byref(ms), ctypes.byref(n))
        assert n.value == r.launches
        assert 0.5 * r.seconds < ms.value * 1e-3 <= r.seconds
    finally:
        lib.igx_profile_kernel(None)
        gpu.set_pr_params(1e-4, 100)
