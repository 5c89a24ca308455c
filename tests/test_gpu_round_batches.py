"""Rounds enqueued beyond the ones a run needs: two batches at most, each of at
most 32 rounds, which is also what a run past its time limit still waits for.
A path from its end takes a round a vertex in the deterministic styles, so the
number of rounds is known."""
import numpy as np
import pytest

from indigo2suite_amd import graph as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 9, 40, 501, 600, 1500])
def test_rounds_beyond_the_last(gpu, n):
    v = np.arange(n - 1, dtype=np.int32)
    g = G.from_edges(n, v, v + 1, f"path{n}").with_weights(1, 1, seed=1)
    with gpu.DeviceGraph(g) as dg:
        for algo, style in (("bfs", "v_topo_push_thread_determ"), ("sssp", "v_topo_push_thread_determ")):
            r = gpu.run(algo, dg, style)
            assert np.array_equal(r.out, np.arange(n))
            assert r.iterations in (n, n + 1)  # the last one finds nothing
            assert 0 <= r.launches - r.iterations <= 64
