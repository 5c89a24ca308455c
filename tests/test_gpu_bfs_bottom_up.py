"""Bottom-up BFS levels on graphs above and below the size from which every
wave has four tiles of 64 vertices side by side (2048 workgroups of four waves:
2,097,152 vertices), of few and of many edges a vertex, with a ragged last
tile, and rows just below and above the 36 neighbours that a lane looks at by
itself on the former.  Levels against the serial oracle."""
import numpy as np
import pytest

import oracle as O
from indigo2suite_amd import graph as G

pytestmark = pytest.mark.gpu


def _with_rows(g, lengths, seed):
    """g and, for each length, 40 further vertices joined to that many of g's"""
    rng = np.random.default_rng(seed)
    src = [np.repeat(np.arange(g.nodes, dtype=np.int32), g.degrees())]
    dst = [g.nlist]
    v = g.nodes
    for length in lengths:
        for _ in range(40):
            src.append(np.full(length, v, np.int32))
            dst.append(rng.choice(g.nodes, length, replace=False).astype(np.int32))
            v += 1
    return G.from_edges(v, np.concatenate(src), np.concatenate(dst), g.name + "_rows")


@pytest.mark.parametrize("n,degree", [(2097152 - 70, 8.0), (2097152 - 320, 8.0), (2097152 + 1, 8.0), (2097152 + 4099, 17.0)])
def test_levels(gpu, n, degree):
    g = _with_rows(G.erdos_renyi(n, degree, seed=3), (34, 35, 36, 37, 38, 100), seed=4)
    src = int(np.flatnonzero(g.degrees() > 0)[0])
    with gpu.DeviceGraph(g) as dg:
        r = gpu.run("bfs", dg, "do_hybrid", src=src)
    assert np.array_equal(r.out, O.bfs_serial(g, src))
