"""MIS on dense graphs, whose members exclude nearly everybody: rows around the
length from which a row is excluded in pieces, few and many pieces a round, and
average degrees around the one from which the pieces are worked off at once.
The greedy set of the oracle, and a clique is done in two rounds whatever the
length of its rows: one that finds the member, one that finds it in every other
row."""
import numpy as np
import pytest

import oracle as O
from indigo2suite_amd import graph as G

pytestmark = pytest.mark.gpu


def _clique(n):
    i, j = np.triu_indices(n, 1)
    return G.from_edges(n, i.astype(np.int32), j.astype(np.int32), f"clique{n}")


@pytest.mark.parametrize("n", [255, 256, 257, 258, 1024, 1025, 1026, 2000, 2050])
def test_clique(gpu, n):
    g = _clique(n)
    with gpu.DeviceGraph(g) as dg:
        r = gpu.run("mis", dg, "v_resume_pull")
    assert np.array_equal(r.out, O.mis_greedy(g).astype(np.int32))
    assert r.iterations == 2


@pytest.mark.parametrize("n,degree", [(3000, 1400.0), (4096, 1100.0), (9000, 250.0), (9000, 262.0), (6000, 3000.0)])
def test_random(gpu, n, degree):
    g = G.erdos_renyi(n, degree, seed=n)
    with gpu.DeviceGraph(g) as dg:
        assert np.array_equal(gpu.run("mis", dg, "v_resume_pull").out, O.mis_greedy(g).astype(np.int32))


@pytest.mark.parametrize("cliques", [16, 17, 40])
def test_many_pieces_at_once(gpu, cliques):
    # as many members in the first round, two pieces each
    one = _clique(1100)
    k = np.arange(cliques)
    g = G.Graph(np.r_[0, (one.nindex[1:][None, :].astype(np.int64) + (k * one.edges)[:, None]).ravel()].astype(np.int32),
                (one.nlist[None, :] + (k * one.nodes)[:, None]).astype(np.int32).ravel(), None, f"cliques{cliques}")
    with gpu.DeviceGraph(g) as dg:
        assert np.array_equal(gpu.run("mis", dg, "v_resume_pull").out, O.mis_greedy(g).astype(np.int32))
