"""Triangle counting where ranks exceed the bitmap's 2^17: disjoint cliques,
whose vertices all have one degree, so that any of them may be ranked there.
The lists of a clique of k vertices have 0 to k - 1 elements: up to 32 they are
counted row by row; longer ones by a workgroup, or, at average degrees from 42
to 160, one wave each up to 128.  Closed form: copies * C(k, 3)."""
import math

import numpy as np
import pytest

import oracle as O
from indigo2suite_amd import graph as G

pytestmark = pytest.mark.gpu


def _cliques(k, copies, extra=0):
    ids = np.arange(k, dtype=np.int32)
    one = np.array([np.delete(ids, v) for v in range(k)], np.int32).reshape(-1)
    nlist = (one[None, :] + (np.arange(copies, dtype=np.int32) * k)[:, None]).reshape(-1)
    nindex = np.arange(k * copies + 1, dtype=np.int64) * (k - 1)
    return G.Graph(np.r_[nindex, np.full(extra, nindex[-1])].astype(np.int32), nlist, None, f"cliques{k}x{copies}")


@pytest.mark.parametrize("k,copies", [(34, 4000), (35, 3745), (35, 3746), (42, 3200), (43, 3150), (44, 3100), (50, 2650), (66, 2100), (97, 1500),
                                      (129, 1020), (130, 1010), (160, 830), (161, 830), (162, 830), (290, 470)])
def test_cliques(gpu, k, copies):
    with gpu.DeviceGraph(_cliques(k, copies, extra=77)) as dg:
        assert gpu.run("tc", dg, "oriented_lds").out == copies * math.comb(k, 3)


def test_random(gpu):
    g = G.erdos_renyi(150001, 75.0, seed=2)
    with gpu.DeviceGraph(g) as dg:
        assert gpu.run("tc", dg, "oriented_lds").out == O.tc_forward(g)
