"""The edge worklist style of CC around the average degree (8) and the length
of the first list (8 items a thread of 2048 workgroups of 256) at which a
thread's items are taken one by one or four at once."""
import numpy as np
import pytest

import oracle as O
from indigo2suite_amd import graph as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,degree", [(30000, 7.9), (30000, 8.1), (300, 40.0), (261000, 16.0), (263500, 16.0)])
def test_labels(gpu, n, degree):
    g = G.erdos_renyi(n, degree, seed=n)
    with gpu.DeviceGraph(g) as dg:
        assert np.array_equal(gpu.run("cc", dg, "e_data_push_thread").out, O.cc_omp_pull(g)[0])
