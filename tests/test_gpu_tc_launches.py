"""The launches that the default triangle counting reports: with edges its
clear, three rank passes, the keep pass, the three launches of the scan, the
orientation, the two counts and the publication; without, the clear and the
publication."""
import numpy as np
import pytest

from indigo2suite_amd import graph as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,launches", [("edges", 12), ("edgeless", 2)])
def test_launches(gpu, name, launches):
    g = G.erdos_renyi(500, 6.0, seed=1) if name == "edges" else G.Graph(np.zeros(6, np.int32), np.zeros(0, np.int32))
    with gpu.DeviceGraph(g) as dg:
        assert gpu.run("tc", dg, "oriented_lds").launches == launches
