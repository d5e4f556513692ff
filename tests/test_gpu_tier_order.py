"""Root tiers sorted on the device against those of an explicit root list, which the host
sorts: whole graphs, ranges that cut every tier, wave tiers of other widths."""
import numpy as np
import pytest

import graphs

pytestmark = pytest.mark.gpu


def dags(gpm):
    yield gpm.orient(gpm.rmat_graph(13, 24, 4))
    yield gpm.orient(graphs.complete(600))
    yield gpm.orient(gpm.csr_from_edges(50, [0], [1]))


def test_ranges_and_lists(gpm):
    for d in dags(gpm):
        n = d.n
        with gpm.DeviceGraph(d, oriented=True) as dg:
            for k in (3, 4):
                whole = dg.clique(k)
                assert dg.clique(k, roots=np.arange(n, dtype=np.uint32)) == whole
                cuts = [0, 1, n // 3, n // 2 + 1, n - 1, n]
                parts = [dg.clique(k, root_begin=a, root_end=b) for a, b in zip(cuts, cuts[1:]) if a < b]
                assert sum(parts) == whole
                lists = [dg.clique(k, roots=np.arange(a, b, dtype=np.uint32))
                         for a, b in zip(cuts, cuts[1:]) if a < b]
                assert parts == lists


@pytest.mark.parametrize("wave_cap", [1, 7, 33, 64])
def test_wave_caps(gpm, wave_cap):
    d = gpm.orient(gpm.rmat_graph(12, 24, 5))
    with gpm.DeviceGraph(d, oriented=True) as dg:
        assert dg.clique(4, wave_cap=wave_cap) == dg.clique(4)
        assert dg.tc(gpm.TC_VERTEX) == dg.clique(3, wave_cap=wave_cap)
