"""GPU parity of the Motif4 identities where their kernels split: ranks past an
LDS band, counters wider than 16 bits, out-lists past the LDS counters, and
graphs at the edges of the light kernels."""
from math import comb

import numpy as np
import pytest

import graphs

pytestmark = pytest.mark.gpu


def motif4(gpm, g):
    with gpm.DeviceGraph(g, oriented=False) as dg:
        first = dg.pattern("Motif4", gpm.FORM_PATTERN)[0]
        assert dg.pattern("Motif4", gpm.FORM_PATTERN)[0] == first
    return first


def test_ranks_past_a_band(gpm, orc):
    """131072 ranks: roots of every class of the 4-cycle tasks, with ends in LDS
    bands and in HBM."""
    g = gpm.rmat_graph(17, 1, 5)
    assert motif4(gpm, g) == orc.motif4(g.offsets, g.adj)


def test_wide_counters(gpm):
    """K(2, 70000): one counter reaches 70000."""
    m = 70000
    leaves = np.arange(2, m + 2, dtype=np.uint32)
    src = np.concatenate([leaves, leaves])
    dst = np.concatenate([np.zeros(m, np.uint32), np.ones(m, np.uint32)])
    g = gpm.csr_from_edges(m + 2, src, dst)
    assert motif4(gpm, g) == [2 * comb(m, 3), 0, 0, comb(m, 2), 0, 0]


@pytest.mark.parametrize("n", [4, 17, 18, 65, 1030, 1100])
def test_complete_graphs(gpm, n):
    """Out-lists up to n - 1: the pair searches, one task, several tasks, and more
    than 1024 positions."""
    assert motif4(gpm, graphs.complete(n)) == [0, 0, 0, 0, 0, comb(n, 4)]


@pytest.mark.parametrize("n,m", [(2, 1), (60, 200), (300, 2700), (5000, 20000)])
def test_small_graphs(gpm, orc, n, m):
    g = graphs.er(n, m, n)
    assert motif4(gpm, g) == orc.motif4(g.offsets, g.adj)


def test_graph_without_edges(gpm):
    assert motif4(gpm, gpm.csr_from_edges(40, [], [])) == [0] * 6
