"""Batches of the matcher around the number of queries whose counts a block adds up
itself, with fewer tasks than queue counters and with many, replayed and in passes."""
import numpy as np
import pytest

import graphs

pytestmark = pytest.mark.gpu

SHAPES = [(3, [(0, 1), (1, 2), (2, 0)]), (4, [(0, 1), (0, 2), (0, 3)]),
          (4, [(0, 1), (1, 2), (2, 0), (2, 3)]), (2, [(0, 1)]),
          (5, [(0, 1), (1, 2), (2, 3), (3, 4)])]


def queries(count, n_labels, seed):
    rng = np.random.default_rng(seed)
    out = []
    for i in range(count):
        n, edges = SHAPES[i % len(SHAPES)]
        out.append((n, edges, rng.integers(0, n_labels, n).tolist()))
    return out


@pytest.mark.parametrize("count", [1, 2, 63, 64, 65, 130])
@pytest.mark.parametrize("n,m", [(5, 6), (60, 300), (3000, 15000)])
def test_batch_sizes(gpm, orc, count, n, m):
    g = graphs.er(n, m, n + count)
    labels = np.random.default_rng(n).integers(0, 3, n).astype(np.uint32)
    qs = queries(count, 3, count)
    want = orc.ceci_batch(g.offsets, g.adj, labels, qs)
    with gpm.DeviceGraph(g, oriented=False, labels=labels, n_labels=3) as dg:
        for _ in range(2):
            assert np.array_equal(dg.match_batch(qs), want)
            assert np.array_equal(dg.match_batch(qs, policy=1), want)
        for _ in range(2):
            assert np.array_equal(dg.match_batch(qs, autotune=0, chunk=1, use_graph=1), want)
        assert np.array_equal(dg.match_batch(qs, pass_budget=4), want)
