"""GPU parity of the 4-cycle matcher's counters against the oracle: one label and
several, opposite corners of equal and different labels, labels past one LDS
band, and queries mixed with others in a batch."""
import numpy as np
import pytest

import graphs

pytestmark = pytest.mark.gpu

SQUARE = [(0, 1), (1, 2), (2, 3), (3, 0)]
PATH_FIRST = [(0, 1), (0, 3), (1, 2), (2, 3)]


def labelled(gpm, g, n_labels, seed=3):
    n = len(g.offsets) - 1
    return np.zeros(n, np.uint32) if n_labels == 1 else gpm.gen_labels(n, n_labels, seed)


@pytest.mark.parametrize("policy", [0, 1])
@pytest.mark.parametrize("labels", [(0, 0, 0, 0), (0, 1, 0, 1), (0, 1, 2, 1), (0, 1, 0, 2),
                                    (1, 1, 0, 2), (2, 2, 0, 0)])
def test_corners(gpm, orc, labels, policy):
    g = graphs.er(400, 4000, 5)
    lab = labelled(gpm, g, 3)
    queries = [(4, SQUARE, list(labels)), (3, [(0, 1), (1, 2), (2, 0)], [0, 1, 2]),
               (4, PATH_FIRST, list(labels))]
    want = orc.ceci_batch(g.offsets, g.adj, lab, queries)
    with gpm.DeviceGraph(g, oriented=False, labels=lab, n_labels=3) as dg:
        for _ in range(3):
            assert dg.match_batch(queries, policy=policy).tolist() == list(want)


@pytest.mark.parametrize("n,m", [(4, 4), (33, 120), (36864, 150000), (36865, 150000),
                                 (80000, 500000)])
def test_bands(gpm, n, m):
    """One label: each 4-cycle is an embedding eight times; its number is the sum of
    C(common neighbours, 2) over the vertex pairs, halved."""
    g = graphs.er(n, m, n)
    src = np.repeat(np.arange(n, dtype=np.int64), np.diff(np.asarray(g.offsets).astype(np.int64)))
    deg = np.diff(np.asarray(g.offsets).astype(np.int64))
    adj = np.asarray(g.adj).astype(np.int64)
    # every wedge u - c - w with u < w, one key per pair (u, w)
    keys = []
    for k in range(int(deg.max()) if len(deg) else 0):
        at = np.asarray(g.offsets)[src].astype(np.int64) + k
        ok = (k < deg[src])
        u, w = adj[ok], adj[at[ok]]
        sel = u < w
        keys.append(u[sel] * n + w[sel])
    _, common = np.unique(np.concatenate(keys), return_counts=True)
    cycles = int((common * (common - 1) // 2).sum()) // 2
    with gpm.DeviceGraph(g, oriented=False, labels=np.zeros(n, np.uint32), n_labels=1) as dg:
        assert dg.match_batch([(4, SQUARE, [0, 0, 0, 0])]).tolist() == [8 * cycles]


def test_hub(gpm):
    """K(2, 65535) and K(2, 65537): a counter's largest value, and a root past it."""
    for m in (65535, 65537):
        leaves = np.arange(2, m + 2, dtype=np.uint32)
        g = gpm.csr_from_edges(m + 2, np.concatenate([leaves, leaves]),
                               np.concatenate([np.zeros(m, np.uint32), np.ones(m, np.uint32)]))
        lab = np.ones(m + 2, np.uint32)
        lab[:2] = 0
        with gpm.DeviceGraph(g, oriented=False, labels=lab, n_labels=2) as dg:
            got = dg.match_batch([(4, SQUARE, [0, 1, 0, 1])]).tolist()
        assert got == [2 * m * (m - 1)]


@pytest.mark.parametrize("kind", ["er", "rmat"])
def test_bands_and_orders_agree_with_the_dfs(gpm, kind):
    """Two labels of more vertices than a band, light roots left to the DFS, every order
    of the cycle, against the DFS of all roots (a replayed graph keeps it)."""
    g = gpm.er_graph(150000, 700000, 3) if kind == "er" else gpm.rmat_graph(17, 6, 3)
    n = len(g.offsets) - 1
    lab = gpm.gen_labels(n, 2, 7)
    with gpm.DeviceGraph(g, oriented=False, labels=lab, n_labels=2) as dg:
        for labels in ((0, 0, 0, 0), (0, 1, 0, 1), (0, 0, 1, 1), (0, 1, 1, 1)):
            for edges in (SQUARE, PATH_FIRST):
                q = [(4, edges, list(labels))]
                want = dg.match_batch(q, autotune=0, chunk=8, use_graph=1).tolist()
                assert dg.match_batch(q, policy=0).tolist() == want
                assert dg.match_batch(q, policy=1).tolist() == want
