"""GPU: 4-cycle queries on one-sided lists (an unsymmetrised edge file) and on lists
with loops give the depth-first search's counts (a replayed graph keeps it)."""
import itertools

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SQUARE = [(0, 1), (1, 2), (2, 3), (3, 0)]
PATH_FIRST = [(0, 1), (0, 3), (1, 2), (2, 3)]


def graph(gpm, n, m, mutual, loops, repeat=False):
    rng = np.random.default_rng(n + m + loops)
    src, dst = rng.integers(0, n, m), (rng.random(m) ** 2 * n).astype(np.int64)
    both = rng.random(m) < mutual
    own = rng.permutation(n)[:loops]
    keep = src != dst
    return gpm.csr_from_edges(n, np.concatenate([src[keep], dst[keep & both], own]).astype(np.uint32),
                              np.concatenate([dst[keep], src[keep & both], own]).astype(np.uint32),
                              gpm.CSR_SORT | (0 if repeat else gpm.CSR_DEDUP))


def queries(n_labels):
    sets = [(0, 0, 0, 0)] if n_labels == 1 else [(0, 0, 0, 0), (0, 1, 0, 1), (0, 1, 1, 0), (1, 0, 0, 0)]
    return [(4, e, list(l)) for l, e in itertools.product(sets, (SQUARE, PATH_FIRST))]


@pytest.mark.parametrize("n_labels", [1, 2])
@pytest.mark.parametrize("n,m,mutual,loops,repeat", [(60, 500, 0.0, 0, False), (400, 6000, 0.4, 0, False),
                                                     (400, 6000, 0.995, 0, False), (300, 3000, 1.0, 30, False),
                                                     (300, 3000, 1.0, 1, False), (80, 900, 1.0, 0, True)])
def test_lists_that_are_not_mirrored(gpm, n, m, mutual, loops, repeat, n_labels):
    g = graph(gpm, n, m, mutual, loops, repeat)
    lab = gpm.gen_labels(n, n_labels, 5)
    with gpm.DeviceGraph(g, oriented=False, labels=lab, n_labels=n_labels) as dg:
        for q in queries(n_labels):
            want = dg.match_batch([q], autotune=0, chunk=8, use_graph=1).tolist()
            assert dg.match_batch([q], policy=0).tolist() == want, q


def test_loops_are_no_edges_of_a_cycle(gpm):
    """Brute force over the injective maps; both policies."""
    n = 24
    g = graph(gpm, n, 120, 1.0, 9)
    a = np.zeros((n, n), bool)
    a[np.repeat(np.arange(n), np.diff(g.offsets.astype(np.int64))), g.adj] = True
    want = sum(a[p, q] and a[q, r] and a[r, s] and a[s, p]
               for p, q, r, s in itertools.permutations(range(n), 4))
    with gpm.DeviceGraph(g, oriented=False, labels=np.zeros(n, np.uint32), n_labels=1) as dg:
        for policy in (0, 1):
            assert dg.match_batch([(4, SQUARE, [0] * 4)], policy=policy).tolist() == [want]


@pytest.mark.parametrize("built", [False, True])
def test_mirrored_lists(gpm, orc, built):
    """Made on the host or on the device, and relabelled: the oracle's counts."""
    s, d = gpm.gen_er(500, 4000, 9)
    host = gpm.csr_from_edges(500, s, d)
    lab = gpm.gen_labels(500, 2, 3)
    dg = (gpm.DeviceGraph.build(500, s, d, labels=lab, n_labels=2) if built
          else gpm.DeviceGraph(host, oriented=False, labels=lab, n_labels=2))
    want = list(orc.ceci_batch(host.offsets, host.adj, lab, queries(2)))
    with dg:
        assert dg.match_batch(queries(2)).tolist() == want
        again, _ = dg.relabel_by_degree()
        with again:
            assert again.match_batch(queries(2)).tolist() == want
