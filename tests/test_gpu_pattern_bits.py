"""GPU parity of the fixed patterns on adjacency bit matrices: sizes around a
matrix's 128-position chunk and 2048-id segment, sets around a 16-entry block,
sparse and dense graphs, and graphs that keep the list path."""
import numpy as np
import pytest

import graphs

pytestmark = pytest.mark.gpu

PIDS = ["P%d" % i for i in range(1, 9)]


def check(gpm, orc, g, pids=PIDS, forms=True):
    with gpm.DeviceGraph(g, oriented=False) as dg:
        for p in pids:
            want = orc.pattern(g.offsets, g.adj, int(p[1:]))
            out, scalar = dg.pattern(p, gpm.FORM_G2MINER)
            assert scalar == want and out[0] == want, (g.n, p)
            if forms:
                out, scalar = dg.pattern(p, gpm.FORM_PATTERN)
                assert scalar == want and out[0] == want, (g.n, p)
                if p in ("P2", "P3", "P7", "P8"):
                    assert out[1] - out[2] == want, (g.n, p)
                assert dg.pattern(p, gpm.FORM_BLOCK_PREFILTER)[1] == want, (g.n, p)


@pytest.mark.parametrize("n,m", [(3, 2), (17, 60), (33, 33), (127, 700), (128, 700), (129, 700), (300, 1500)])
def test_small_graphs(gpm, orc, n, m):
    g = graphs.er(n, m, n + m)
    check(gpm, orc, g)
    with gpm.DeviceGraph(g, oriented=False) as dg:
        assert dg.pattern("Motif4", gpm.FORM_G2MINER)[0] == orc.motif4(g.offsets, g.adj)


@pytest.mark.parametrize("n", [2047, 2048, 2049, 4100])
def test_segment_edges(gpm, orc, n):
    """A dense core whose ids are spread over all segments, so that sets and
    lists cross them (2049 and 4100 ids: two and three segments)."""
    rng = np.random.default_rng(n)
    core = np.sort(rng.permutation(n)[:120])
    core[-1] = n - 1
    i, j = np.nonzero(np.triu(rng.random((120, 120)) < 0.6, 1))
    ring = np.arange(n - 1)
    src, dst = np.concatenate([core[i], ring]), np.concatenate([core[j], ring + 1])
    g = gpm.csr_from_edges(n, src.astype(np.uint32), dst.astype(np.uint32))
    check(gpm, orc, g, ["P1", "P2", "P3", "P5", "P6", "P7", "P8"] if n < 4000 else ["P2", "P6", "P7"])


def test_both_paths_give_the_same_sums(gpm):
    """h[1] and h[2] of the counting formulation on the matrices and on lists:
    isolated vertices past the matrix limit take a graph to the lists."""
    g = gpm.rmat_graph(9, 16, 3)
    big = gpm.csr_from_edges(20000, np.repeat(np.arange(g.n, dtype=np.uint32), g.degrees()), g.adj)
    with gpm.DeviceGraph(g, oriented=False) as a, gpm.DeviceGraph(big, oriented=False) as b:
        for p in PIDS:
            for form in (gpm.FORM_G2MINER, gpm.FORM_PATTERN, gpm.FORM_BLOCK_PREFILTER):
                assert a.pattern(p, form) == b.pattern(p, form), (p, form)


def test_repeated_entries_keep_the_lists(gpm):
    """A list that holds an entry twice has no bit matrix: same counts as the
    graph with isolated vertices past the matrix limit."""
    off = np.array([0, 3, 5, 7, 8], dtype=np.uint32)
    adj = np.array([1, 1, 2, 0, 2, 0, 1, 0], dtype=np.uint32)
    small = gpm.HostCSR(off, adj)
    big = gpm.HostCSR(np.concatenate([off, np.full(20000, off[-1], np.uint32)]), adj)
    with gpm.DeviceGraph(small, oriented=False) as a, gpm.DeviceGraph(big, oriented=False) as b:
        for p in PIDS:
            assert a.pattern(p, gpm.FORM_G2MINER) == b.pattern(p, gpm.FORM_G2MINER), p
