"""GPU Motif4 identities on graphs whose lists are one-sided (an unsymmetrised edge
file): the call ends, and its numbers are the identities' own sums over the lists
as they are, recounted here."""
from math import comb

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MOD = 1 << 64


def recount(gpm, orc, g):
    """motif_count.hip's sums on the host: degrees are list lengths, ranks are by
    (degree, id), the DAG keeps every entry that goes up, and the 4-cycle corners
    walk the entries below a root and theirs."""
    off = np.asarray(g.offsets).astype(np.int64)
    adj = np.asarray(g.adj).astype(np.int64)
    deg = np.diff(off)
    n = len(deg)
    rank = np.empty(n, np.int64)
    rank[np.lexsort((np.arange(n), deg))] = np.arange(n)
    lists = [None] * n  # by rank
    d = np.empty(n, np.int64)
    for v in range(n):
        lists[rank[v]] = np.sort(rank[adj[off[v]:off[v + 1]]])
        d[rank[v]] = deg[v]
    up = [x[np.searchsorted(x, v + 1):] for v, x in enumerate(lists)]
    sets = [set(x.tolist()) for x in up]
    c = {(u, int(v)): 0 for u in range(n) for v in up[u]}
    for u in range(n):
        for v in sets[u]:
            for w in sets[u] & sets[v]:
                c[u, v] += 1
                c[u, w] += 1
                c[v, w] += 1
    tri = sum(c.values()) // 3
    star = sum(comb(int(x), 3) for x in d)
    paw = sum(k * int(d[u] + d[v] - 4) for (u, v), k in c.items()) % MOD // 2
    dia = sum(k * (k - 1) for k in c.values()) // 2
    path = sum(int((d[u] - 1) * (d[v] - 1)) for u, v in c) - 3 * tri
    cyc = 0
    for u in range(n):
        low = lists[u][lists[u] < u]
        if len(low):
            ends = np.concatenate([lists[v][lists[v] < u] for v in low])
            k = np.unique(ends, return_counts=True)[1]
            cyc += int((k * (k - 1) // 2).sum())
    dag = gpm.orient(g)
    k4 = orc.clique(dag.offsets, dag.adj, 4)
    i_dia = dia - 6 * k4
    i_cyc = cyc - i_dia - 3 * k4
    i_paw = paw - 4 * i_dia - 12 * k4
    i_path = path - 2 * i_paw - 4 * i_cyc - 6 * i_dia - 12 * k4
    i_star = star - i_paw - 2 * i_dia - 4 * k4
    return [x % MOD for x in (i_star, i_path, i_paw, i_cyc, i_dia, k4)]


def directed(gpm, n, src, dst):
    return gpm.csr_from_edges(n, np.asarray(src, np.uint32), np.asarray(dst, np.uint32),
                              gpm.CSR_SORT | gpm.CSR_DEDUP | gpm.CSR_DROP_SELF)


def motif4(gpm, g):
    with gpm.DeviceGraph(g, oriented=False) as dg:
        first = dg.pattern("Motif4", gpm.FORM_PATTERN)[0]
        assert dg.pattern("Motif4", gpm.FORM_PATTERN)[0] == first
        assert dg.pattern("P1", gpm.FORM_PATTERN)[0][0] == first[0]
        assert dg.pattern("P4", gpm.FORM_PATTERN)[0][0] == first[1]
    return first


@pytest.mark.parametrize("mids,ends,pool", [(8, 6, 40), (20, 100, 2100), (20, 102, 2100),
                                            (150, 100, 6000), (150, 100, 15000), (300, 280, 70000)])
def test_ends_past_the_lists_that_point_back(gpm, orc, mids, ends, pool):
    """Roots whose middle vertices mostly do not list them: the wedges a root walks
    (up to 84000, to more ends than the light roots' table has slots) are not the
    entries that point at it.  No triangles."""
    rng = np.random.default_rng(mids + ends)
    roots = 3
    low = roots + mids + np.arange(pool)
    src, dst = [], []
    for i in range(mids):
        src.append(np.full(ends, roots + i))
        dst.append(low[(i * ends) % pool + np.arange(ends)] if pool >= mids * ends
                   else low[np.sort(rng.permutation(pool)[:ends])])
    for r in range(roots):
        src.append(np.full(mids, r))
        dst.append(roots + np.arange(mids))
    # a middle vertex's list is shorter than a root's, as ranks need it to be
    extra = max(0, ends + 8 - mids)
    sink = roots + mids + pool
    for r in range(roots):
        src.append(np.full(extra, r))
        dst.append(sink + np.arange(extra))
    src += [np.array([roots, roots + 1])]  # two of them point back at root 0
    dst += [np.array([0, 0])]
    g = directed(gpm, sink + extra, np.concatenate(src), np.concatenate(dst))
    assert motif4(gpm, g) == recount(gpm, orc, g)


@pytest.mark.parametrize("n,m,mutual,loops", [(40, 300, 0.0, 0), (300, 6000, 0.3, 0), (300, 6000, 0.999, 0),
                                              (120, 3000, 1.0, 1), (1500, 30000, 0.5, 20)])
def test_triangles_of_one_sided_lists(gpm, orc, n, m, mutual, loops):
    """A random digraph with some, nearly all and all edges in both lists, and loops."""
    rng = np.random.default_rng(n + m)
    src, dst = rng.integers(0, n, m), (rng.random(m) ** 2 * n).astype(np.int64)
    both = rng.random(m) < mutual
    own = rng.permutation(n)[:loops]
    keep = src != dst
    g = gpm.csr_from_edges(n, np.concatenate([src[keep], dst[keep & both], own]).astype(np.uint32),
                           np.concatenate([dst[keep], src[keep & both], own]).astype(np.uint32),
                           gpm.CSR_SORT | gpm.CSR_DEDUP)
    assert motif4(gpm, g) == recount(gpm, orc, g)
