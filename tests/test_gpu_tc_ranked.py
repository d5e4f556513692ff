"""GPU parity of the vertex-centric triangle count on the relabelled DAG:
out-degrees around its groups, windows and blocks, ids above and below its
bitmap, lists long enough to be searched, and graphs that keep the hash kernels."""
import numpy as np
import pytest

import graphs

pytestmark = pytest.mark.gpu


def check(gpm, orc, d):
    want = orc.tc(d.offsets, d.adj)
    with gpm.DeviceGraph(d, oriented=True) as dg:
        assert dg.tc(gpm.TC_VERTEX) == want
        assert dg.tc(gpm.TC_VERTEX) == want
        assert dg.tc_repeat(gpm.TC_VERTEX, 3) == want
    return want


@pytest.mark.parametrize("degree", [2, 3, 7, 8, 9, 15, 16, 17, 18, 63, 64, 65, 255, 256, 257, 300, 700])
def test_hub_degrees(gpm, orc, degree):
    """Hubs of one out-degree over a shared random DAG, so that the lists a hub
    streams are longer and shorter than a window; many hubs, so that every
    group of lanes holds some."""
    rng = np.random.default_rng(degree)
    base, hubs = 900, 70
    i, j = np.nonzero(np.triu(rng.random((base, base)) < 0.15, 1))
    src, dst = [hubs + i], [hubs + j]
    for h in range(hubs):
        src.append(np.full(degree, h))
        dst.append(hubs + rng.permutation(base)[:degree])
    src, dst = np.concatenate(src).astype(np.uint32), np.concatenate(dst).astype(np.uint32)
    assert check(gpm, orc, gpm.csr_from_edges(base + hubs, src, dst, gpm.CSR_SORT)) >= 0


@pytest.mark.parametrize("n", [65536, 65537, 70000, 200000])
def test_ids_below_the_bitmap(gpm, orc, n):
    """Power-law graphs whose lists reach below the top 65536 ids."""
    g = gpm.rmat_graph(18, 4, n)
    keep = np.repeat(np.arange(g.n), g.degrees()) < n
    src, dst = np.repeat(np.arange(g.n, dtype=np.uint32), g.degrees())[keep], g.adj[keep]
    sub = gpm.csr_from_edges(n, src[dst < n], dst[dst < n])
    assert check(gpm, orc, gpm.orient(sub)) > 0


def test_long_lists_are_searched(gpm, orc):
    """Roots of 20 ids whose lists hold 400 and more."""
    rng = np.random.default_rng(3)
    roots, mid, far = 50, 40, 3000
    src, dst = [], []
    for r in range(roots):
        src.append(np.full(20, r))
        dst.append(roots + np.sort(rng.permutation(mid)[:20]))
    for m in range(mid):
        src += [np.full(mid - 1 - m, roots + m), np.full(450, roots + m)]
        dst += [roots + np.arange(m + 1, mid), roots + mid + np.sort(rng.permutation(far)[:450])]
    src, dst = np.concatenate(src).astype(np.uint32), np.concatenate(dst).astype(np.uint32)
    assert check(gpm, orc, gpm.csr_from_edges(roots + mid + far, src, dst, gpm.CSR_SORT)) > 0


def test_other_graphs(gpm, orc):
    """Near-uniform degrees, an order that is not by degree, a graph that is no
    DAG, and empty ones."""
    check(gpm, orc, gpm.orient(gpm.er_graph(3000, 48000, 5)))
    d = gpm.orient(gpm.rmat_graph(12, 16, 6))
    check(gpm, orc, gpm.sort_by_degree(d)[0])
    cyclic = gpm.csr_from_edges(4, [0, 1, 2, 0, 1], [1, 2, 0, 3, 3], gpm.CSR_SORT)
    check(gpm, orc, cyclic)
    check(gpm, orc, gpm.csr_from_edges(5, [], [], gpm.CSR_SORT))
    check(gpm, orc, gpm.orient(graphs.complete(130)))
