"""GPU: the vertex-centric triangle count's kernels for relabelled DAGs, on graphs that
are shown here to take them: the orientation of a symmetric graph is ordered by
(total degree, id), and isolated vertices keep the mean list length low against
the length an entry meets."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CORE, ROOTS, ISOLATED = 900, 70, 4000


def cored(gpm, degree, density, seed=0):
    """ROOTS vertices of the given degree, joined to a core whose vertices all have a
    larger one, so that every root's list holds its whole neighbourhood."""
    rng = np.random.default_rng(1000 * degree + seed)
    i, j = np.nonzero(np.triu(rng.random((CORE, CORE)) < density, 1))
    src, dst = [i], [j]
    for r in range(ROOTS):
        src.append(np.full(degree, CORE + r))
        dst.append(rng.permutation(CORE)[:degree])
    src, dst = (np.concatenate(x).astype(np.uint32) for x in (src, dst))
    g = gpm.csr_from_edges(CORE + ROOTS + ISOLATED, src, dst)
    d = gpm.orient(g)
    deg = d.degrees()
    assert (deg[CORE:CORE + ROOTS] == degree).all()
    # the rule of vertex_tiers, and that the order is topological
    met = (deg.astype(float) ** 2).sum() / deg.sum()
    assert met >= 2.0 * deg.sum() / d.n
    s, t = np.repeat(np.arange(d.n), deg), d.adj.astype(np.int64)
    total = g.degrees()
    assert ((total[s] < total[t]) | ((total[s] == total[t]) & (s < t))).all()
    return d


def check(gpm, orc, d):
    want = orc.tc(d.offsets, d.adj)
    with gpm.DeviceGraph(d, oriented=True) as dg:
        assert dg.tc(gpm.TC_VERTEX) == want
        names = [name for name, _ in dg.kernel_breakdown()]
        assert dg.tc(gpm.TC_VERTEX) == want
        assert dg.tc_repeat(gpm.TC_VERTEX, 3) == want
    return names


@pytest.mark.parametrize("degree", [2, 3, 7, 8, 9, 15, 16, 17, 18, 63, 64, 65, 255, 256, 257, 300, 700])
def test_root_degrees(gpm, orc, degree):
    """Around the groups of 8 and 16 lanes, windows of 64 entries, batches and blocks of
    256; the core's lists are from 0 to 800 and more long."""
    check(gpm, orc, cored(gpm, degree, 0.9))


@pytest.mark.parametrize("degree", [17, 20, 40])
def test_long_lists_are_searched(gpm, orc, degree):
    """Streamed roots of which some lists are more than 16 times as long as theirs."""
    d = cored(gpm, degree, 0.9, 1)
    deg = d.degrees()
    first = d.offsets[CORE].astype(np.int64)
    met = deg[d.adj[first:first + ROOTS * degree]]
    assert (met > 16 * degree).sum() > 50 and (met <= 16 * degree).sum() > 50
    check(gpm, orc, d)


@pytest.mark.parametrize("most", [16, 17])
def test_small_roots(gpm, orc, most):
    """No vertex has more than 16 later neighbours, so nothing is streamed; or 17."""
    rng = np.random.default_rng(5)
    n, core = 3000, 200
    ring = np.arange(core)
    src = [np.repeat(np.arange(core, n), most)] + [ring] * 7
    dst = [np.concatenate([rng.permutation(core)[:most] for _ in range(core, n)])]
    dst += [(ring + k) % core for k in range(1, 8)]
    g = gpm.csr_from_edges(20 * n, np.concatenate(src).astype(np.uint32), np.concatenate(dst).astype(np.uint32))
    d = gpm.orient(g)
    assert d.degrees().max() == most
    names = check(gpm, orc, d)
    assert ("tc_vertex_block" in names) == (most > 16) and "tc_vertex_wave" in names


@pytest.mark.parametrize("degree", [9, 17, 64, 257])
def test_an_order_that_is_not_by_degree(gpm, orc, degree):
    """Roots that come before a chain of the core in every order but have the larger
    total degree: the clique count leaves an order behind that the triangle count uses."""
    rng = np.random.default_rng(degree)
    core = 600
    i, j = np.nonzero(np.triu(rng.random((core, core)) < 0.1, 1))
    src, dst = [ROOTS + i], [ROOTS + j]
    for r in range(ROOTS):
        src.append(np.full(degree, r))
        dst.append(ROOTS + rng.permutation(core)[:degree])
    src, dst = (np.concatenate(x).astype(np.uint32) for x in (src, dst))
    d = gpm.csr_from_edges(ROOTS + core + ISOLATED, src, dst, gpm.CSR_SORT)
    want = orc.tc(d.offsets, d.adj)
    with gpm.DeviceGraph(d, oriented=True) as dg:
        assert dg.tc(gpm.TC_VERTEX) == want  # hash kernels
        assert dg.clique(3) == want          # Kahn's order
        assert dg.tc(gpm.TC_VERTEX) == want  # the kernels above, on that order
        if 16 < degree <= 256:
            assert "tc_vertex_block" in [name for name, _ in dg.kernel_breakdown()]
