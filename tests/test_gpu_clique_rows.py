"""GPU parity: k-clique counts where the row build and the k = 5 count can go
wrong: out-degrees around the edges of a 16-position block, a 64-bit row word
and a 128-position chunk, sparse and dense local graphs, hub ids inside and
outside the id bitmap, and orders that are not by degree."""
from math import comb

import numpy as np
import pytest

import graphs

pytestmark = pytest.mark.gpu


def hub_dag(gpm, degree, density, seed, tail=0):
    """A hub with `degree` out-neighbours, a random DAG of the given density
    among them, and a second layer that the first half of them points to;
    `tail` further vertices carry edges that keep the ids apart."""
    rng = np.random.default_rng(seed)
    n = 1 + 2 * degree + tail
    src, dst = [np.zeros(degree, np.int64)], [np.arange(1, degree + 1)]
    i, j = np.nonzero(np.triu(rng.random((degree, degree)) < density, 1))
    src.append(1 + i)
    dst.append(1 + j)
    i, j = np.nonzero(rng.random((degree // 2, degree)) < 0.2)
    src.append(1 + i)
    dst.append(1 + degree + j)
    if tail:
        src.append(1 + 2 * degree + np.arange(tail - 1))
        dst.append(2 + 2 * degree + np.arange(tail - 1))
    src, dst = np.concatenate(src).astype(np.uint32), np.concatenate(dst).astype(np.uint32)
    return gpm.csr_from_edges(n, src, dst, gpm.CSR_DEDUP | gpm.CSR_SORT)


@pytest.mark.parametrize("degree", [65, 80, 81, 127, 128, 129, 192, 255, 257, 383, 385, 511, 512, 513, 640, 769, 1000])
def test_hub_degrees_vs_oracle(gpm, orc, degree):
    for density, seed in ((0.02, 1), (0.25, 2)) + (((0.9, 3),) if degree < 130 else ()):
        d = hub_dag(gpm, degree, density, 100 * degree + seed)
        want = [orc.clique(d.offsets, d.adj, k) for k in (3, 4, 5)]
        with gpm.DeviceGraph(d, oriented=True) as dg:
            assert [dg.clique(k) for k in (3, 4, 5)] == want, density
            assert list(dg.clique_all()) == want, density
            parts = [dg.clique(5, policy=gpm.SCHED_DEGREE_SPLIT), dg.clique_all(policy=gpm.SCHED_DEGREE_SPLIT)[2]]
            assert parts == [want[2]] * 2, density


@pytest.mark.parametrize("tail", [32768 - 2 * 300 - 1, 32768 - 2 * 300, 32768 - 300, 100000])
def test_ids_below_the_bitmap(gpm, orc, tail):
    """The hub's neighbours sit at, across and below the first id of the
    bitmap (the order falls back to Kahn's: the tail comes last)."""
    d = hub_dag(gpm, 300, 0.3, tail, tail=tail)
    want = [orc.clique(d.offsets, d.adj, k) for k in (3, 4, 5)]
    with gpm.DeviceGraph(d, oriented=True) as dg:
        assert [dg.clique(k) for k in (3, 4, 5)] == want
        assert list(dg.clique_all()) == want


def test_degree_order_and_kahn_agree(gpm, orc):
    """A degree-oriented graph is relabelled by degree on the device; the same
    DAG with its ids permuted ties differently and takes the host's order."""
    g = gpm.rmat_graph(13, 16, 9)
    d = gpm.orient(g)
    want = [orc.clique(d.offsets, d.adj, k) for k in (3, 4, 5)]
    perm = np.random.default_rng(5).permutation(d.n).astype(np.uint32)
    src = np.repeat(np.arange(d.n, dtype=np.uint32), d.degrees())
    p = gpm.csr_from_edges(d.n, perm[src], perm[d.adj], gpm.CSR_SORT)
    for dag in (d, p):
        with gpm.DeviceGraph(dag, oriented=True) as dg:
            assert list(dg.clique_all()) == want
            assert dg.clique(5, policy=gpm.SCHED_DEGREE_SPLIT) == want[2]


@pytest.mark.parametrize("n", [3, 4, 11, 12, 13, 24, 63, 64, 65, 66])
def test_wave_tier_complete(gpm, n):
    """Roots of 1 .. n - 1 later vertices: one and several windows of row searches."""
    with gpm.DeviceGraph(gpm.orient(graphs.complete(n)), oriented=True) as dag:
        for k in (3, 4, 5):
            assert dag.clique(k) == comb(n, k)


@pytest.mark.parametrize("met", [2, 3, 13, 40])
def test_wave_tier_long_lists(gpm, met):
    """500 vertices joined to `met` of a complete graph's 200 each: lists far longer
    than the roots'."""
    core, m = graphs.complete(200), 500
    src = np.repeat(np.arange(200), 199)
    outer = np.repeat(200 + np.arange(m), met)
    inner = (np.arange(m)[:, None] * 7 + np.arange(met) * (200 // met)).reshape(-1) % 200
    g = gpm.csr_from_edges(200 + m, np.concatenate([src, outer]), np.concatenate([core.adj, inner]))
    with gpm.DeviceGraph(gpm.orient(g), oriented=True) as dag:
        for k in (3, 4, 5):
            assert dag.clique(k) == comb(200, k) + m * comb(met, k - 1)


@pytest.mark.parametrize("degree", [65, 96, 97, 300, 512, 700, 1000])
def test_k4_split(gpm, orc, degree):
    """4-cliques of hubs cut into parts of row blocks, more of them than row blocks too."""
    d = hub_dag(gpm, degree, 0.3, degree)
    want = orc.clique(d.offsets, d.adj, 4)
    with gpm.DeviceGraph(d, oriented=True) as dg:
        assert dg.clique(4) == want
        assert dg.clique(4, policy=gpm.SCHED_DEGREE_SPLIT) == want
