"""Orientation by entries against the host's, where its steps and words end: graphs
around 64 and 2048 entries, long runs of isolated vertices, hubs, no edges; and
edge lists the build refuses."""
import numpy as np
import pytest

import graphs

pytestmark = pytest.mark.gpu


def spread(gpm, n, m, gap):
    """m edges of a star over vertices gap apart, and a path at the end."""
    leaves = np.arange(1, m + 1, dtype=np.uint32) * gap
    assert int(leaves[-1]) < n
    return gpm.csr_from_edges(n, np.zeros(m, np.uint32), leaves)


@pytest.mark.parametrize("case", ["none", "one", "star31", "star32", "star33", "star1024",
                                  "star1025", "gaps", "complete65", "er", "rmat"])
def test_orient(gpm, case):
    g = {"none": lambda: gpm.csr_from_edges(70, [], []),
         "one": lambda: gpm.csr_from_edges(2, [0], [1]),
         "star31": lambda: spread(gpm, 40, 31, 1), "star32": lambda: spread(gpm, 40, 32, 1),
         "star33": lambda: spread(gpm, 40, 33, 1), "star1024": lambda: spread(gpm, 1025, 1024, 1),
         "star1025": lambda: spread(gpm, 1026, 1025, 1),
         "gaps": lambda: spread(gpm, 400000, 300, 1300),
         "complete65": lambda: graphs.complete(65), "er": lambda: gpm.er_graph(5000, 40000, 2),
         "rmat": lambda: gpm.rmat_graph(13, 12, 3)}[case]()
    want = gpm.orient(g)
    with gpm.DeviceGraph(g, oriented=False) as dg, dg.orient() as dag:
        got = dag.to_host()
        assert dag.info()[2] == int(np.diff(np.asarray(want.offsets).astype(np.int64)).max(initial=0))
    assert np.array_equal(got.offsets, want.offsets)
    assert np.array_equal(got.adj, want.adj)


@pytest.mark.parametrize("at", [0, 63, 999])
@pytest.mark.parametrize("bad", [100, 0xFFFFFFFF])
def test_build_refuses_endpoints(gpm, at, bad):
    s = np.arange(1000, dtype=np.uint32) % 100
    d = (s * 7 + 1).astype(np.uint32) % 100
    for flags in (gpm.CSR_CLEAN, 0):
        for side in (s, d):
            broken = side.copy()
            broken[at] = bad
            args = (broken, d) if side is s else (s, broken)
            with pytest.raises(gpm.GpmError):
                gpm.DeviceGraph.build(100, *args, flags)
