"""GPU: the bit matrix patterns on graphs of several 2048-id segments: lists of ids gathered
over segments, sets past one list, and sets of a few ids, against the list kernels
(isolated vertices past the matrices' limit) and closed forms."""
from math import comb

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PIDS = ["P%d" % i for i in range(1, 9)]
LIST_PATH = 17000


def both_paths(gpm, n, src, dst, jobs):
    src, dst = np.asarray(src, np.uint32), np.asarray(dst, np.uint32)
    small, big = (gpm.csr_from_edges(k, src, dst) for k in (n, LIST_PATH))
    with gpm.DeviceGraph(small, oriented=False) as a, gpm.DeviceGraph(big, oriented=False) as b:
        for p, form in jobs:
            assert a.pattern(p, form) == b.pattern(p, form), (p, form)


def hubs(m, n, seed):
    """Two adjacent hubs over m leaves, ids spread over n."""
    ids = np.random.default_rng(seed).permutation(n)[:m + 4].astype(np.int64)
    h1, h2, leaves, rest = ids[0], ids[1], ids[2:m + 2], ids[m + 2:]
    src = np.concatenate([[h1], np.full(m, h1), np.full(m, h2)])
    return h1, h2, leaves, rest, src, np.concatenate([[h2], leaves, leaves])


@pytest.mark.parametrize("m,n", [(2047, 4100), (2048, 4096), (2049, 4096), (2500, 8300), (4090, 4096),
                                 (6000, 16384)])
def test_sets_past_a_list(gpm, m, n):
    """A hub's leaves are R1, R2 and the columns of P3, and of P7 for the hubs' own edge."""
    _, _, _, _, src, dst = hubs(m, n, m)
    g = gpm.csr_from_edges(n, src.astype(np.uint32), dst.astype(np.uint32))
    with gpm.DeviceGraph(g, oriented=False) as dg:
        for form in (gpm.FORM_G2MINER, gpm.FORM_PATTERN):
            assert dg.pattern("P3", form)[1] == 2 * m * comb(m, 3)
            assert dg.pattern("P7", form)[1] == 2 * comb(m, 3)


@pytest.mark.parametrize("m,n", [(600, 4097), (2100, 4100), (2100, 16384)])
def test_hubs_on_both_paths(gpm, m, n):
    """The hubs with a pendant each, and a matching on some of their leaves."""
    h1, h2, leaves, rest, src, dst = hubs(m, n, m + n)
    src = np.concatenate([src, rest, leaves[:40:2]])
    dst = np.concatenate([dst, [h1, h2], leaves[1:40:2]])
    both_paths(gpm, n, src, dst, [(p, f) for p in ("P1", "P2", "P4", "P5", "P6", "P8")
                                  for f in ((0,) if p in ("P1", "P4") else (0, 1))])


@pytest.mark.parametrize("n,degree", [(2049, 17), (4096, 25), (4200, 24), (6144, 30), (9001, 34), (16384, 46)])
def test_near_uniform_lists(gpm, n, degree):
    """Sets of a few ids a segment, common neighbours of none to a few."""
    s, d = gpm.gen_er(n, n * degree // 2, n)
    jobs = [(p, f) for p in PIDS for f in (0, 1) if (p, f) not in (("P1", 1), ("P4", 1))] + [("P4", 2), ("Motif4", 0)]
    both_paths(gpm, n, s, d, jobs)


@pytest.mark.parametrize("n,size", [(4500, 12), (9000, 30), (16000, 50)])
def test_communities(gpm, n, size):
    """Dense groups whose ids lie in every segment: as many common neighbours as others."""
    rng = np.random.default_rng(n)
    ids = rng.permutation(n)
    src, dst = [], []
    for at in range(0, n - size, 6 * size):
        i, j = np.nonzero(np.triu(rng.random((size, size)) < 0.8, 1))
        src.append(ids[at + i])
        dst.append(ids[at + j])
    hub = np.full(n // 20, ids[-1])  # takes the graph over the matrices' line
    src.append(hub)
    dst.append(rng.integers(0, n, n // 20))
    both_paths(gpm, n, np.concatenate(src), np.concatenate(dst), [(p, f) for p in PIDS for f in (0, 1)])
