"""GPU: the 4-cycle tasks of the Motif4 identities that need many ranks: a root's first
and second band of ranks as tasks of their own and a third that reaches past its
band, with counters of 16 and of 32 bits.  Bipartite graphs, so that their
4-cycles can be counted by the pairs of one side."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BAND = {16: 2 * 39936, 32: 39936}  # ranks of a band of LDS counters
OWN_TASKS = 1 << 17                # wedges of a root whose second band is a task of its own


def pairs(x):
    return x * (x - 1) // 2


@pytest.mark.parametrize("bits,hubs,mids,ends,past", [(16, 2, 2000, 240000, True), (16, 5, 65535, 100000, False),
                                                      (32, 2, 66000, 160000, True), (32, 3, 70000, 45000, False)])
def test_ranks_past_two_bands(gpm, bits, hubs, mids, ends, past):
    """Hubs over all middle vertices, and ends of 2 - 5 of them: a hub's wedges end at
    every rank, the ends' being the lowest.  past: more than a band of ranks is left
    below the two, so some are counted in HBM."""
    rng = np.random.default_rng(mids + ends)
    k = rng.integers(2, 6, ends)
    x = np.repeat(np.arange(ends), k)
    m = rng.integers(0, mids, len(x))
    both = np.unique(x * mids + m)  # distinct (end, middle)
    x, m = both // mids, both % mids
    first_mid, first_hub = ends, ends + mids
    src = np.concatenate([x, np.repeat(first_hub + np.arange(hubs), mids)])
    dst = np.concatenate([first_mid + m, np.tile(first_mid + np.arange(mids), hubs)])
    g = gpm.csr_from_edges(first_hub + hubs, src.astype(np.uint32), dst.astype(np.uint32))
    deg = g.degrees()
    rank = np.empty(g.n, np.int64)
    rank[np.lexsort((np.arange(g.n), deg))] = np.arange(g.n)
    hub = rank[first_hub:]
    assert (hub >= first_hub).all() and len(x) >= OWN_TASKS
    # below a hub's two bands there are more ranks, and more than a band of them
    assert (hub.min() - 2 * BAND[bits] > BAND[bits]) == past and hub.min() > 2 * BAND[bits]
    assert (mids >= 65536) == (bits == 32)
    # Opposite pairs among ends and hubs: every end's middles are every hub's; two hubs
    # share all middles; two ends share those of equal pairs.
    kx = np.bincount(x, minlength=ends)
    keys = []
    start = np.concatenate([[0], np.cumsum(kx)[:-1]])
    for a in range(5):
        for b in range(a + 1, 5):
            has = kx > b
            keys.append(m[start[has] + a] * mids + m[start[has] + b])  # ascending within an end
    mult = np.unique(np.concatenate(keys), return_counts=True)[1]
    cycles = int(hubs * pairs(kx).sum() + pairs(hubs) * pairs(mids) + pairs(mult).sum())
    star = int((deg * (deg - 1) * (deg - 2) // 6).sum())
    path = int(((deg[src] - 1) * (deg[dst] - 1)).sum())
    with gpm.DeviceGraph(g, oriented=False) as dg:
        for _ in range(2):
            assert dg.pattern("Motif4", gpm.FORM_PATTERN)[0] == [star, path - 4 * cycles, 0, cycles, 0, 0]
