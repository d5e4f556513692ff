"""GPU: 4-cycle walks over middle vertices with few entries below the root, which the
lanes read by themselves, mixed with longer ones, against the oracle and, for K(a, m),
the closed form."""
import numpy as np
import pytest

from test_gpu_motif_bands import motif4

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mids", [3, 64, 700, 3000])
def test_mixed_lengths(gpm, orc, mids):
    """Middles of 1 - 7 of 7 hubs: 0 - 6 entries below a root, with tasks of the hash
    table (few middles) and of the counters."""
    rng = np.random.default_rng(mids)
    k = rng.integers(1, 8, mids)
    dst = np.concatenate([rng.permutation(7)[:x] for x in k])
    src = 7 + np.repeat(np.arange(mids), k)
    g = gpm.csr_from_edges(7 + mids, src.astype(np.uint32), dst.astype(np.uint32))
    assert motif4(gpm, g) == orc.motif4(g.offsets, g.adj)


@pytest.mark.parametrize("hubs", [2, 3, 4])
def test_two_sides(gpm, hubs):
    """K(a, m): every list but the hubs' has a entries."""
    m = 5000
    src, dst = np.repeat(np.arange(hubs), m), np.tile(hubs + np.arange(m), hubs)
    g = gpm.csr_from_edges(hubs + m, src.astype(np.uint32), dst.astype(np.uint32))
    deg = g.degrees()
    cycles = hubs * (hubs - 1) // 2 * (m * (m - 1) // 2)
    star = int((deg * (deg - 1) * (deg - 2) // 6).sum())
    path = int(((deg[src] - 1) * (deg[dst] - 1)).sum())
    assert motif4(gpm, g) == [star, path - 4 * cycles, 0, cycles, 0, 0]
