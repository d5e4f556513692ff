"""GPU parity of the fixed patterns' list kernels and the block mask with the oracle:
graphs whose ids reach past 16384, the most the bit matrices take, spread over the
mask's 64 blocks and gathered in one."""
import numpy as np
import pytest

import graphs

pytestmark = pytest.mark.gpu

PAST_MATRICES = 16385


def cases(gpm):
    return {
        "er_small": graphs.er(40, 160, 1),
        "er_dense": graphs.er(30, 200, 2),
        "wheel": graphs.wheel(130),
        "complete": graphs.complete(12),
        "bipartite": graphs.complete_bipartite(9, 14),
        "hubs": gpm.rmat_graph(9, 6, 3),
    }


def place(gpm, g, ids, n):
    """The graph on n vertices with vertex v renamed ids[v]."""
    src = np.repeat(np.arange(g.n), g.degrees())
    return gpm.csr_from_edges(n, ids[src].astype(np.uint32), ids[g.adj].astype(np.uint32))


@pytest.mark.parametrize("name", ["er_small", "er_dense", "wheel", "complete", "bipartite", "hubs"])
@pytest.mark.parametrize("n,spread", [(PAST_MATRICES, True), (PAST_MATRICES, False), (70001, True)])
def test_lists_vs_oracle(gpm, orc, name, n, spread):
    small = cases(gpm)[name]
    ids = np.random.default_rng(n).permutation(n)[:small.n] if spread else n - small.n + np.arange(small.n)
    g = place(gpm, small, ids, n)
    with gpm.DeviceGraph(g, oriented=False) as dg:
        for pid in range(1, 9):
            p, want = f"P{pid}", orc.pattern(g.offsets, g.adj, pid)
            out, scalar = dg.pattern(p, gpm.FORM_G2MINER)
            assert scalar == want and out[0] == want, p
            out, scalar = dg.pattern(p, gpm.FORM_PATTERN)
            assert scalar == want and out[0] == want, p
            if pid in (2, 3, 7, 8):
                assert out[1] - out[2] == want, p
            out, scalar = dg.pattern(p, gpm.FORM_BLOCK_PREFILTER)
            assert scalar == want and out[0] == want, p
            if pid in (4, 5, 6):
                assert out[1] == want, p
        assert dg.pattern("Motif4", gpm.FORM_G2MINER)[0] == orc.motif4(g.offsets, g.adj)
