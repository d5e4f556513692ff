"""GPU: the fixed patterns on one-sided lists (an unsymmetrised edge file) and lists
with loops give the same numbers on the bit matrices' graphs as on lists."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LIST_PATH = 20000  # vertices: past the matrices' limit


@pytest.mark.parametrize("n,m,mutual,loops", [(30, 200, 0.0, 0), (200, 1500, 0.0, 0), (200, 2500, 0.5, 0),
                                              (90, 1200, 0.98, 0), (64, 700, 1.0, 5), (150, 1500, 0.5, 5)])
def test_one_sided_lists(gpm, n, m, mutual, loops):
    rng = np.random.default_rng(n + m)
    src, dst = rng.integers(0, n, m), (rng.random(m) ** 2 * n).astype(np.int64)
    both = rng.random(m) < mutual
    own = rng.permutation(n)[:loops]
    keep = src != dst
    src, dst = (np.concatenate([src[keep], dst[keep & both], own]).astype(np.uint32),
                np.concatenate([dst[keep], src[keep & both], own]).astype(np.uint32))
    flags = gpm.CSR_SORT | gpm.CSR_DEDUP
    small, big = (gpm.csr_from_edges(k, src, dst, flags) for k in (n, LIST_PATH))
    with gpm.DeviceGraph(small, oriented=False) as a, gpm.DeviceGraph(big, oriented=False) as b:
        for form in (gpm.FORM_G2MINER, gpm.FORM_PATTERN, gpm.FORM_BLOCK_PREFILTER):
            for p in ["P%d" % i for i in range(1, 9)] + ["Motif4"]:
                assert a.pattern(p, form) == b.pattern(p, form), (p, form)
