"""Inputs checked where the device reads them: list order of the set primitives (with
the entry that breaks it), finite features of the work estimator, and outputs packed
or copied whole."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def lists(sizes, start=1000):
    """Increasing lists, each beginning below the end of the one before it."""
    return [np.arange(start - 3 * i, start - 3 * i + n, dtype=np.uint32) for i, n in enumerate(sizes)]


@pytest.mark.parametrize("side", [0, 1])
@pytest.mark.parametrize("at", [(0, 1), (0, 64), (2, 1), (4, 299), (5, 1), (6, 1999)])
@pytest.mark.parametrize("equal", [False, True])
def test_order_of_lists(gpm, side, at, equal):
    sizes = [65, 0, 2, 1, 300, 2, 2000, 0]
    good = lists(sizes)
    other = lists([3] * len(sizes), 50)
    pairs = list(zip(*((good, other) if side == 0 else (other, good))))
    counts, _ = gpm.setops(gpm.SETOP_ISECT_COUNT, 0, pairs)
    assert counts.tolist() == [0] * len(sizes)
    k, i = at
    broken = [x.copy() for x in good]
    broken[k][i] = broken[k][i - 1] - (0 if equal else 1)
    pairs = list(zip(*((broken, other) if side == 0 else (other, broken))))
    with pytest.raises(gpm.GpmError) as e:
        gpm.setops(gpm.SETOP_ISECT_COUNT, 0, pairs)
    assert f"list {'AB'[side]} is not strictly increasing at entry {sum(sizes[:k]) + i}" in str(e.value)


@pytest.mark.parametrize("keep", [0, 1, 3, 4, 5, 64])
def test_short_and_long_results(gpm, keep):
    """keep of every 64 entries of A are in B: results packed below a quarter."""
    rng = np.random.default_rng(keep)
    pairs = []
    for n in (0, 1, 63, 64, 65, 640, 5000):
        a = np.cumsum(rng.integers(1, 5, n)).astype(np.uint32)
        pairs.append((a, a[np.arange(n) % 64 < keep]))
    pairs.append((pairs[5][0][:10], pairs[6][0]))  # B longer than A
    _, got = gpm.setops(gpm.SETOP_ISECT, 0, pairs)
    assert all(np.array_equal(g, np.intersect1d(a, b)) for g, (a, b) in zip(got, pairs))
    _, got = gpm.setops(gpm.SETOP_DIFF, 0, pairs)
    assert all(np.array_equal(g, np.setdiff1d(a, b)) for g, (a, b) in zip(got, pairs))
    _, got = gpm.setops(gpm.SETOP_FUSE, 0, pairs)
    for (ga, gab, gb), (a, b) in zip(got, pairs):
        assert np.array_equal(ga, np.setdiff1d(a, b))
        assert np.array_equal(gab, np.intersect1d(a, b))
        assert np.array_equal(gb, np.setdiff1d(b, a))


@pytest.mark.parametrize("n", [1, 16, 17, 1000, 40000])
@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf, -1.0, -2.0])
def test_features(gpm, n, bad):
    rng = np.random.default_rng(n)
    p = [np.zeros(4), np.ones(4), rng.normal(size=(64, 4)), np.zeros(64),
         rng.normal(size=(64, 64)), np.zeros(64), rng.normal(size=(1, 64)), np.zeros(1)]
    feat = rng.uniform(0, 100, (n, 4)).astype(np.float32)
    feat[0] = [np.finfo(np.float32).max, -0.5, 0, 1]
    assert gpm.mlp_predict(feat, *p).shape == (n,)
    for row, col in ((0, 0), (n - 1, 3), (n // 2, 2)):
        broken = feat.copy()
        broken[row, col] = bad
        with pytest.raises(gpm.GpmError):
            gpm.mlp_predict(broken, *p)
