"""GPU: device memory of matching batches is given back."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


def free_bytes():
    hip = C.CDLL("/opt/rocm/lib/libamdhip64.so")  # the runtime libgpm is linked against
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_plan_trials_keep_nothing(gpm):
    """Batches of new queries under the learned policy, each tried on a sample of its
    plans: one label on 200000 vertices, so a trial holds 1.6 MB of roots a plan."""
    g = gpm.er_graph(200000, 400000, 3)
    path = [(i, i + 1) for i in range(7)]
    with gpm.DeviceGraph(g, oriented=False, labels=[0] * g.n, n_labels=1) as dg:
        # a path and chords that leave few embeddings
        batch = lambda k: [(8, path + [(0, 2), (1, 3), (2, 4 + k % 4), (0, 3 + k // 4)], [0] * 8)]  # noqa: E731
        dg.match_batch(batch(0), policy=1)
        before = free_bytes()
        for k in range(1, 16):
            dg.match_batch(batch(k), policy=1)
        assert before - free_bytes() < 8 << 20
