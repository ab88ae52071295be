"""A full contact buffer on a grid of more blocks than the GPU holds at once: blocks start while others raise
the overflow, the call is restored, the buffer grown, and the results are those of a context that had the room."""
import numpy as np
import pytest

from parity import LISTS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("capacity", [1, 4000])
def test_overflow_with_more_blocks_than_fit(L, S, capacity):
    # 2,048 blocks of the narrow phase, of which three fit a compute unit
    sc = S.scene_c2(n=6000, n_types=3, n_grid=24, n_nodes=128, cell_xy=0.15, gap=-0.2, seed=31)
    ref = sc.load(L.Sim(sc.cfg))
    small = sc.load(L.Sim({**sc.cfg, "contact_capacity": capacity}))
    ref.step(6)
    small.step(6)
    a, b = small.get_particles(), ref.get_particles()
    for k in ("pos", "quat", "vel", "angvel", "force", "torque"):
        assert np.array_equal(a[k], b[k]), k
    total = 0
    for l in range(5):
        ca, cb = small.contacts(l), ref.contacts(l)
        total += len(cb["master"])
        for k in ca:
            assert np.array_equal(ca[k], cb[k]), f"{LISTS[l]}: {k}"
    assert ref.counters()["recoveries"] == 0
    assert total > capacity and small.counters()["recoveries"] >= 1
