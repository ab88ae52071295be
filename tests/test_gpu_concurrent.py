"""Contexts stepped at once from several host threads with the broad phase's automatic grid: no barrier gives up
(an error with no_recovery), and every state is that of the context stepped alone."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [600, 4000])
def test_contexts_at_once(L, S, n):
    scs = []
    for k in range(6):
        sc = S.scene_c2(n=n, n_types=2, n_grid=24, n_nodes=96, cell_xy=0.1, gap=-0.1, seed=40 + k)
        sc.particles["vel"][:, :2] = np.random.default_rng(k).normal(0.0, 3.0, (n, 2))  # rebuilds and wraps
        sc.cfg["no_recovery"] = 1
        scs.append(sc)
    at_once, alone = ([sc.load(L.Sim(sc.cfg)) for sc in scs] for _ in range(2))
    errs = []

    def run(sim):
        try:
            for _ in range(5):
                sim.step(20)
        except Exception as ex:  # reported below
            errs.append(ex)
    th = [threading.Thread(target=run, args=(s,)) for s in at_once]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not errs, errs
    for k, (a, b) in enumerate(zip(at_once, alone)):
        b.step(100)
        pa, pb = a.get_particles(), b.get_particles()
        for key in ("pos", "quat", "vel", "angvel", "force", "torque"):
            assert np.array_equal(pa[key], pb[key]), f"context {k}: {key} differs"
