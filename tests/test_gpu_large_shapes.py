"""Shapes whose narrow-phase LDS lets two blocks or one on a compute unit (more than 15 and more than 30 clusters of
nodes), with more pairs than wavefronts fit, in the batches the library chooses: against the oracle, and against batches
of one pair bit for bit."""
import numpy as np
import pytest

from oracle_binding import oracle_sim
from parity import step_and_compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nodes,side", [(1100, 13), (2200, 10)])
def test_automatic_batches(L, S, nodes, side):
    shapes = []
    h = 2.0 / 19
    sdf, org = S.superellipsoid_grid(1, 1, 1, 0.5, 0.5, 26, h)
    S._add_shape(shapes, sdf, org, h, S.superellipsoid_nodes(1, 1, 1, 0.5, 0.5, nodes), 2500.0)
    n = side ** 3
    P = S._particles(n)
    k = np.arange(n)
    P["pos"][:] = np.stack([k % side, k // side % side, k // side ** 2], 1) * 3.996e-3 + 0.01  # 4 um into one another
    P["scale"][:] = 2e-3
    P["quat"][:] = (1.0, 0.0, 0.0, 0.0)
    P["vel"][:] = np.random.default_rng(nodes).normal(0.0, 0.01, (n, 3))
    P["inv_mass"][:] = 1.0 / (shapes[0]["mass"] * 2e-3 ** 3)
    P["inv_inertia"][:] = shapes[0]["inv_inertia"] / 2e-3 ** 5
    P["kn"][:], P["ks"][:], P["mu"][:], P["e"][:] = 1e5, 4e4, 0.5, 0.5
    cfg = {"domain_min": (0, 0, 0), "domain_max": (0.08, 0.08, 0.08), "dt": 2e-7, "no_certificates": 1}
    sc = S.Scene(cfg=cfg, shapes=shapes, particles=P, walls=S._walls_dict(0))
    gpu = sc.load(L.Sim(sc.cfg))
    counts, _ = step_and_compare(gpu, sc.load(oracle_sim(sc.cfg)), 3, lists=(0,))
    assert counts[0]["pp"] > 1000
    clusters = 15 if nodes == 1100 else 30
    assert nodes > 64 * clusters and gpu.counters()["pairs"] > 256 * 4 * (2 if nodes == 1100 else 1)  # (the premises)
    one = sc.load(L.Sim({**sc.cfg, "narrow_batch": 1}))
    one.step(3)
    a, b = gpu.get_particles(), one.get_particles()
    for key in ("pos", "quat", "vel", "angvel", "force", "torque"):
        assert np.array_equal(a[key], b[key]), key
