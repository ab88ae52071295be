"""Masters with more candidates than the search keeps, near periodic faces: searched a second time, partners
first and images after them, into their own part of the pair list.  Contacts against the oracle, and the lists of
the two launch forms against each other."""
import numpy as np
import pytest

from oracle_binding import oracle_sim
from parity import step_and_compare

pytestmark = pytest.mark.gpu


def _scene(S, periodic):
    n = 1200
    rng = np.random.default_rng(5)
    shapes = []
    h = 2.0 / 15
    sdf, org = S.superellipsoid_grid(1, 1, 1, 1, 1, 20, h)
    S._add_shape(shapes, sdf, org, h, S.superellipsoid_nodes(1, 1, 1, 1, 1, 64), 2500.0)
    P = S._particles(n)
    side = 0.04
    P["scale"][:] = np.where(np.arange(n) % 50 == 7, 8e-3, 7e-4)
    P["pos"][:] = rng.uniform(0.0, side, (n, 3))
    P["quat"][:] = rng.normal(size=(n, 4))
    P["quat"][:] /= np.linalg.norm(P["quat"], axis=1, keepdims=True)
    P["inv_mass"][:] = 1e3
    P["inv_inertia"][:] = np.array([1e9, 1e9, 1e9, 0.0, 0.0, 0.0])
    P["kn"][:], P["ks"][:], P["mu"][:], P["e"][:] = 10.0, 4.0, 0.3, 0.5
    # (max.y >= max.z, as the ghost test wants it)
    cfg = {"domain_min": (0, 0, 0), "domain_max": (side, side, side), "dt": 1e-7, **periodic}
    return S.Scene(cfg=cfg, shapes=shapes, particles=P, walls=S._walls_dict(0))


@pytest.mark.parametrize("launches", [0, 1])
@pytest.mark.parametrize("periodic", [{"periodic_x": 1, "periodic_y": 1}, {"periodic_sector": 1}], ids=["xy", "sector"])
def test_images_of_large_masters(L, S, periodic, launches):
    sc = _scene(S, periodic)
    gpu = sc.load(L.Sim({**sc.cfg, "broad_phase_launches": launches}))
    ref = sc.load(oracle_sim(sc.cfg))
    counts, _ = step_and_compare(gpu, ref, 2, lists=(0, 2, 3, 4), ctol=1e-9)
    got = gpu.pairs()
    per = np.bincount(got["master"], minlength=sc.n_particles)
    images = np.bincount(got["master"][got["type"] >= 2], minlength=sc.n_particles)
    assert ((per > 32) & (images > 0)).sum() >= 5  # (the premise)
    assert sum(c["pp"] for c in counts) > 0
    other = sc.load(L.Sim({**sc.cfg, "broad_phase_launches": 1 - launches}))
    other.step(2)
    for k, v in other.pairs().items():
        assert np.array_equal(v, got[k]), k
