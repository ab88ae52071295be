"""The narrow phase's contact lists at the edges of their layout, on the GPU against the oracle (run on an
MI355X): contact sets bit for bit, forces and torques within 1e-5 relative (parity.py).

A body's contact mask has a bit for each of its first 31 pairs and one for all others, as master and as
partner: bodies with 20, 31, 32 and 70 contacting neighbours, as the first and as the last body of the
list.  A batch keeps its first 128 candidate slots in LDS, takes slots 64 at a time and its sub-cluster
entries 64 at a time: flat faces of 1,500 nodes pressed together, in batches of 1, 2 and 8 pairs."""
import numpy as np
import pytest

from oracle_binding import oracle_sim
from parity import step_and_compare

pytestmark = pytest.mark.gpu


def _bodies(S, shapes, kind, pos, scale, cfg, vel):
    n = len(kind)
    P = S._particles(n)
    P["shape"], P["scale"], P["pos"], P["vel"] = np.asarray(kind, np.int32), np.asarray(scale, float), pos, vel
    P["quat"][:] = (1.0, 0.0, 0.0, 0.0)
    for i in range(n):
        sh = shapes[kind[i]]
        P["inv_mass"][i] = 1.0 / (sh["mass"] * scale[i] ** 3)
        P["inv_inertia"][i] = sh["inv_inertia"] / scale[i] ** 5
    P["kn"][:], P["ks"][:], P["mu"][:], P["e"][:] = 1e5, 4e4, 0.5, 0.5
    return S.Scene(cfg=cfg, shapes=shapes, particles=P, walls=S._walls_dict(0))


@pytest.mark.parametrize("neighbours", [20, 31, 32, 70])
@pytest.mark.parametrize("hub_first", [True, False])
def test_hub_with_many_contacts(L, S, neighbours, hub_first):
    shapes = []
    h = 2.0 / 27
    sdf, org = S.superellipsoid_grid(1, 1, 1, 1, 1, 34, h)
    for nodes in (4000, 100):  # the hub's, the neighbours'
        S._add_shape(shapes, sdf, org, h, S.superellipsoid_nodes(1, 1, 1, 1, 1, nodes), 2500.0)
    rng = np.random.default_rng(neighbours)
    d = S.fibonacci_directions(neighbours)
    small = 0.6e-3
    ring = (10e-3 + small - 2e-4) * d  # 0.2 mm into the hub, whose own nodes (as master) are 0.5 mm apart
    hub = np.zeros((1, 3))
    pos = np.concatenate([hub, ring] if hub_first else [ring, hub]) + 0.05
    scale = np.array([10e-3] + [small] * neighbours if hub_first else [small] * neighbours + [10e-3])
    vel = rng.normal(0.0, 0.05, (neighbours + 1, 3))
    cfg = {"domain_min": (0, 0, 0), "domain_max": (0.1, 0.1, 0.1), "gravity": (0, 0, -9.81), "dt": 1e-7}
    kind = [0] + [1] * neighbours if hub_first else [1] * neighbours + [0]
    sc = _bodies(S, shapes, kind, pos, scale, cfg, vel)
    ref = sc.load(oracle_sim(sc.cfg))
    counts, worst = step_and_compare(sc.load(L.Sim(sc.cfg)), ref, 6, lists=(0,), log=print)
    c = ref.contacts(0)
    assert len(np.unique(c["slave"] if hub_first else c["master"] // 100)) == neighbours
    print("worst", worst)


@pytest.mark.parametrize("narrow_batch", [1, 2, 8])
def test_many_candidates_in_a_batch(L, S, narrow_batch):
    shapes = []
    h = 2.0 / 35
    e = 2.0 / 8.0
    sdf, org = S.superellipsoid_grid(1, 1, 1, e, e, 42, h)
    S._add_shape(shapes, sdf, org, h, S.superellipsoid_nodes(1, 1, 1, e, e, 1500), 2500.0)
    k = np.arange(12)
    pos = np.stack([k % 3, k // 3 % 2, k // 6], 1) * 3.99e-3 + 0.01  # faces 10 um into one another
    vel = np.random.default_rng(3).normal(0.0, 0.01, (12, 3))
    cfg = {"domain_min": (0, 0, 0), "domain_max": (0.04, 0.04, 0.04), "dt": 2e-7, "narrow_batch": narrow_batch}
    sc = _bodies(S, shapes, [0] * 12, pos, [2e-3] * 12, cfg, vel)
    counts, worst = step_and_compare(sc.load(L.Sim(sc.cfg)), sc.load(oracle_sim({**sc.cfg, "narrow_batch": 0})), 5,
                                     lists=(0,), log=print)
    assert counts[0]["pp"] > 20 * 128  # 20 pairs of faces, most with more than 128 contacts
    print("worst", worst)
