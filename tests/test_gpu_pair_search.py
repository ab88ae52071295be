"""The pair search at the edges of its layout, on the GPU (run on an MI355X): one 32-lane group searches a
master's neighbourhood, 32 grid rows and 4 x 32 items at a time from a list of 256, keeps the first 32
candidates in a slab and searches again beyond that; walls come from a mask of up to 64, beyond that a lane
each.  Against brute force over all pairs (every pair whose bounding spheres come within the skin, none
further apart), with the search's FP32 margin."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _scene(S, scale, pos, n_walls, side):
    shapes = []
    h = 2.0 / 15
    sdf, org = S.superellipsoid_grid(1, 1, 1, 1, 1, 20, h)
    S._add_shape(shapes, sdf, org, h, S.superellipsoid_nodes(1, 1, 1, 1, 1, 64), 2500.0)
    n = len(scale)
    P = S._particles(n)
    P["scale"], P["pos"] = scale, pos
    P["quat"][:, 0] = 1.0
    P["inv_mass"][:] = 1.0
    P["inv_inertia"][:] = np.array([1.0, 1.0, 1.0, 0.0, 0.0, 0.0])
    wsdf, wo, wh = S.plane_wall_shape(0.6 * side, 2.0 ** -7)
    wid = S._add_shape(shapes, wsdf, wo, wh, np.zeros((0, 3)))
    W = S._walls_dict(n_walls)
    W["shape"][:], W["radius"][:], W["quat"][:, 0] = wid, side, 1.0
    for k in range(n_walls):
        W["pos"][k] = 0.5 * side, 0.5 * side, -0.5 * side * k / n_walls
    cfg = {"domain_min": (0, 0, 0), "domain_max": (side, side, side), "dt": 1e-9}
    return S.Scene(cfg=cfg, shapes=shapes, particles=P, walls=W)


@pytest.mark.parametrize("launches", [0, 1])
@pytest.mark.parametrize("n,small,walls", [(1, 1e-3, 1), (31, 2e-3, 0), (33, 2e-3, 63), (700, 1e-3, 64), (700, 1e-3, 65),
                                           (2500, 4e-4, 3)])
def test_pairs_equal_brute_force(L, S, n, small, walls, launches):
    rng = np.random.default_rng(n + walls)
    side = 0.04
    scale = np.where(rng.random(n) < 0.02, 5e-3, small)  # a few large ones: hundreds of items, over 32 candidates
    pos = rng.uniform(0.0, side, (n, 3))
    sc = _scene(S, scale, pos, walls, side)
    sim = sc.load(L.Sim({**sc.cfg, "broad_phase_launches": launches}))
    sim.step(1)
    got = sim.pairs()
    r = scale * np.linalg.norm(sc.shapes[0]["nodes"], axis=1).max()
    skin = 0.08 * r.max()
    d = np.linalg.norm(pos[:, None] - pos[None], axis=2)
    reach = r[:, None] + r[None] + skin
    upper = np.triu(np.ones((n, n), bool), 1)
    pp = got["type"] == 0
    listed = np.zeros((n, n), bool)
    listed[got["master"][pp], got["partner"][pp]] = True
    assert pp.sum() == listed.sum()  # none twice
    assert not (upper & (d <= reach * (1 - 1e-12)) & ~listed).any()
    assert not (listed & ~(upper & (d <= reach * (1 + 4e-6) + 1e-6))).any()
    # walls: every particle within reach of a wall's plane inside its slab's extent is listed with it
    pw = got["type"] == 1
    near = np.abs(pos[:, None, 2] - sc.walls["pos"][None, :, 2]) <= r[:, None]
    wl = np.zeros((n, max(walls, 1)), bool)
    wl[got["master"][pw], got["partner"][pw]] = True
    assert pw.sum() == wl.sum()
    assert not (near[:, :walls] & ~wl[:, :walls]).any()
    # in order: masters ascending, particle partners before walls
    assert np.all(np.diff(got["master"]) >= 0)
    same = np.diff(got["master"]) == 0
    assert np.all(np.diff(got["type"])[same] >= 0)
    if n >= 2500:  # (the premise: masters that search a second time)
        assert np.bincount(got["master"], minlength=n).max() > 32
