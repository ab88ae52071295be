"""A wall that is set between two phases of a step is detected where it then is, contact arms and all: the contacts
equal those of a wall that its velocity carried to the same place."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_wall_set_before_the_narrow_phase(L, S):
    sc = S.scene_c2(n=300, n_types=2, n_grid=24, n_nodes=128, cell_xy=0.06, gap=-0.1, seed=11)
    sc.cfg["no_certificates"] = 1
    # the lowest bodies reach 0.2 mm into the floor
    P = sc.particles
    low = np.array([(sc.shapes[s]["nodes"] * k)[:, 2].min() for s, k in zip(P["shape"], P["scale"])])
    P["quat"][:] = (1.0, 0.0, 0.0, 0.0)
    bed = P["pos"][:, 2] < P["pos"][:, 2].min() + 1e-3
    P["pos"][bed, 2] = sc.walls["pos"][0, 2] - low[bed] - 2e-4
    P["vel"][:] = 0.0
    moved = {k: v.copy() for k, v in sc.walls.items()}
    moved["vel"][0] = 0.0, 0.0, 2.0
    there = moved["pos"] + sc.cfg["dt"] * moved["vel"]

    carried = S.Scene(cfg=sc.cfg, shapes=sc.shapes, particles=P, walls=moved).load(L.Sim(sc.cfg))
    put = sc.load(L.Sim(sc.cfg))
    for name in carried.STEP_PHASES:
        if name == "narrow":
            put.set_walls(pos=there)
            assert np.array_equal(carried.get_walls()["pos"], there)
        put.phase(name)
        carried.phase(name)
    a, b = put.contacts(L.LIST_PW), carried.contacts(L.LIST_PW)
    assert len(b["master"]) > 0
    for k in ("master", "slave", "overlap", "point", "normal"):
        assert np.array_equal(a[k], b[k]), k
