"""A quarter sector's candidate pairs at the default skin, the one users run, are reused too: bodies cross both faces
at 5 m/s, and there are no more rebuilds than turns and half skins travelled ask for.  (That contacts are the oracle's at
this skin, test_gpu_sector_reuse.py checks over as many steps as rounding differences stay within its bounds.)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_default_skin_reuses_pairs(L, S):
    sc = S.scene_c2(n=400, n_types=3, n_grid=24, n_nodes=128, cell_xy=0.05, gap=-0.05, seed=29)
    sc.cfg.update(periodic_x=0, periodic_y=0, periodic_sector=1, gravity=(0.0, 0.0, 0.0))
    P = sc.particles
    rng = np.random.default_rng(29)
    P["vel"][:] = rng.normal(0.0, 0.3, (sc.n_particles, 3))
    lo = np.array(sc.cfg["domain_min"])
    for axis in (0, 1):
        near = np.argsort(P["pos"][:, axis])[:10]
        P["vel"][near, axis] = -5.0
    steps = 260
    fast = (np.abs(P["vel"]).max(1) >= 5.0).sum()
    gpu = sc.load(L.Sim(sc.cfg))
    q0 = gpu.get_particles()["quat"].copy()
    gpu.profile_begin(steps)
    images = 0
    for _ in range(steps // 20):
        gpu.step(20)
        images += sum(len(gpu.contacts(l)["master"]) for l in (2, 3, 4))
    rebuilds = gpu.profile_end()["rebuilds"]
    turned = np.abs(np.abs(np.sum(q0 * gpu.get_particles()["quat"], axis=1)) - 1.0) > 0.05
    rad = max(np.linalg.norm(s["nodes"], axis=1).max() for s in sc.shapes if len(s["nodes"])) * P["scale"].max()
    travelled = steps * 5.0 * sc.cfg["dt"] / (0.5 * 0.08 * rad)  # half skins of the fastest body
    print("rebuilds", rebuilds, "turned", turned.sum(), "half skins", travelled)
    assert turned.sum() > 0 and images > 0
    # (twice the travel: the list is rebuilt for whichever body is first, and a body may be struck)
    assert rebuilds <= fast + 2 * np.ceil(travelled) + 2 < steps / 2
