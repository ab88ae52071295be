"""Candidate pairs of a quarter sector reused between rebuilds, on the GPU (run on an MI355X): bodies cross both
faces while the others drift within the skin, so lists built before a turn, across it and long after it are
used; contact sets bit for bit and forces within 1e-5 of the oracle's, with turns before and after detection,
with a skin wide enough for several steps, the default one and none."""
import numpy as np
import pytest

from oracle_binding import oracle_sim
from parity import step_and_compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("skin", [2e-3, -1.0, 0.0])
@pytest.mark.parametrize("wrap_after", [True, False])
def test_reused_sector_pairs_match_oracle(L, S, skin, wrap_after):
    sc = S.scene_c2(n=500, n_types=3, n_grid=24, n_nodes=128, cell_xy=0.05, gap=-0.15, seed=23)
    sc.cfg.update(periodic_x=0, periodic_y=0, periodic_sector=1, gravity=(0.0, 0.0, 0.0), skin=skin)
    sc.cfg["quirks"] = L.QUIRK_ALL if wrap_after else L.QUIRK_ALL & ~4
    P = sc.particles
    rng = np.random.default_rng(23)
    P["vel"][:, :2] = rng.normal(0.0, 1.0, (sc.n_particles, 2))
    lo = np.array(sc.cfg["domain_min"])
    near_x = P["pos"][:, 0] - lo[0] < 6e-3
    near_y = P["pos"][:, 1] - lo[1] < 6e-3
    P["vel"][near_x, 0] = -25.0  # across x = min within a few steps
    P["vel"][near_y & ~near_x, 1] = -25.0
    gpu = sc.load(L.Sim(sc.cfg))
    ref = sc.load(oracle_sim(sc.cfg))
    gpu.profile_begin(40)
    counts, worst = step_and_compare(gpu, ref, 40, lists=(0, 1, 2, 3, 4), log=print)
    prof = gpu.profile_end()
    ghost = sum(c["gx"] + c["gy"] + c["gxy"] for c in counts)
    print("rebuilds", prof["rebuilds"], "image contacts", ghost, "worst", worst)
    assert ghost > 0
    if skin > 0:
        assert prof["rebuilds"] <= 30  # (the premise: lists are reused)
    assert np.abs(gpu.get_particles()["quat"] - ref.get_particles()["quat"]).max() < 1e-12
