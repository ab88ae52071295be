"""Batches of the narrow phase at the edges of a block's turns, on the GPU (run on an MI355X): a block's four
wavefronts take a batch each per turn and reserve their contact slots together, so blocks whose last turn is
partly or wholly empty, many turns of one block and every batch size, against one pair per batch on the default
grid, bit for bit, and against the oracle."""
import numpy as np
import pytest

from oracle_binding import oracle_sim
from parity import compare_contacts, compare_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [0, 1, 2, 4, 8])
@pytest.mark.parametrize("n,blocks", [(2, 1), (8, 3), (60, 1), (600, 7)])
def test_turns_agree(L, S, n, blocks, batch):
    sc = S.scene_c2(n=n, n_types=3, n_grid=20, n_nodes=64, cell_xy=0.02 if n < 20 else 0.05, gap=-0.25, seed=n)
    sc.cfg["no_certificates"] = 1  # (every pair is evaluated every step)
    one = sc.load(L.Sim({**sc.cfg, "narrow_batch": 1}))
    sim = sc.load(L.Sim({**sc.cfg, "narrow_batch": batch, "narrow_blocks": blocks}))
    ref = sc.load(oracle_sim(sc.cfg))
    for s in range(3):
        for x in (one, sim, ref):
            x.step(1)
        for l in range(5):
            ca, cb = sim.contacts(l), one.contacts(l)
            for k in ca:
                assert np.array_equal(ca[k], cb[k]), f"step {s} list {l}: {k}"
        for l in range(2):
            compare_contacts(sim.contacts(l), ref.contacts(l), f"step {s} list {l}")
        a, b = sim.get_particles(), one.get_particles()
        for k in ("pos", "quat", "vel", "angvel", "force", "torque"):
            assert np.array_equal(a[k], b[k]), f"step {s}: {k}"
        compare_state(a, ref.get_particles())
