"""The pair check at the edges of its tiles, on the GPU (run on an MI355X): lists of up to 131,072 pairs go in
tiles of 256 with a pair per thread, longer ones in tiles of 1024.  With and without certificates (few or all
pairs of a tile evaluated, one round of records or several) contacts and states are the same bit for bit, and
small systems match the oracle."""
import numpy as np
import pytest

from oracle_binding import oracle_sim
from parity import compare_contacts, compare_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 60, 600, 30000, 60000])
def test_tiles_agree(L, S, n):
    sc = S.scene_c2(n=n, n_types=3, n_grid=20, n_nodes=64, cell_xy=0.05 if n < 1000 else 0.15, gap=-0.15, seed=n)
    sc.particles["vel"][:] = np.random.default_rng(n).normal(0.0, 1.0, (n, 3))
    cert = sc.load(L.Sim(sc.cfg))
    full = sc.load(L.Sim({**sc.cfg, "no_certificates": 1}))
    ref = sc.load(oracle_sim(sc.cfg)) if n <= 600 else None
    for s in range(4):
        cert.step(1)
        full.step(1)
        for l in range(5):
            ca, cb = cert.contacts(l), full.contacts(l)
            for k in ca:
                assert np.array_equal(ca[k], cb[k]), f"step {s} list {l}: {k}"
        a, b = cert.get_particles(), full.get_particles()
        for k in ("pos", "quat", "vel", "angvel", "force", "torque"):
            assert np.array_equal(a[k], b[k]), f"step {s}: {k}"
        if ref is not None:
            ref.step(1)
            for l in range(2):
                compare_contacts(cert.contacts(l), ref.contacts(l), f"step {s} list {l}")
            compare_state(a, ref.get_particles())
    pairs = cert.counters()["pairs"]
    print("pairs", pairs)
    if n == 30000:
        assert 65536 < pairs <= 131072  # (the premises: one list on each side of the line)
    if n == 60000:
        assert pairs > 131072
