"""The end of a step at the edges of its blocks, on the GPU (run on an MI355X): a block of its own closes the
step's counters beside the body blocks, full ones or with one body in the last.  Steps in one call, one by one
and with separate launches leave the same state and counters."""
import numpy as np
import pytest

from oracle_binding import oracle_sim
from parity import compare_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block", [0, 64])
@pytest.mark.parametrize("n", [1, 64, 255, 256, 257])
def test_counters_and_state(L, S, n, block):
    sc = S.scene_c2(n=n, n_types=3, n_grid=20, n_nodes=64, cell_xy=0.03, gap=-0.2, seed=n)
    sc.cfg["block_size"] = block
    many = sc.load(L.Sim(sc.cfg))
    single = sc.load(L.Sim(sc.cfg))
    plain = sc.load(L.Sim({**sc.cfg, "no_fused_steps": 1}))
    ref = sc.load(oracle_sim(sc.cfg))
    for x in (many, plain, single):
        x.profile_begin(6)
    many.step(6)
    plain.step(6)
    for _ in range(6):
        single.step(1)
    ref.step(6)
    a = many.get_particles()
    for other in (plain, single):
        b = other.get_particles()
        for k in ("pos", "quat", "vel", "angvel", "force", "torque"):
            assert np.array_equal(a[k], b[k]), k
        assert many.counters() == other.counters()
    work = [{k: v for k, v in x.profile_end().items() if isinstance(v, int)} for x in (many, plain, single)]
    assert work[0] == work[1] == work[2]
    compare_state(a, ref.get_particles())
