"""One optimizer step of the culling surrogate at the edges of its layout, on the GPU (run on an MI355X): 64
samples per block and sixteen blocks' partial gradients read together, so one block, sixteen, seventeen and
thirty-three, against the FP64 restatement.  The samples are drawn again here from the kernel's hash; a first Adam
step moves each weight by the learning rate against its gradient's sign, which the gradients' bound (2e-2 of a
tensor's norm, as for the gradient itself) settles for every larger element."""
import sys
from pathlib import Path

import numpy as np
import pytest

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "oracle"))
import surrogate_ref as R  # noqa: E402

pytestmark = pytest.mark.gpu
SIZES = (("W1", (112, 64)), ("b1", (64,)), ("W2", (64, 64)), ("b2", (64,)), ("W3", (64, 64)), ("b3", (64,)),
         ("W4", (64, 64)), ("b4", (64,)), ("w5", (64,)), ("b5", (1,)), ("emb", (3, 16)))


def _hash(x):
    x = x + np.uint64(0x9E3779B97F4A7C15)
    x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return x ^ (x >> np.uint64(31))


def _samples(shapes, n, seed, inv_len, clamp):
    i = np.arange(n, dtype=np.uint64)
    h = [_hash(np.uint64(seed) ^ i)]
    h += [_hash(h[0])]
    h += [_hash(h[1])]
    x, t = np.empty((n, 3)), np.empty(n)
    slot = (i % np.uint64(len(shapes))).astype(np.int32)
    for k in range(n):
        sh = shapes[slot[k]]
        sdf = sh["sdf"].transpose(2, 1, 0)  # (stored z, y, x)
        dims = np.array(sdf.shape)
        if (k // len(shapes)) % 2 == 0:
            g = np.array([int(h[a][k]) % int(dims[a]) for a in range(3)], float)
        else:
            g = np.array([np.float32(int(h[a][k]) >> 40) * np.float32(2.0 ** -24) * np.float32(dims[a] - 1)
                          for a in range(3)], float)
        c = np.clip(np.floor(g), 0, dims - 2).astype(int)
        f = np.clip(g - c, 0, 1)
        v = sdf[c[0]:c[0] + 2, c[1]:c[1] + 2, c[2]:c[2] + 2].astype(float)
        v = v[0] * (1 - f[0]) + v[1] * f[0]
        v = v[0] * (1 - f[1]) + v[1] * f[1]
        t[k] = np.clip((v[0] * (1 - f[2]) + v[1] * f[2]) * inv_len, -clamp, clamp)
        x[k] = np.asarray(sh["origin"]) + g * sh["spacing"]
    return x.astype(np.float32).astype(np.float64), slot, t


def _unflatten(w):
    P, off = {}, 0
    for name, shape in SIZES:
        size = int(np.prod(shape))
        P[name] = w[off:off + size].astype(np.float64).reshape(shape)
        off += size
    return P


@pytest.mark.parametrize("batch", [64, 16 * 64, 17 * 64, 33 * 64])
def test_first_step_matches_oracle(L, S, batch):
    sc = S.scene_c2(n=600, n_types=3, n_grid=24, n_nodes=128, cell_xy=0.06, gap=-0.15)
    sim = sc.load(L.Sim(sc.cfg))
    lr, clamp, seed = 1e-3, 0.6, 5
    prm = dict(batch=batch, samples=batch, validation=64, lr=lr, lr_final=lr, clamp=clamp, seed=seed)
    sim.surrogate_train(iterations=0, **prm)
    w0 = sim.surrogate_weights(3)
    rep = sim.surrogate_train(iterations=1, **prm)
    w1 = sim.surrogate_weights(3)
    inv_len = np.float32(1.0 / rep["length_scale"])
    x, slot, t = _samples(sc.shapes[:3], batch, seed ^ 0x51, inv_len, clamp)
    loss, G, _ = R.loss_and_grads(_unflatten(w0), x, slot, t, inv_len, bf=True)
    assert rep["final_loss"] == pytest.approx(loss, rel=2e-3)
    step = _unflatten(w1.astype(np.float64) - w0.astype(np.float64))
    P0 = _unflatten(w0)
    for name, _shape in SIZES:
        g, d = np.asarray(G[name]).reshape(step[name].shape), step[name]
        sure = np.abs(g) > 2.1e-2 * np.linalg.norm(g)
        assert sure.any(), name
        tol = lr * (1e-8 / (np.abs(g[sure]) - 2e-2 * np.linalg.norm(g)) + 1e-5) + 1.2e-7 * (np.abs(P0[name][sure]) + lr)
        assert (np.abs(d[sure] + lr * np.sign(g[sure])) <= tol).all(), name
