"""Warm-start network at ragged and small volumes: x extents that are no multiple of a brick's 16,
fewer rows than a brick, and sizes on either side of each launch shape of the convolutions."""
import numpy as np
import pytest

from oracle import warmnet as W

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.linalg.norm(np.asarray(a, dtype=np.float64) - b) / max(np.linalg.norm(b), 1e-30))


@pytest.mark.parametrize("shape", [(4, 8, 64), (8, 4, 64), (20, 8, 64), (36, 32, 64), (72, 64, 32)])
def test_ragged_volumes_match_oracle(shape):
    """Bounds of the existing forward / gradient test: bf16 rounding at the same points on both
    sides, other summation orders (1e-2 forward, 3e-2 per gradient block)."""
    from plask_amd import warmstart
    nx, ny, nz = shape
    rng = np.random.default_rng(5)
    p = warmstart.init_params(7)
    off = 0
    for ci, co in W.LAYERS:
        off += 27 * ci * co
        p[off:off + co] = rng.normal(0.0, 0.05, co)
        off += co
    x = rng.standard_normal((nz, ny, nx, 8)).astype(np.float32)
    t = rng.standard_normal((nz, ny, nx)).astype(np.float32)
    print("warmnet shapes", shape, flush=True)
    net = warmstart.WarmNet(shape, max_samples=1)
    net.set_params(p)
    net.set_loss(0.0)
    net.set_sample(0, x.reshape(-1, 8), t.ravel())
    y_gpu = net.predict_sample(0)
    loss_gpu, g_gpu = net.gradient(0)
    loss, g, y = W.loss_grad(p.astype(np.float64), x.astype(np.float64), t.astype(np.float64), rb=True, lam=0.0)
    assert _rel(y_gpu, y.ravel()) <= 1e-2
    assert abs(loss_gpu - loss) <= 1e-2 * loss
    off = 0
    for ci, co in W.LAYERS:
        for n in (27 * ci * co, co):
            assert _rel(g_gpu[off:off + n], g[off:off + n]) <= 3e-2, (ci, co, n)
            off += n
    assert _rel(g_gpu[off:], g[off:]) <= 1e-2
