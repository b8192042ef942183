"""FP32 forms: where a quantity is a double rounded once, the results show one rounding."""
import numpy as np
import pytest

from hip_runtime import DeviceArray
from plask_amd.fem import PF_FP32_REFINE, PF_FP32_RELIABLE, PF_FP64, PRECOND_LINE, FemContext

pytestmark = pytest.mark.gpu

U = 2.0 ** -24  # unit roundoff of FP32


@pytest.mark.parametrize("shape", [(40, 33, 3), (25, 30, 9), (21, 20, 16), (600, 13)])
def test_line_factors_round_once(shape):
    """Lines of one segment (at most 16 planes) with a load on the last plane only: the forward sweep
    is zero below it, and the back substitution is z_k = -c'_k z_(k+1), so the ratios of neighbouring
    planes show c'.  FP64 gives them to 1e-13; in FP32 they may be off by the rounding of c' and that
    of the product, 2 U, and not by the roundings of two factors that make up c'."""
    rng = np.random.default_rng(sum(shape))
    c = FemContext()
    c.set_grid([np.cumsum(np.r_[0.0, rng.uniform(0.3, 2.0, n - 1)]) for n in shape])
    ne, nn, nz = int(np.prod([n - 1 for n in shape])), int(np.prod(shape)), shape[-1]
    plane = nn // nz
    c.set_coeffs(rng.uniform(0.5, 50.0, ne), rng.uniform(0.5, 50.0, ne))
    c.set_source(np.zeros(ne))
    c.set_dirichlet(np.arange(1, dtype=np.int64), np.full(1, 300.0))
    r = np.zeros((nz, plane))
    r[-1] = rng.uniform(0.5, 1.0, plane).astype(np.float32)
    print("line factors", shape, flush=True)
    z64, z32 = [c.precond_apply(r.ravel(), p, PRECOND_LINE).reshape(nz, plane)[:, 1:] for p in (PF_FP64, PF_FP32_RELIABLE)]
    c64, c32 = z64[:-1] / z64[1:], z32[:-1] / z32[1:]
    assert np.abs(z32).min() > 2.0 ** -100
    err = np.abs(c32 / c64 - 1.0)
    print("largest error %.3f U" % (err.max() / U), flush=True)
    assert err.max() <= 2.0 * U * (1.0 + 1e-5), err.max() / U
    c.close()


@pytest.mark.parametrize("rows", [1, 2, 5])
def test_layer_sizes_round_once_2d(rows):
    """2D operator without in-plane conductivity, kv = 1 and w = 12: next to a row of ones, (A x)_k is
    that of one layer, 3 (1 / h) times a power of two.  FP64 gives it to 1e-15; FP32 rounds 1 / h and
    its product with 3: 2 U."""
    nz = 3001
    z = np.cumsum(np.r_[0.0, np.random.default_rng(4).uniform(0.05, 2.0, nz - 1)])
    c = FemContext()
    c.set_grid([np.array([0.0, 12.0]), z])
    c.set_coeffs(np.zeros(nz - 1), np.ones(nz - 1))
    c.set_source(np.zeros(nz - 1))
    c.set_dirichlet(np.zeros(1, np.int64), np.full(1, 300.0))
    c.set_launch(16, rows)
    x = np.zeros((nz, 2))
    x[::3] = 1.0  # the rows between see one layer each
    print("layer sizes", rows, flush=True)
    ref = c.apply(x.ravel()).reshape(nz, 2)
    xd, yd = DeviceArray(x.ravel().astype(np.float32)), DeviceArray(np.zeros(2 * nz, np.float32))
    assert c.L.pf_apply(c.h, PF_FP32_REFINE, xd.ptr, yd.ptr) == 0
    y = yd.get().astype(np.float64).reshape(nz, 2)
    xd.close()
    yd.close()
    k = np.arange(1, nz - 1)[np.arange(1, nz - 1) % 3 != 0]
    err = np.abs(y[k] / ref[k] - 1.0)
    print("largest error %.3f U" % (err.max() / U), flush=True)
    assert err.max() <= 2.0 * U * (1.0 + 1e-5), err.max() / U
    c.close()
