"""Operator, line preconditioner and V-cycle at the sizes where the default launch shapes and the
separator scan change: few and many rows per tile, one plane per block, 24 segments in a scan of
32 lanes, one and two separators per lane, lines too long for the scan."""
import numpy as np
import pytest

import oracle as O
from oracle import multigrid as MG
from plask_amd.fem import PF_FP32_RELIABLE, PF_FP64, PRECOND_LINE, PRECOND_MG, FemContext

pytestmark = pytest.mark.gpu


def _problem(shape, cyl=False):
    rng = np.random.default_rng(sum(shape))
    axes = [np.cumsum(np.r_[0.0, rng.uniform(0.05, 2.0, n - 1)]) for n in shape]
    g = O.Grid(axes, cyl=cyl)
    kh, kv = rng.uniform(0.5, 150.0, g.nelems), rng.uniform(0.5, 150.0, g.nelems)
    plane = g.nnodes // shape[-1]
    dn = np.r_[np.arange(plane), rng.choice(np.arange(plane, g.nnodes), 3, replace=False)].astype(np.int64)
    c = FemContext()
    c.set_grid(axes, cylindrical=cyl)
    c.set_coeffs(kh, kv)
    c.set_source(np.zeros(g.nelems))
    c.set_dirichlet(dn, np.full(len(dn), 300.0))
    return g, axes, kh, kv, dn, c


@pytest.mark.parametrize("shape", [(2, 2, 2), (17, 17, 5), (25, 19, 37), (128, 3, 9), (300, 2, 3), (65, 65, 8),
                                   (2, 3), (33, 63), (33, 64), (33, 257), (700, 65), (300, 201), (600, 401),
                                   (1000, 1001)])
def test_default_launch_shapes_apply(shape):
    """y = A x (FP64) against the oracle's element sums: rounding of 27 products, 1e-13 of the largest."""
    g, axes, kh, kv, dn, c = _problem(shape)
    print("launch shapes apply", shape, flush=True)
    mask = np.zeros(g.nnodes, np.uint8)
    mask[dn] = 1
    x = np.random.default_rng(1).uniform(-1, 1, g.nnodes)
    ref = O.apply(g, 0, kh, kv, mask, x)
    y = c.apply(x)
    assert np.abs(y - ref).max() <= 1e-13 * np.abs(ref).max()
    c.close()


@pytest.mark.parametrize("rows", [1, 2, 3, 4, 7, 64])
def test_rows_per_thread_2d(rows):
    """The 2D operator with every unrolling and with remainders: plain (as above) and fused into
    CG, whose solutions of one system (cond ~1e5, rtol 1e-12) agree to 1e-7 of their size."""
    g, axes, kh, kv, dn, c = _problem((33, 65), cyl=True)
    print("rows per thread", rows, flush=True)
    mask = np.zeros(g.nnodes, np.uint8)
    mask[dn] = 1
    x = np.random.default_rng(1).uniform(-1, 1, g.nnodes)
    c.set_source(np.random.default_rng(3).uniform(0, 1e16, g.nelems))
    ref_t, _ = c.solve(x0=np.full(g.nnodes, 300.0), precision=PF_FP64, rtol=1e-12, precond=PRECOND_LINE)
    c.set_launch(16, rows)
    ref = O.apply(g, 0, kh, kv, mask, x)
    assert np.abs(c.apply(x) - ref).max() <= 1e-13 * np.abs(ref).max()
    for prec in (PF_FP64, PF_FP32_RELIABLE):
        t, st = c.solve(x0=np.full(g.nnodes, 300.0), precision=prec, rtol=1e-12 if prec == PF_FP64 else 1e-10,
                        precond=PRECOND_LINE)
        assert st.status == 0 and np.abs(t - ref_t).max() <= 1e-7 * np.abs(ref_t).max()
    c.close()


@pytest.mark.parametrize("shape", [(4, 10000), (2, 4097), (7, 5001)])
def test_default_rows_can_be_set_2d(shape):
    """A tall narrow grid takes one row per thread by default (fewer than 60000 nodes): the same shape
    set by hand gives the same bits, and so does one of few long marches to the rounding of the operator."""
    g, axes, kh, kv, dn, c = _problem(shape)
    print("rows by hand", shape, flush=True)
    x = np.random.default_rng(1).uniform(-1, 1, g.nnodes)
    y = c.apply(x)
    c.set_launch(16, 1)
    assert np.array_equal(c.apply(x), y)
    c.set_launch(16, shape[1])
    assert np.abs(c.apply(x) - y).max() <= 1e-13 * np.abs(y).max()
    c.set_launch(16, 1)
    t, st = c.solve(x0=np.full(g.nnodes, 300.0), precision=PF_FP64, rtol=1e-10, precond=PRECOND_LINE)
    assert st.status == 0 and np.abs(t - 300.0).max() <= 300.0 * 1e-6
    c.close()


@pytest.mark.parametrize("rows,planes", [(2, 1), (3, 1), (4, 1), (4, 7), (31, 40)])
def test_reductions_over_many_blocks(rows, planes):
    """Grid reductions of one block, of 64 and less (one ticket) and of more (group tickets, the
    last group short): every launch shape gives the same CG solve, cond ~1e5, rtol 1e-12."""
    g, axes, kh, kv, dn, c = _problem((11, 30, 40))
    c.set_source(np.random.default_rng(3).uniform(0, 1e16, g.nelems))
    print("reductions", rows, planes, flush=True)
    kw = dict(x0=np.full(g.nnodes, 300.0), precision=PF_FP64, rtol=1e-12)
    ref, s0 = c.solve(precond=PRECOND_LINE, **kw)
    c.set_launch(rows, planes)
    for precond in (PRECOND_LINE, PRECOND_MG):
        t, st = c.solve(precond=precond, **kw)
        assert st.status == 0 and np.abs(t - ref).max() <= 1e-7 * np.abs(ref).max()
        assert precond == PRECOND_MG or abs(st.iters - s0.iters) <= 2
    c.close()


@pytest.mark.parametrize("shape", [(3, 3, 192), (5, 4, 520), (4, 3, 521), (3, 4, 1024), (5, 520), (5, 521), (4, 1032),
                                   (4, 1033)])
def test_long_lines_vcycle(shape):
    """One V-cycle against the CPU statement of it (its line solves are direct): 1e-10 in FP64,
    norm-wise 1e-3 with FP32 line solves, as in the other V-cycle tests."""
    g, axes, kh, kv, dn, c = _problem(shape)
    print("long lines", shape, flush=True)
    r = np.random.default_rng(2).uniform(-1, 1, g.nnodes)
    r[dn] = 0.0
    z_ref = MG.VCycle(axes, kh, kv, dn).apply(r)
    z = c.precond_apply(r, PF_FP64, PRECOND_MG)
    assert np.abs(z - z_ref).max() <= 1e-10 * np.abs(z_ref).max()
    z32 = c.precond_apply(r, PF_FP32_RELIABLE, PRECOND_MG)
    assert np.linalg.norm(z32 - z_ref) <= 1e-3 * np.linalg.norm(z_ref)
    c.set_line_segment(-1)
    zl = c.precond_apply(r, PF_FP64, PRECOND_LINE)
    c.set_line_segment(0)
    assert np.abs(c.precond_apply(r, PF_FP64, PRECOND_LINE) - zl).max() <= 1e-10 * np.abs(zl).max()
    c.close()


@pytest.mark.parametrize("rtol", [1e-3, 1e-6, 1e-8, 1e-10, 1e-12])
def test_last_iterations_in_a_short_graph(rtol):
    """The stop is met at another iteration of the chunk for every rtol; whether the last ones run
    in the chunk's graph or in the short one, iterations and bits are those of checks every 2."""
    g, axes, kh, kv, dn, c = _problem((17, 15, 24))
    c.set_source(np.random.default_rng(3).uniform(0, 1e16, g.nelems))
    print("short graph", rtol, flush=True)
    kw = dict(x0=np.full(g.nnodes, 300.0), precision=PF_FP64, precond=PRECOND_MG)
    for _ in range(3):  # replayed, and with another tolerance between
        a, sa = c.solve(rtol=rtol, **kw)
        c.solve(rtol=1e-5, **kw)
    b, sb = c.solve(rtol=rtol, check_every=2, **kw)
    assert sa.iters == sb.iters and np.array_equal(a, b)
    c.close()


def test_first_solves_of_a_grid():
    """The short last part of a solve runs as plain launches, is captured and is replayed in the first
    three solves after a grid is set: all have the iterations and bits of checks every 2."""
    g, axes, kh, kv, dn, c = _problem((17, 15, 24))
    kw = dict(x0=np.full(g.nnodes, 300.0), precision=PF_FP64, precond=PRECOND_MG, rtol=1e-9)
    q = np.random.default_rng(3).uniform(0, 1e16, g.nelems)
    print("first solves", flush=True)
    c.set_source(q)
    ref, sr = c.solve(check_every=2, **kw)
    for _ in range(2):
        c.set_grid(axes)
        c.set_coeffs(kh, kv)
        c.set_source(q)
        c.set_dirichlet(dn, np.full(len(dn), 300.0))
        for _ in range(4):
            t, st = c.solve(**kw)
            assert st.iters == sr.iters and np.array_equal(t, ref)
    c.close()
