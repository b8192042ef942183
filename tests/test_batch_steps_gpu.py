"""Batches whose instances advance together (multigrid preconditioner), at the sizes where the
launch shapes change: meshes without coarse levels, rows and columns around a segment and a
block, one and two separators per scan lane, lines too long for the scan (persistent kernel)."""
import numpy as np
import pytest

import oracle as O
from hip_runtime import memory_used
from plask_amd import workloads
from plask_amd.batch import PROGRESS, ShockleyBatch
from plask_amd.fem import FemError

pytestmark = pytest.mark.gpu


def _instance(n0, n1, seed, junction=True):
    rng = np.random.default_rng(seed)
    r = np.r_[0.0, np.cumsum(rng.uniform(0.5, 1.5, n0 - 1))]
    z = np.r_[0.0, np.cumsum(rng.uniform(0.05, 0.15, n1 - 1))]
    E0 = n0 - 1
    sig = np.exp(rng.uniform(np.log(10.0), np.log(1e3), n1 - 1))
    sh, sv = np.repeat(sig, E0), np.repeat(sig, E0)
    jlo = (n1 - 1) // 2
    jhi = jlo + 1 if junction else jlo
    sh[jlo * E0:jhi * E0], sv[jlo * E0:jhi * E0] = 0.0, 5.0
    # contact over the top row but its last node, the whole bottom row, one fixed node on the side
    top = (n1 - 1) * n0 + np.arange(n0 - 1)
    side = [(n1 // 2) * n0 + n0 - 1] if n1 > 4 else []
    dn = np.r_[np.arange(n0), top, side].astype(np.int64)
    dv = np.r_[np.zeros(n0), np.full(len(top), 1.5), np.full(len(side), 0.4)]
    return dict(axes=[r, z], sh=sh, sv=sv, dir_nodes=dn, dir_vals=dv, jlo=jlo, jhi=jhi, beta=8.0, js=1.0)


def _oracle(p, loops):
    r, z = p["axes"]
    g = O.Grid([r, z], cyl=True)
    E0 = len(r) - 1
    elems = np.arange(p["jlo"] * E0, p["jhi"] * E0)
    J = []
    if len(elems):
        bot = [[e % E0 + p["jlo"] * len(r), e % E0 + 1 + p["jlo"] * len(r)] for e in elems]
        top = [[e % E0 + p["jhi"] * len(r), e % E0 + 1 + p["jhi"] * len(r)] for e in elems]
        J = [dict(elems=elems, bottom=bot, top=top, height=z[p["jhi"]] - z[p["jlo"]], beta=p["beta"], js=p["js"])]
    return O.electrical_compute(g, p["sh"].copy(), p["sv"].copy(), p["dir_nodes"], p["dir_vals"], J, loops, maxerr=0.0)


@pytest.mark.parametrize("sizes", [
    [(2, 2), (2, 3), (3, 8), (3, 9), (2, 40)],                    # no coarse level
    [(4, 7), (4, 8), (5, 17), (9, 16), (33, 64), (65, 65)],       # segments of axis 1, tails
    [(300, 8), (513, 5), (600, 9), (129, 33), (30, 3)],           # widest sweep blocks
    [(7, 512), (12, 513), (5, 521), (20, 528), (3, 1032)],        # 63 to 128 separators
    [(20, 130), (4, 1033), (2, 2)],                               # a line too long for the scan
])
def test_steps_match_oracle(sizes):
    """CG stops at 1e-13 of each loop's start residual, so the potentials agree with the direct
    solve to the conditioning of the systems times that, as in the other batch tests: 1e-8."""
    insts = [_instance(n0, n1, 10 * k + n1, junction=(k % 3 != 1 and n1 > 2)) for k, (n0, n1) in enumerate(sizes)]
    b = ShockleyBatch(insts)
    print("batch steps", sizes, flush=True)
    for _ in range(2):  # the second solve replays the graphs on the state the first one left
        V, stats, _t = b.solve(maxloops=3, maxerr=1e-30, rtol=1e-13, precond=3)
        for size, p, v, s in zip(sizes, insts, V, stats):
            Vr, loops = _oracle(p, 3)[0], _oracle(p, 3)[4]
            assert s["status"] in (0, 2) and s["loops"] <= 3, (size, s)
            assert np.abs(v - Vr).max() <= 1e-8 * np.abs(Vr).max(), (size, np.abs(v - Vr).max(), s)


def test_steps_progress_and_options():
    """progress comes after every loop_budget loops; loop and iteration limits end the loop with
    the status of the persistent kernel; block and nwg choose nothing here."""
    insts = [_instance(20 + 9 * k, 40 + 11 * k, k) for k in range(4)]
    b = ShockleyBatch(insts)
    seen = []
    o = b.opts(maxloops=5, maxerr=1e-30, rtol=1e-12, loop_budget=2)
    o.progress = PROGRESS(lambda *a: seen.append(a[:3]))
    b.opts = lambda **kw: o
    V, stats, _t = b.solve()
    del b.opts
    assert [s[0] for s in seen] == [1, 2, 3] and seen[-1][1:] == (4, 4), seen
    V2, stats2, _t = b.solve(maxloops=5, maxerr=1e-30, rtol=1e-12, block=256, nwg=3)
    for a, c in zip(V, V2):
        assert np.array_equal(a, c)
    # iteration limit in every loop, error limit never met and met at once
    for maxerr in (1e-30, 1e9):
        kw = dict(maxloops=5, maxit=2, maxerr=maxerr, rtol=1e-12)
        st, sp = b.solve(precond=3, **kw)[1], b.solve(precond=2, **kw)[1]
        for a, c in zip(st, sp):
            assert (a["status"], a["loops"], a["iters"]) == (c["status"], c["loops"], c["iters"]), (a, c)


def test_autotune_keeps_the_persistent_schedule():
    """The persistent kernel's tuned schedule outlives an autotune of the step-by-step solve, which
    has none to choose (600 devices of 4 x 7 nodes: the fewest threads and most workgroups win)."""
    b = ShockleyBatch([_instance(4, 7, k) for k in range(600)])
    kw = dict(maxloops=4, maxerr=1e-30)
    tuned = b.autotune(precond=2, **kw)[:2]
    steps = b.autotune(precond=3, **kw)
    print("tuned", tuned, "after the steps", steps[:2], flush=True)
    assert steps[2] > 0 and steps[:2] == tuned


def test_tables_come_with_the_first_multigrid_solve():
    """The tables of the step-by-step solve are built by the first solve that uses them, which takes
    more than five values per node.  Where they pass the limit the persistent kernel solves the batch:
    no memory beyond what its line-preconditioned solve has taken (the runtime's scratch memory for
    that kernel and stream), the same statuses, and potentials to the conditioning of the systems
    times the tolerance (1e-8, as above)."""
    kw = dict(maxloops=2, maxerr=1e-30, rtol=1e-13)
    sizes = [(150 + 37 * k, 410 + 60 * k) for k in range(6)]
    insts = [_instance(n0, n1, k) for k, (n0, n1) in enumerate(sizes)]
    nodes = sum(n0 * n1 for n0, n1 in sizes)
    print("step tables", sizes, flush=True)

    def growth(batch):
        batch.solve(precond=2, maxloops=1, maxit=20)
        at = memory_used()
        V, stats, _t = batch.solve(precond=3, **kw)
        values = (memory_used() - at) / (8.0 * nodes)
        print("grows by %.2f values per node" % values, flush=True)
        return V, stats, values

    b = ShockleyBatch(insts)
    V, stats, values = growth(b)
    assert values > 5
    with pytest.raises(FemError, match="before the first multigrid solve"):
        b.set_step_memory(-1)
    for limit in (0, 3 * 8 * nodes):  # none of the tables, and some of them
        p = ShockleyBatch(insts)
        p.set_step_memory(limit)
        Vp, sp, values = growth(p)
        assert values < 1
        for v, q, s, r in zip(V, Vp, stats, sp):
            assert s["status"] == r["status"] and s["loops"] == r["loops"], (s, r)
            assert np.abs(v - q).max() <= 1e-8 * np.abs(v).max()
        tuned = p.autotune(precond=3, **kw)
        assert tuned[2] > 0
        p.close()


# seeds of stiff devices (conductivities over seven decades) whose CG stops with a true residual
# above its recursive one, so that the loop asks for a second run
STIFF = (3000, 3005, 3008, 3009, 3011)


def _stiff_and_easy():
    stiff = [workloads.shockley_cyl_batch(n_inst=1, seed0=s, nr_range=(12, 40), nz_range=(30, 70))[0] for s in STIFF]
    easy = [_instance(20 + 3 * k, 40 + 5 * k, k) for k in range(4)]
    insts, is_stiff = [], []
    for k in range(5):  # next to each other in the launches
        for group, name in ((stiff, True), (easy, False)):
            if k < len(group):
                insts.append(group[k])
                is_stiff.append(name)
    return insts, np.array(is_stiff)


@pytest.mark.parametrize("loops", [1, 4])
def test_second_runs_of_stiff_instances(loops):
    """CG starts once more from the true residual where that has not followed the recursive one: in
    the first loop for the stiff devices and for no easy one, while the others wait.  Restarts as in
    the persistent kernel in the first loop (later ones start from potentials that differ by rounding),
    statuses and loops as with the line preconditioner, potentials as the oracle's (1e-8, as above)."""
    insts, stiff = _stiff_and_easy()
    kw = dict(maxloops=loops, maxerr=1e-30, rtol=1e-12)
    print("second runs", loops, flush=True)
    b = ShockleyBatch(insts)
    p = ShockleyBatch(insts)
    p.set_step_memory(0)  # the persistent kernel
    line = b.solve(precond=2, **kw)[1]
    for _ in range(2):  # the second solve replays the graphs on the state of the first
        V, stats, _t = b.solve(precond=3, **kw)
        restarts = np.array([s["restarts"] for s in stats])
        print("restarts", restarts, flush=True)
        assert (restarts[stiff] > 0).all()
        if loops == 1:
            assert (restarts[~stiff] == 0).all()
            assert restarts.tolist() == [s["restarts"] for s in p.solve(precond=3, **kw)[1]]
        for q, v, s, r in zip(insts, V, stats, line):
            Vr = _oracle(q, loops)[0]
            assert (s["status"], s["loops"]) == (r["status"], r["loops"]) == (2, loops)
            assert np.abs(v - Vr).max() <= 1e-8 * np.abs(Vr).max(), (np.abs(v - Vr).max(), s)


def test_steps_as_plain_launches(monkeypatch):
    """Without graphs (as under a tracing profiler, whose environment turns them off) the same bits."""
    insts, _ = _stiff_and_easy()
    kw = dict(maxloops=4, maxerr=1e-30, rtol=1e-12, precond=3)
    print("plain launches", flush=True)
    V, stats, _t = ShockleyBatch(insts).solve(**kw)
    monkeypatch.setenv("ROCPROF_OUTPUT_PATH", "x")  # read when a batch is created
    p = ShockleyBatch(insts)
    monkeypatch.delenv("ROCPROF_OUTPUT_PATH")
    for _ in range(2):
        Vp, sp, _t = p.solve(**kw)
        assert stats == sp
        for v, q in zip(V, Vp):
            assert np.array_equal(v, q)
