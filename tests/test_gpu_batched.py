"""GPU tests of the batched solver: every problem of an uneven batch agrees
with the CPU oracle run on that problem alone (same start vector, same
algorithm), in FP64 and in mixed precision, with either sweep kernel (a
workgroup per problem, or lock-step over row chunks) and the autotuner."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _problems(sa, orc):
    from slepc_amd.batch import uneven_laplacians
    P = uneven_laplacians(P=7, seed=2, lo=20, hi=70)
    return P


@pytest.mark.parametrize("sweep", ["persistent", "wide", "auto"])
@pytest.mark.parametrize("mixed", [False, True])
def test_batched_matches_oracle(sa, orc, mixed, sweep):
    from slepc_amd.batch import Batch
    csrs = _problems(sa, orc)
    v0 = [orc.rand_uniform(orc.sub_seed(9, p), A.n) for p, A in enumerate(csrs)]
    B = Batch(csrs)
    B.set_sweep(sweep)
    B.solve(8, 24, 1e-10, "LM", mixed=mixed, v0=v0)
    info = B.sweep_info()
    assert info["mode"] == (sweep if sweep != "auto" else info["mode"]) and info["mode"] in ("persistent", "wide")
    if sweep == "auto":
        assert info["ms_persistent"] > 0 and info["ms_wide"] > 0
    err = B.errors()
    for p, A in enumerate(csrs):
        nconv, its, reason = B.converged(p)
        assert reason == 1 and nconv >= 8
        Ao = orc.CSR(A.n, A.rowptr, A.col, A.val)
        r = orc.eps_solve(Ao, 8, 24, 1e-10, "LM", True, v0=v0[p])
        vals = np.array([B.eigenpair(p, i, False)[0] for i in range(8)])
        w = np.linalg.eigvalsh(Ao.to_dense())
        for v in vals:
            assert np.min(np.abs(w - v)) < 1e-10 * abs(v)
        assert np.allclose(np.sort(vals), np.sort(r["eigr"][:8]), rtol=1e-10, atol=0)
        if not mixed:
            assert abs(its - r["its"]) <= max(2, 0.2 * r["its"])
        assert np.all(err[p] <= 1e-10), err[p]
    st = B.stats()
    assert st["matvecs"] > 0 and (st["matvecs32"] > 0) == mixed


def _chain(sa, n, seed):
    """A symmetric tridiagonal matrix of n rows with a few separated ends."""
    rng = np.random.default_rng(seed)
    d = rng.uniform(1.0, 2.0, n)
    d[rng.choice(n, min(n, 8), replace=False)] += 2.0 + np.arange(min(n, 8))
    e = rng.uniform(0.1, 0.3, n - 1)
    r = np.concatenate([np.arange(n), np.arange(n - 1), np.arange(1, n)])
    c = np.concatenate([np.arange(n), np.arange(1, n), np.arange(n - 1)])
    v = np.concatenate([d, e, e])
    o = np.lexsort((c, r))
    rp = np.zeros(n + 1, np.int32)
    rp[1:] = np.cumsum(np.bincount(r, minlength=n))
    return sa.CSR(n, rp, c[o].astype(np.int32), v[o])


# rows of the problems, ncv, precision: one problem of a block and one of a row
# more; all that one launch takes and more (256 workgroups); a basis of 32, 33
# and 63 columns; rows that take every size of row block (4, 8, 11, 16, 22 chunks)
RESIDENT = [
    ([256], 24, False), ([257, 40, 1024, 1025], 32, False), ([300] * 256 + [290], 20, False),
    ([511, 90, 64, 65], 33, True), ([4097, 130], 63, False), ([250000, 100], 16, False),
    ([20000] * 9, 24, False), ([20000] * 17 + [33], 24, True)]


def check_resident(sa, rows, ncv, mixed, ran):
    """The resident sweep and the lock-step one give the same eigenvalues (both
    have converged to the tolerance) and error estimates below it.  ran: how
    the sweeps asked to be resident are to have run."""
    from slepc_amd.batch import Batch
    csrs = [_chain(sa, n, 7 + i % 5) for i, n in enumerate(rows)]
    out = []
    for sweep in ("persistent", "wide"):
        B = Batch(csrs)
        B.set_sweep(sweep)
        B.solve(4, ncv, 1e-10, "LM", mixed=mixed)
        assert B.sweep_info()["mode"] == ("persistent" if sweep == "persistent" and ran == "resident" else "wide")
        assert all(B.converged(p)[2] == 1 for p in range(len(rows)))
        assert np.all(B.errors() <= 1e-10)
        out.append(np.array([[B.eigenpair(p, i, False)[0] for i in range(4)] for p in range(len(rows))]))
        counts = B.sweep_counts()
        if sweep == "persistent" and ran == "gave_up":     # and then not tried for a while
            assert counts["resident"] == 0 and counts["gave_up"] >= 1, counts
        else:
            assert counts[ran if sweep == "persistent" else "slots"] == sum(counts.values()) > 0
    assert np.allclose(out[0], out[1], rtol=1e-10, atol=0)


@pytest.mark.parametrize("rows,ncv,mixed", RESIDENT)
def test_batched_resident_sweep_edges(sa, rows, ncv, mixed):
    check_resident(sa, rows, ncv, mixed, "resident")


def test_batched_beyond_the_registers(sa):
    """A problem of one row more than 256 workgroups hold: "persistent" and the
    autotuner run lock-step and say so, and the resident sweep is not timed."""
    check_resident(sa, [256 * 64 * 22 + 1, 100], 12, False, "slots")
    from slepc_amd.batch import Batch
    B = Batch([_chain(sa, n, 7) for n in (256 * 64 * 22 + 1, 100)])
    B.solve(4, 12, 1e-10, "LM")
    info, sched = B.sweep_info(), B.schedule()
    assert info["mode"] == sched["kind"] == "wide" and info["ms_persistent"] == -1.0 and info["ms_wide"] > 0.0
    assert sched["ms"][0] == -1.0 and B.sweep_counts()["resident"] == 0


GIVE_UP = """
import sys, numpy as np
sys.path.insert(0, %r)
sys.path.insert(0, %r)
import slepc_amd as sa
import test_gpu_batched as t
sa.init(0)
t.check_resident(sa, [2000, 300, 5000], 24, False, "gave_up")
t.check_resident(sa, [2000, 300, 5000], 24, True, "gave_up")
"""


def test_batched_resident_sweep_gives_up():
    """With no polls allowed the resident sweep gives up half-way and the
    lock-step sweep starts over: the same results."""
    import os
    import subprocess
    import sys
    here = os.path.dirname(os.path.abspath(__file__))
    env = dict(os.environ, SLEPC_AMD_SWEEP_POLLS="0")
    subprocess.run([sys.executable, "-c", GIVE_UP % (os.path.dirname(here), here)], check=True, env=env, timeout=100)


@pytest.mark.parametrize("P", [1, 7, 8, 9, 33])
def test_batched_projected_problems_on_host_threads(sa, orc, P):
    """From 8 problems on the projected problems go to the solve's own host
    threads; problems that converge early leave fewer than 8 to the later
    rounds.  Every problem's values are the oracle's."""
    from slepc_amd.batch import Batch, uneven_laplacians
    csrs = uneven_laplacians(P=P, seed=5, lo=12, hi=40)
    v0 = [orc.rand_uniform(orc.sub_seed(3, p), A.n) for p, A in enumerate(csrs)]
    B = Batch(csrs)
    for _ in range(2):
        B.solve(4, 16, 1e-10, "LM", v0=v0)
        for p, A in enumerate(csrs):
            assert B.converged(p)[2] == 1
            w = np.linalg.eigvalsh(orc.CSR(A.n, A.rowptr, A.col, A.val).to_dense())
            for i in range(4):
                v = B.eigenpair(p, i, False)[0]
                assert np.min(np.abs(w - v)) < 1e-10 * abs(v)


def test_batched_c5_shapes(sa):
    """The 512-problem family: sizes span 1k..65k rows and all converge."""
    from slepc_amd.batch import Batch, uneven_laplacians
    csrs = uneven_laplacians(P=512, seed=2)
    ns = np.array([A.n for A in csrs])
    assert ns.min() >= 32 * 32 and ns.max() <= 256 * 256
    B = Batch(csrs[:64])
    B.solve(8, 24, 1e-10, "LM", mixed=True)
    err = B.errors()
    assert np.all(err <= 1e-10)


def test_batched_fv_family_ncv64_matches_single_solves(sa, orc):
    """The parameterised FV family at ncv 64 (lock-step sweep, the one-workgroup
    sweep holds at most 63 columns): every problem matches the single-problem
    solver and, on the smallest grid, the CPU oracle."""
    from slepc_amd.batch import Batch
    thetas = [sa.fv_theta(5, s) for s in range(4)]
    csrs = [sa.fv2d(g, g, th) for g, th in zip((24, 32, 40, 48), thetas)]
    v0 = [sa.rand_uniform(0, A.n) for A in csrs]
    B = Batch(csrs)
    B.solve(16, 64, 1e-10, "LR", v0=v0)
    assert B.sweep_info()["mode"] == "wide"
    err = B.errors()
    assert np.all(err <= 1e-10), err
    for p, A in enumerate(csrs):
        nconv, its, reason = B.converged(p)
        assert reason == 1 and nconv >= 16
        vals = np.sort([B.eigenpair(p, i, False)[0] for i in range(16)])
        E = sa.EPS()
        E.setOperators(sa.Mat(A))
        E.setProblemType(True)
        E.setWhichEigenpairs("LR")
        E.setDimensions(16, 64)
        E.setTolerances(1e-10)
        E.setInitialSpace(v0[p])
        E.solve()
        single = np.sort([E.getEigenpair(i, vectors=False)[0] for i in range(16)])
        assert np.allclose(vals, single, rtol=1e-10, atol=0)
        if p == 0:
            r = orc.eps_solve(orc.CSR(A.n, A.rowptr, A.col, A.val), 16, 64, 1e-10, "LR", True, v0=v0[p])
            assert np.allclose(vals, np.sort(r["eigr"][:16]), rtol=1e-10, atol=0)


@pytest.mark.parametrize("sweep", ["persistent", "wide"])
@pytest.mark.parametrize("mixed", [False, True])
def test_batched_true_residual_matches_oracle(sa, orc, mixed, sweep):
    """EPSSetTrueResidual for the whole batch (candidate Ritz vectors of all
    problems formed and evaluated on the device at once): every problem
    gives the oracle's values with its true-residual branch, the error
    estimates are explicit residuals (equal to EPSComputeError of the
    returned pair to rounding), and every pair meets the tolerance."""
    from slepc_amd.batch import Batch
    csrs = _problems(sa, orc)
    v0 = [orc.rand_uniform(orc.sub_seed(9, p), A.n) for p, A in enumerate(csrs)]
    B = Batch(csrs)
    B.set_sweep(sweep)
    B.set_true_residual(True)
    B.solve(8, 24, 1e-10, "LM", mixed=mixed, v0=v0)
    err = B.errors()
    for p, A in enumerate(csrs):
        nconv, its, reason = B.converged(p)
        assert reason == 1 and nconv >= 8
        Ao = orc.CSR(A.n, A.rowptr, A.col, A.val)
        r = orc.eps_solve(Ao, 8, 24, 1e-10, "LM", True, v0=v0[p], trueres=True)
        vals = np.array([B.eigenpair(p, i, False)[0] for i in range(8)])
        assert np.allclose(np.sort(vals), np.sort(r["eigr"][:8]), rtol=1e-10, atol=0)
        if not mixed:
            assert abs(its - r["its"]) <= max(2, 0.2 * r["its"])
        assert np.all(err[p] <= 1e-10), err[p]


@pytest.mark.parametrize("mixed", [False, True])
def test_batched_graph_replay_equals_direct_launches(sa, orc, mixed):
    """Lock-step restart sweeps replayed from captured HIP graphs give the
    same bits as the same sweeps launched one kernel at a time.  A second
    solve of the same batch replays the sweeps captured by the first (the
    signatures repeat), with the solver's own host work and device kernels
    between the replays; every replay feeds the next restart, so any wrong
    replay would change the trajectory."""
    from slepc_amd.batch import Batch
    csrs = _problems(sa, orc)
    v0 = [orc.rand_uniform(orc.sub_seed(9, p), A.n) for p, A in enumerate(csrs)]

    def run(B):
        B.solve(8, 24, 1e-10, "LM", mixed=mixed, v0=v0)
        vals = [[B.eigenpair(p, i, False)[0] for i in range(8)] for p in range(len(csrs))]
        its = [B.converged(p)[1] for p in range(len(csrs))]
        return np.array(vals), its, B.errors()

    B = Batch(csrs)
    B.set_sweep("wide")
    B.set_true_residual(True)
    v1, it1, e1 = run(B)
    g1 = B.graph_stats()
    assert g1["captures"] >= 1 and g1["cached"] >= 1
    v2, it2, e2 = run(B)
    g2 = B.graph_stats()
    assert g2["replays"] > g1["replays"]
    assert np.array_equal(v1, v2) and it1 == it2
    B.set_graphs(False)
    v3, it3, e3 = run(B)
    assert B.graph_stats() == g2                     # nothing captured or replayed
    assert np.array_equal(v1, v3) and it1 == it3
    assert np.all(e1 <= 1e-10) and np.array_equal(e1, e3)
    for p, A in enumerate(csrs[:3]):
        r = orc.eps_solve(orc.CSR(A.n, A.rowptr, A.col, A.val), 8, 24, 1e-10, "LM", True, v0=v0[p], trueres=True)
        assert np.allclose(np.sort(v1[p]), np.sort(r["eigr"][:8]), rtol=1e-10, atol=0)


def test_batched_schedule_autotuner(sa, orc):
    """The schedule autotuner times the one-workgroup sweep and three
    lock-step tile schedules on the first restart round and keeps the
    fastest; the solve then matches the oracle and a later solve reuses the
    choice without timing again."""
    from slepc_amd.batch import Batch
    csrs = _problems(sa, orc)
    v0 = [orc.rand_uniform(orc.sub_seed(9, p), A.n) for p, A in enumerate(csrs)]
    B = Batch(csrs)
    B.set_sweep("auto")
    B.solve(8, 24, 1e-10, "LM", v0=v0)
    sc = B.schedule()
    timed = [t for t in sc["ms"] if t > 0]
    assert len(timed) >= 3
    slot = 0 if sc["kind"] == "persistent" else None
    if slot is not None:
        assert sc["ms"][0] == min(timed)
    else:
        assert min(timed) in sc["ms"][1:] and sc["lanes"] in (4, 8, 16, 32) and sc["nt"] in (0, 1)
    err = B.errors()
    assert np.all(err <= 1e-10)
    for p, A in enumerate(csrs[:3]):
        r = orc.eps_solve(orc.CSR(A.n, A.rowptr, A.col, A.val), 8, 24, 1e-10, "LM", True, v0=v0[p])
        vals = np.sort([B.eigenpair(p, i, False)[0] for i in range(8)])
        assert np.allclose(vals, np.sort(r["eigr"][:8]), rtol=1e-10, atol=0)
    B.solve(8, 24, 1e-10, "LM", v0=v0)       # reuses the tuned schedule
    assert B.schedule()["kind"] == sc["kind"] and B.schedule()["lanes"] == sc["lanes"]


def test_batched_ncv_autotuner_and_per_problem_ncv(sa, orc):
    """The basis-size autotuner picks, per size class, the candidate ncv with
    the least time per converged pair on sampled problems; solve(ncv=0) then
    runs every problem with its class's ncv, and each problem agrees with the
    oracle run alone with that ncv."""
    from slepc_amd.batch import Batch
    csrs = _problems(sa, orc)
    cand = [16, 24, 32]
    B = Batch(csrs)
    B.set_true_residual(True)
    per = B.autotune_ncv(8, 1e-10, cand, which="LM", nclass=2, nsample=2, seed=3)
    tun = B.ncv_tuning()
    assert tun["scores"].shape == (2, 3) and np.all(np.isfinite(tun["scores"]))
    bests = {cand[int(np.argmin(tun["scores"][c]))] for c in range(2)}
    assert set(per.tolist()) == bests                # each problem takes its class's best
    ns = np.array([A.n for A in csrs])
    assert tun["class_hi"][0] <= tun["class_hi"][1] == ns.max()
    v0 = [orc.rand_uniform(orc.sub_seed(9, p), A.n) for p, A in enumerate(csrs)]
    B.solve(8, 0, 1e-10, "LM", v0=v0)
    assert np.array_equal(B.ncv(), per)
    err = B.errors()
    assert np.all(err <= 1e-10)
    for p, A in enumerate(csrs):
        r = orc.eps_solve(orc.CSR(A.n, A.rowptr, A.col, A.val), 8, int(per[p]), 1e-10, "LM", True, v0=v0[p],
                          trueres=True)
        vals = np.sort([B.eigenpair(p, i, False)[0] for i in range(8)])
        assert np.allclose(vals, np.sort(r["eigr"][:8]), rtol=1e-10, atol=0)
