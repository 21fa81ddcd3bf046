"""The resident Arnoldi sweep (csrc/sa_sweep.hip): the Arnoldi relation and
orthogonality at the edges of its row blocks, column slots and operator
staging, and the same results when its waits give up and the sweep runs slot
by slot instead."""
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EPS = {"fp64": 2.2e-16, "fp32": 6e-8}


def _csr(sa, kind, n, seed=3):
    """band: neighbours and a far diagonal; ragged: empty rows and rows whose
    columns are spread over the whole matrix (more remote entries than the
    resident kernel lists, so that it reads the operator from memory)."""
    rng = np.random.default_rng(seed)
    if kind == "band":
        offs = [0, 1, -1, 37, -211]
        r, c = zip(*[(np.arange(n), np.arange(n) + o) for o in offs])
        r, c = np.concatenate(r), np.concatenate(c)
    else:
        k = rng.integers(0, 40, n)
        r = np.repeat(np.arange(n), k)
        c = rng.integers(0, n, len(r))
    keep = (c >= 0) & (c < n)
    r, c = r[keep], c[keep]
    key = np.unique(r.astype(np.int64) * n + c)
    r, c = key // n, key % n
    rp = np.zeros(n + 1, np.int32)
    rp[1:] = np.cumsum(np.bincount(r, minlength=n))
    return sa.CSR(n, rp, c.astype(np.int32), rng.uniform(-1.0, 1.0, len(c)))


def _matvec(A, X):
    p = np.concatenate([np.zeros((1, X.shape[1])), np.cumsum(A.val[:, None] * X[A.col], axis=0)])
    return p[A.rowptr[1:]] - p[A.rowptr[:-1]]


def check_relation(sa, n, m, kind, prec, ran="resident"):
    """ran: how the orthonormalisation of the start vector and the two sweeps are
    to have run, as BV.sweep_counts names it (or its whole answer)."""
    P = sa.FP64 if prec == "fp64" else sa.FP32
    A = _csr(sa, kind, n)
    if prec == "fp32":
        A.val = A.val.astype(np.float32).astype(np.float64)
    M, V = sa.Mat(A, P), sa.BV(n, m + 1, P)
    V.set_column(0, sa.rand_uniform(5, n))
    V.orthonormalize_column(0)
    for k in (0, m // 2):                     # a first sweep, and one from column m // 2
        mm, beta, bd = V.mat_arnoldi(M, k, m)
        assert mm == m and not bd
        X, H = V.get_matrix(m + 1), V.coefficients(1, m + 1)
        assert beta == pytest.approx(H[m, m - 1], rel=1e-15)
        H = np.vstack([H, np.zeros((m + 1 - H.shape[0], m))]) if H.shape[0] < m + 1 else H[:m + 1]
        # each column: at most ~40 products per row, m updates, all of size <= 40 * ||x||_2
        eps = EPS[prec]
        rel = _matvec(A, X[:, :m]) - X @ np.triu(H, -1)
        assert np.linalg.norm(rel, axis=0).max() <= 40 * (m + 40) * eps
        assert np.abs(X.T @ X - np.eye(m + 1)).max() <= 100 * (m + 1) * eps
    assert V.sweep_counts() == (ran if isinstance(ran, dict) else dict(dict(resident=0, gave_up=0, slots=0), **{ran: 3}))


# rows: one and two chunks, the last row block with one row, exactly 64 blocks
# and one row more (1 -> 2 -> 4 chunks per block), 256 blocks of 4 chunks and
# one row more (6 chunks); columns: the last of a slot, one more, a full basis
@pytest.mark.parametrize("n,m,kind,prec", [
    (64, 7, "band", "fp64"), (65, 33, "band", "fp64"), (257, 32, "ragged", "fp64"), (4096, 64, "band", "fp64"),
    (4097, 65, "ragged", "fp64"), (8193, 97, "band", "fp64"), (16385, 20, "ragged", "fp32"),
    (65536, 64, "band", "fp64"), (65537, 12, "band", "fp64"), (98305, 40, "band", "fp32"),
    (4097, 126, "band", "fp32"), (180224, 10, "band", "fp64")])
def test_sweep_relation(sa, n, m, kind, prec):
    check_relation(sa, n, m, kind, prec)


@pytest.mark.parametrize("n,m,kind,prec", [
    (180225, 12, "band", "fp64"), (200001, 32, "band", "fp64"), (131073, 33, "ragged", "fp64"),
    (65537, 40, "band", "fp64"), (260000, 30, "band", "fp32")])
def test_sweep_relation_half_the_workgroups(sa, n, m, kind, prec):
    """With other solves announced the sweep takes half the CUs where they hold
    the basis, and all of them where they do not."""
    before = sa.set_concurrent_solves(2)
    try:
        check_relation(sa, n, m, kind, prec)
    finally:
        sa.set_concurrent_solves(max(1, before))


CODE = """
import sys, numpy as np
sys.path.insert(0, %r)
import slepc_amd as sa
sa.init(0)
A = sa.lap2d(70, 61)
V = sa.BV(A.n, 34)
V.set_column(0, sa.rand_uniform(5, A.n))
V.orthonormalize_column(0)
M = sa.Mat(A)
V.mat_arnoldi(M, 0, 32)
W = sa.BV(A.n, 34)
W.set_matrix(V.get_matrix(33))
W.set_column(33, sa.rand_uniform(6, A.n))
nrm, lindep = W.orthonormalize_column(33)
count = lambda B: [B.sweep_counts()[k] for k in ("resident", "gave_up", "slots")]
first = [count(V), count(W)]
for _ in range(17):
    V.mat_arnoldi(M, 0, 32)
np.savez(sys.argv[1], V=W.get_matrix(34), H=V.coefficients(0, 33), h=W.coefficients(33, 34), nrm=nrm,
         first=first, later=count(V))
"""


SLOTS = """
import sys
sys.path.insert(0, %r)
sys.path.insert(0, %r)
import slepc_amd as sa
import test_gpu_sweep as t
sa.init(0)
# one chunk of 128 rows and its neighbours, more chunks than workgroups; basis
# widths on both sides of every kernel's column limit
for n, m, prec in ((127, 17, "fp64"), (128, 33, "fp32"), (129, 49, "fp64"), (3001, 66, "fp64"),
                   (3001, 98, "fp64"), (2999, 126, "fp32"), (65663, 30, "fp64"), (65663, 30, "fp32")):
    # twice the kernel gives up, the third call does not try it
    t.check_relation(sa, n, min(m, n - 1), "band", prec, dict(resident=0, gave_up=2, slots=1))
    print(n, m, prec, flush=True)
"""


def test_slots_relation():
    """The same relation slot by slot (csrc/sa_gw.hip)."""
    env = dict(os.environ, SLEPC_AMD_SWEEP_POLLS="0")
    subprocess.run([sys.executable, "-c", SLOTS % (ROOT, os.path.join(ROOT, "tests"))], check=True, env=env,
                   timeout=100)


def test_slots_relation_large(sa):
    """Beyond the registers' capacity, no override needed."""
    check_relation(sa, 200001, 64, "band", "fp64", dict(resident=1, gave_up=0, slots=2))
    check_relation(sa, 270001, 20, "band", "fp64", "slots")


def test_one_row(sa):
    """A single row: one workgroup, which waits for nobody."""
    V = sa.BV(1, 2)
    V.set_column(0, [-3.0])
    nrm, lindep = V.orthonormalize_column(0)
    assert nrm == 3.0 and not lindep and V.get_column(0)[0] == -1.0
    assert V.sweep_counts() == dict(resident=1, gave_up=0, slots=0)


PASSES = """
import ctypes as C, sys
sys.path.insert(0, %r)
import slepc_amd as sa
sa.init(0)
count = sa.lib().sa_bv_get_pass_count
count.argtypes = [C.c_void_p, C.POINTER(C.c_int64)]
A = sa.lap2d(70, 61)
M, p = sa.Mat(A), C.c_int64()
tally = dict(resident=0, gave_up=0, slots=0)
for i in range(150):
    V = sa.BV(A.n, 4)
    V.set_column(0, sa.rand_uniform(5, A.n))
    V.scale_column(0, 1.0 / V.norm_column(0))
    for r in range(1, 5):
        V.mat_arnoldi(M, 0, 3)
        sa.check(count(V.h, C.byref(p)))
        assert p.value == 6 * r, (i, r, p.value, V.sweep_counts())
    for k, v in V.sweep_counts().items():
        tally[k] += v
print(tally)
"""


@pytest.mark.parametrize("polls", ["0", "12", "16"])
def test_passes_of_a_sweep_that_gave_up_count_once(polls):
    """Three columns of two passes each, whether the resident kernel finished,
    gave up (also when its lead workgroup alone finished) or was not tried."""
    env = dict(os.environ, SLEPC_AMD_SWEEP_POLLS=polls)
    subprocess.run([sys.executable, "-c", PASSES % ROOT], check=True, env=env, timeout=100)


def test_sweep_gives_up_and_starts_over(tmp_path):
    """With no polls allowed, every wait that is not met at once gives up: the
    kernel ends, and the host's slot-by-slot sweep returns the same basis (the
    orthonormalised column included, whose input the kernel may have
    overwritten), to the rounding of two summation orders.  Of 19 calls in a row
    five try the kernel (the 1st, 2nd, 4th, 8th and 16th)."""
    out = []
    for polls in (None, "0"):
        env = dict(os.environ)
        env.pop("SLEPC_AMD_SWEEP_POLLS", None)
        if polls is not None:
            env["SLEPC_AMD_SWEEP_POLLS"] = polls
        f = str(tmp_path / ("r%s.npz" % polls))
        subprocess.run([sys.executable, "-c", CODE % ROOT, f], check=True, env=env, timeout=100)
        out.append(np.load(f))
    a, b = out
    assert a["first"].tolist() == [[2, 0, 0], [1, 0, 0]] and a["later"].tolist() == [19, 0, 0]
    assert b["first"].tolist() == [[0, 2, 0], [0, 1, 0]] and b["later"].tolist() == [0, 5, 14]
    assert np.abs(a["V"] - b["V"]).max() <= 1e-12
    assert np.abs(a["H"] - b["H"]).max() <= 1e-13 and np.abs(a["h"] - b["h"]).max() <= 1e-13
    assert float(a["nrm"]) == pytest.approx(float(b["nrm"]), rel=1e-14)


# up to 32 columns of the resident sweep, one row and 22 rows per lane, and up to
# 16 of the streaming slots
@pytest.mark.parametrize("n,j", [(65, 7), (354000, 1), (354000, 10), (354000, 31), (400001, 2), (400001, 16)])
def test_fp32_products_are_added_in_fp64(sa, n, j):
    """Orthonormalising an FP32 column: coefficients and norm equal those of the
    stored values in FP64.  A product of two FP32 numbers is exact in FP64 and
    a sum of FP64 is at most 40 additions deep on either side, so the two differ
    by at most 80 eps of ||x|| ||v||; FP32 sums of a few rows are 1e-10 off at
    these sizes."""
    rng = np.random.default_rng(n + j)
    V = sa.BV(n, j + 1, sa.FP32)
    B = np.linalg.qr(rng.standard_normal((n, j)))[0]
    for i in range(j):
        V.set_column(i, B[:, i])
    V.set_column(j, rng.standard_normal(n))
    X, v = V.get_matrix(j), V.get_column(j)      # as stored
    nrm, lindep = V.orthonormalize_column(j)
    H = V.coefficients(j, j + 1)[:, 0]
    ref, h = np.linalg.norm(v), X.T @ v
    assert not lindep
    assert np.abs(H[:j] - h).max() <= 80 * EPS["fp64"] * ref
    assert nrm == pytest.approx(np.sqrt(ref * ref - h @ h), rel=200 * EPS["fp64"])


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("n,stream", [(3001, False), (400001, False), (400001, True)])
def test_columns_beyond_a_breakdown_stay(sa, n, stream, prec):
    """A^2 = 0 on the start vector: the sweep breaks down at column 2 of 7 and
    leaves the columns after it alone, in the resident kernel and slot by slot
    with both SpMV layouts."""
    P = sa.FP64 if prec == "fp64" else sa.FP32
    # rows 2i take row 2i + 1: with a start vector on the odd rows, A v is on the even ones and A A v = 0
    r = np.arange(0, n - 1, 2)
    rp = np.zeros(n + 1, np.int32)
    rp[1:] = np.cumsum(np.isin(np.arange(n), r))
    prev = sa.set_spmv_stream_bytes(0) if stream else None
    M = sa.Mat(sa.CSR(n, rp, (r + 1).astype(np.int32), np.ones(len(r))), P)
    if stream:
        sa.set_spmv_stream_bytes(prev)
    V = sa.BV(n, 8, P)
    x = np.zeros(n)
    x[1::2] = 1.0
    V.set_column(0, x)
    V.orthonormalize_column(0)
    for j in range(3, 8):
        V.set_column(j, np.full(n, 7.0 + j))
    m, beta, breakdown = V.mat_arnoldi(M, 0, 7)
    assert (m, beta, breakdown) == (2, 0.0, True)
    for j in range(3, 8):
        assert np.all(V.get_column(j) == 7.0 + j)


def test_concurrent_sweeps_share_the_cus(sa):
    """Five threads whose sweeps need more than the CUs together (128 workgroups
    of 65,536 rows with other solves announced, 256 of 180,000): they wait for
    one another in turn, and each gets the bits that it gets alone."""
    import concurrent.futures as cf

    def work(n, m, seed):
        M, V = sa.Mat(_csr(sa, "band", n, seed)), sa.BV(n, m + 1)
        out = []
        for k in range(6):
            V.set_column(0, sa.rand_uniform(seed + k, n))
            V.orthonormalize_column(0)
            V.mat_arnoldi(M, 0, m)
            out.append((V.get_column(m), V.coefficients(1, m + 1)))
        return out

    jobs = [(65536, 40, 1), (180000, 36, 2), (65536, 40, 3), (180000, 36, 4), (65536, 40, 5)]
    before = sa.set_concurrent_solves(len(jobs))
    try:
        alone = [work(*j) for j in jobs]
        with cf.ThreadPoolExecutor(len(jobs)) as ex:
            together = list(ex.map(lambda j: work(*j), jobs))
    finally:
        sa.set_concurrent_solves(max(1, before))
    for a, b in zip(alone, together):
        for (x, h), (y, g) in zip(a, b):
            assert np.array_equal(x, y) and np.array_equal(h, g)
