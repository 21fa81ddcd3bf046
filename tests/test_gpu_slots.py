"""The decisions of the Gram-Schmidt step that ordinary data rarely takes: a
failed norm estimate, a third pass, a scaling alone, linear dependence, and
refinement never and always.  Each on a basis beyond the registers (the slots,
csrc/sa_gw.hip) and on a small one (the resident kernel), against the rule in
numpy."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ETA = 0.7071


def dgks(V, v, refine):
    """BVOrthogonalizeGS (src/sys/classes/bv/interface/bvorthog.c:145-217) and the
    scaling of BVOrthonormalizeColumn (:417-422): coefficients, norm, lindep,
    passes and the new column.  V need not be orthonormal."""
    h, passes, v = np.zeros(V.shape[1]), 0, v.copy()

    def cgs(estimate=True):
        nonlocal v, h, passes
        c = V.T @ v
        onrm, est = np.linalg.norm(v), v @ v - c @ c
        h += c
        v = v - V @ c
        passes += 1
        return onrm, np.sqrt(est) if estimate and est > 0.0 else np.linalg.norm(v)

    if refine == "never":
        onrm, nrm = cgs(False)
        lindep = nrm == 0.0
    elif refine == "always":
        cgs()
        onrm, nrm = cgs()
        lindep = nrm < ETA * onrm
    else:
        onrm, nrm = cgs()
        while nrm < ETA * onrm and passes < 3:
            onrm, nrm = cgs()
        lindep = nrm < ETA * onrm
    return h, nrm, lindep, passes, v / nrm


# cosine between the first two columns, and the new column as a u + b w with u
# their normalised sum and w orthogonal to all.  A pass scales the part along u
# by -cosine and the norm estimate takes (1 + cosine) of its square away, so the
# decisions are far from rounding:
CASES = {
    "one pass, estimate": (0.0, 0.1, 1.0),          # hardly anything along u
    "two passes": (0.0, 1.0, 0.1),                  # orthonormal columns, v mostly along them
    "failed estimate, scaling alone": (0.75, 1.0, 0.0),
    "failed estimate, then a pass": (0.4, 1.0, 0.6),
    "three passes": (0.5, 1.0, 0.5),
    "three failed estimates, dependent": (0.7, 1.0, 0.0),
}


@pytest.mark.parametrize("refine", ["ifneeded", "never", "always"])
@pytest.mark.parametrize("j,prec", [(2, "fp64"), (20, "fp64"), (60, "fp64"), (110, "fp64"), (3, "fp32"), (70, "fp32"),
                                    (110, "fp32")])
@pytest.mark.parametrize("large", [False, True])
def test_rare_decisions(sa, large, j, prec, refine):
    P, eps = (sa.FP64, 2.2e-16) if prec == "fp64" else (sa.FP32, 6e-8)
    # one row more than the registers of 256 workgroups hold, or 33 chunks and a row
    n = (262144 if prec == "fp64" else 360448) + 1 if large else 2113
    count = sa.lib().sa_bv_get_pass_count
    count.argtypes = [C.c_void_p, C.POINTER(C.c_int64)]
    rng = np.random.default_rng(j)
    # orthonormal columns (disjoint supports); the reference works on coordinates in them
    Q = np.zeros((n, j + 1))
    owner = rng.integers(0, j + 1, n)
    Q[np.arange(n), owner] = rng.choice([-1.0, 1.0], n)
    Q /= np.linalg.norm(Q, axis=0)
    B = sa.BV(n, j + 1, P)
    B.set_orthogonalization(refine)
    for i in range(2, j):
        B.set_column(i, Q[:, i])
    done = 0
    for name, (cosine, a, b) in CASES.items():
        X = np.eye(j + 1)[:, :j]
        X[:2, 1] = cosine, np.sqrt(1.0 - cosine ** 2)
        u = X[:, 0] + X[:, 1]
        v = a * u / np.linalg.norm(u)
        v[j] = b
        for i, y in ((0, X[:, 0]), (1, X[:, 1]), (j, v)):
            B.set_column(i, Q @ y)
        h, nrm, lindep, passes, x = dgks(X, v, refine)
        got_nrm, got_lindep = B.orthonormalize_column(j)
        p = C.c_int64()
        sa.check(count(B.h, C.byref(p)))
        assert (got_lindep, p.value - done) == (lindep, passes), name
        done = p.value
        # three passes of j updates, and dot products of some 30 additions one after
        # another, all of size 1, in the basis's precision
        tol = 30 * (j + 10) * eps
        H = B.coefficients(j, j + 1)[:, 0]
        assert np.abs(H[:j] - h).max() <= tol, name
        assert abs(got_nrm - nrm) <= tol and abs(H[j] - (0.0 if lindep else nrm)) <= tol, name
        assert np.linalg.norm(B.get_column(j) - Q @ x) <= tol / nrm, name
    assert B.sweep_counts() == dict(resident=0 if large else len(CASES), gave_up=0, slots=len(CASES) if large else 0)
