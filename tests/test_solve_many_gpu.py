"""Several right-hand sides through the device LDL^T at once: the same answers as one at a time and
as the dense solve, over group remainders, and when the workspace takes them in several passes."""
import numpy as np
import pytest

from symforce_amd import _capi as capi
import oracle_wrap as ow
from test_cholesky import MATRICES

pytestmark = pytest.mark.gpu
# Both sides are backward stable: they differ by a small multiple (16 here) of eps * cond(A), with
# cond(A) <= 3e6 for the damped Hessians below (checked).
MAX_COND = 3e6
RTOL = 16 * np.finfo(np.float64).eps * MAX_COND


def graph_case():
    op = ow.OracleProblem(capi.gen_pose_graph(250, 75, 4))
    cp, ri = op.hessian_structure()
    h = op.linearize()["hessian_values"].copy()
    h[cp[:-1]] += 1.0
    return op.N, cp, ri, h


CASES = {"graph_250": graph_case, "ba_circle": MATRICES["ba_circle_H"],
         "robot3d": MATRICES["robot3d_H"]}


def dense(n, cp, ri, v):
    a = np.zeros((n, n))
    cols = np.repeat(np.arange(n), np.diff(cp))
    a[ri, cols] = v
    a[cols, ri] = v
    return a


@pytest.mark.parametrize("nrhs", [1, 2, 3, 4, 5, 8, 13, 67])
@pytest.mark.parametrize("name", sorted(CASES))
def test_matches_single_and_dense(name, nrhs):
    n, cp, ri, v = CASES[name]()
    a = dense(n, cp, ri, v)
    assert np.linalg.cond(a) <= MAX_COND
    chol = capi.HipCholesky(n, cp, ri)
    chol.factorize(v)
    b = np.random.default_rng(nrhs).standard_normal((n, nrhs))
    x = chol.solve(b)
    scale = np.abs(x).max(axis=0)
    assert np.all(np.abs(x - np.linalg.solve(a, b)) <= RTOL * scale)
    for k in range(min(nrhs, 9)):
        assert np.all(np.abs(x[:, k] - chol.solve(b[:, k])) <= RTOL * scale[k])
    again = chol.solve(b[:, ::-1])  # the workspace and counters of a second call
    assert np.all(np.abs(again[:, ::-1] - x) <= RTOL * scale)


def test_more_than_one_pass():
    prob = capi.gen_pose_graph(5000, 1500, 3)
    hp = capi.HipProblem(prob)
    cp, ri = hp.hessian_structure()
    v = hp.linearize()["hessian_values"]
    v[cp[:-1]] += 1.0
    chol = capi.HipCholesky(hp.N, cp, ri, np.arange(0, hp.N + 1, 6, dtype=np.int32),
                            ordering=capi.ORDERING_NESTED_DISSECTION)
    chol.factorize(v)
    nrhs = (256 << 20) // (40 * hp.N) + 6  # the workspace limit, and a remainder of six
    b = np.random.default_rng(0).standard_normal((hp.N, nrhs))
    x = chol.solve(b)
    for k in (0, 1, nrhs - 7, nrhs - 6, nrhs - 1):
        one = chol.solve(b[:, k])
        # cond(A) is not known here: the residual is held instead, |b - A x| <= 1e-12 |A| |x|
        r = np.zeros(hp.N)
        cols = np.repeat(np.arange(hp.N), np.diff(cp))
        np.add.at(r, ri, v * x[cols, k])
        off = ri != cols
        np.add.at(r, cols[off], v[off] * x[ri[off], k])
        assert np.abs(r - b[:, k]).max() <= 1e-12 * np.abs(v).max() * np.abs(x[:, k]).max()
        assert np.abs(one - x[:, k]).max() <= 1e-6 * np.abs(one).max()
