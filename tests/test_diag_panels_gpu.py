"""The diagonal blocks of the device LDL^T at the widths and below-row counts where their 16-column
panels and 64-row chunks end: dense matrices (chains of supernodes 64 columns wide and a remainder)
and arrow matrices (one block coupled to a border), solved and factored against numpy; and the form
with the right-hand side eliminated along, through optimizer runs on pose chains held to the oracle."""
import numpy as np
import pytest

from symforce_amd import _capi as capi
import oracle_wrap as ow
from test_cholesky import dense_to_lower_csc
from test_optimizer_gpu import assert_same_trajectory

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


def ldl(a):
    """Unit lower L and d of a = L diag(d) L^T by Cholesky (a is SPD and well conditioned)."""
    c = np.linalg.cholesky(a)
    d = np.diag(c)
    return c / d, d * d


def check(a):
    n, cp, ri, v = dense_to_lower_csc(a)
    cond = np.linalg.cond(a)
    assert cond < 1e3
    chol = capi.HipCholesky(n, cp, ri, ordering=capi.ORDERING_NATURAL)
    chol.factorize(v)
    b = np.random.default_rng(n).standard_normal(n)
    x = chol.solve(b)
    # both solutions are backward stable with constants of order n: n eps cond(A), times 4
    tol = 4 * n * EPS * cond
    want = np.linalg.solve(a, b)
    assert np.abs(x - want).max() <= tol * np.abs(want).max()
    low, d = ldl(a)
    assert np.all(np.abs(chol.d() - d) <= tol * np.abs(d).max())
    lp, li, lv = chol.factor_l()
    got = np.zeros((n, n))
    got[li, np.repeat(np.arange(n), np.diff(lp))] = lv
    assert np.abs(got + np.eye(n) - low).max() <= tol


def spd(n, seed):
    m = np.random.default_rng(seed).standard_normal((n, n))
    return m @ m.T / n + np.eye(n)


@pytest.mark.parametrize("n", [1, 2, 3, 4, 7, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 80,
                               96, 127, 128, 129, 191, 200])
def test_dense(n):
    check(spd(n, n))


@pytest.mark.parametrize("cols,border", [(5, 1), (16, 3), (17, 40), (33, 63), (48, 64), (64, 65),
                                         (63, 127), (20, 129)])
def test_arrow(cols, border):
    # three blocks of `cols` columns, each coupled to the same `border` rows only
    n = 3 * cols + border
    a = spd(n, n)
    for i in range(3):
        for j in range(3):
            if i != j:
                a[i * cols:(i + 1) * cols, j * cols:(j + 1) * cols] = 0
    a += 3 * np.eye(n)
    check(a)


@pytest.mark.parametrize("poses", [1, 2, 3, 5, 8, 10, 11, 16, 21, 22, 40])
def test_right_hand_side_along(poses):
    prob = capi.gen_pose_smoothing(poses, 42)
    params = capi.default_params(iterations=6)
    for ordering in (capi.ORDERING_NATURAL, capi.ORDERING_MIN_DEGREE):
        got = capi.HipOptimizer(prob, params, capi.solver_options(ordering=ordering)).optimize()
        assert_same_trajectory(got, ow.OracleProblem(prob).optimize(params), rtol=1e-8)
