"""The backward substitution's single launch over the narrow levels: supernodes of one and several
128-row chunks, a wide level below the narrow ones and a narrow one below that, repeated solves on one handle, and right-hand
sides that are not finite (results wait for one another by value, so every NaN has to arrive)."""
import numpy as np
import pytest

from symforce_amd import _capi as capi
from test_cholesky import dense_to_lower_csc

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


def spd(n, seed):
    m = np.random.default_rng(seed).standard_normal((n, n))
    return m @ m.T / n + np.eye(n)


def check(chol, a, seed):
    cond = np.linalg.cond(a)
    b = np.random.default_rng(seed).standard_normal(len(a))
    want = np.linalg.solve(a, b)
    # both solutions are backward stable with constants of order n: n eps cond(A), times 4
    assert np.abs(chol.solve(b) - want).max() <= 4 * len(a) * EPS * cond * np.abs(want).max()


@pytest.mark.parametrize("n", [64, 65, 192, 193, 256, 257, 321, 450])
def test_chunks(n):
    a = spd(n, n)
    _, cp, ri, v = dense_to_lower_csc(a)
    chol = capi.HipCholesky(n, cp, ri, ordering=capi.ORDERING_NATURAL)
    for k in range(3):
        chol.factorize(v * (k + 1.0))
        check(chol, a * (k + 1.0), k)
        check(chol, a * (k + 1.0), 10 + k)


@pytest.mark.parametrize("leaves,border", [(511, 3), (513, 1), (600, 150), (1100, 70)])
def test_wide_level_below(leaves, border):
    # columns coupled to the border only: as many leaf supernodes as columns
    n = leaves + border
    rng = np.random.default_rng(n)
    a = np.zeros((n, n))
    a[leaves:, :leaves] = rng.standard_normal((border, leaves)) / np.sqrt(n)
    a = a + a.T
    a[leaves:, leaves:] = spd(border, border)
    a += 4 * np.eye(n)
    _, cp, ri, v = dense_to_lower_csc(a)
    keep = v != 0
    cols = np.repeat(np.arange(n), np.diff(cp))[keep]
    cp = np.searchsorted(cols, np.arange(n + 1)).astype(np.int32)
    chol = capi.HipCholesky(n, cp, ri[keep], ordering=capi.ORDERING_NATURAL)
    chol.factorize(v[keep])
    check(chol, a, 1)
    check(chol, a, 2)


@pytest.mark.parametrize("leaves,middle,border", [(2, 200, 260), (1, 180, 300), (2, 255, 257)])
def test_narrow_level_below_a_wide_one(leaves, middle, border):
    # `leaves` columns coupled to each middle column (one block each, 180 to 510 in all), the middle
    # columns coupled to the border (three chunks each: more than 512 blocks), a dense border
    n0, n1 = leaves * middle, (leaves + 1) * middle
    n = n1 + border
    rng = np.random.default_rng(n)
    a = np.zeros((n, n))
    a[n0 + np.arange(n0) // leaves, np.arange(n0)] = rng.uniform(-1, 1, n0)
    a[n1:, n0:n1] = rng.standard_normal((border, middle)) / np.sqrt(n)
    a = a + a.T
    a[n1:, n1:] = spd(border, border)
    a += 4 * np.eye(n)
    _, cp, ri, v = dense_to_lower_csc(a)
    keep = v != 0
    cols = np.repeat(np.arange(n), np.diff(cp))[keep]
    cp = np.searchsorted(cols, np.arange(n + 1)).astype(np.int32)
    chol = capi.HipCholesky(n, cp, ri[keep], ordering=capi.ORDERING_NATURAL)
    assert chol.info()["levels"] == 2 + -(-border // 64)
    chol.factorize(v[keep])
    check(chol, a, 1)
    check(chol, a, 2)


@pytest.mark.parametrize("n", [5, 64, 200, 321])
def test_not_finite(n):
    a = spd(n, n)
    _, cp, ri, v = dense_to_lower_csc(a)
    chol = capi.HipCholesky(n, cp, ri, ordering=capi.ORDERING_NATURAL)
    chol.factorize(v)
    for bits in (0xFFFFFFFFFFFFFFFF, 0x7FF8000000000000, 0x7FF0000000000001):
        b = np.ones(n)
        b[-1] = np.array([bits], dtype=np.uint64).view(np.float64)[0]
        assert np.isnan(chol.solve(b)).all()  # a dense factor carries it everywhere
    check(chol, a, 3)
