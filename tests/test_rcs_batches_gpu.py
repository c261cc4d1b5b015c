"""The reduced camera system's pair sums at the pair counts where their batches of eight and work
items of 512 end: few cameras with few to many common points, the Schur path's run held to the
full-system LDL^T's (an independent assembly and factorization of the same Hessian)."""
import numpy as np
import pytest

from symforce_amd import _capi as capi
from test_optimizer_gpu import assert_same_trajectory

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cams", [2, 4])
@pytest.mark.parametrize("points", [7, 8, 9, 15, 16, 17, 31, 33, 511, 513, 1030])
def test_pair_counts(cams, points):
    prob = capi.gen_ba_snavely(cams, points, seed=points)
    params = capi.default_params(iterations=3, initial_lambda=1.0)
    a, b = (capi.HipOptimizer(prob, params, capi.solver_options(linear_solver=k)).optimize()
            for k in (capi.SOLVER_SCHUR, capi.SOLVER_CHOLESKY))
    assert_same_trajectory(a, b, rtol=1e-8)  # the Schur tests' bound for these systems
    np.testing.assert_allclose(a["values"], b["values"], rtol=0,
                               atol=1e-7 * max(1.0, np.abs(b["values"]).max()))
