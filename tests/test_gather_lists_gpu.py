"""Linearization entries whose contribution lists are short, long and very long (a thread, 16 lanes
and a block each), at the lengths where the kernel's dealing changes, against the FP64 oracle with
the tolerances of test_linearize_gpu.py."""
import numpy as np
import pytest

from symforce_amd import _capi as capi
import oracle_wrap as ow
import problem_builders as pb

from test_linearize_gpu import assert_linearization_close

pytestmark = pytest.mark.gpu


def check(prob):
    got, op = capi.HipProblem(prob).linearize(), ow.OracleProblem(prob)
    assert_linearization_close(got, op.linearize(), *op.hessian_structure())


@pytest.mark.parametrize("n", [1, 4, 8, 9, 16, 17, 63, 64, 65, 511, 512, 513, 1024, 3001])
def test_one_key_with_n_factors(n):
    # every entry of the 5 x 5 Hessian and of the rhs sums n contributions
    prob, _ = pb.gnc_problem(np.random.default_rng(n).standard_normal((n, 5)))
    check(prob)


@pytest.mark.parametrize("cams,points", [(3, 7), (9, 40), (8, 600), (17, 520)])
def test_cameras_and_points_mix_list_lengths(cams, points):
    # a camera's entries sum `points` contributions, a point's `cams`, a pair's one
    check(capi.gen_ba_circle(cams, points, 5))
