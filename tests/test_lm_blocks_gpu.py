"""The LM run's three Values blocks and its fused reductions: the optimized keys are retracted from
one block into another while the constants reach a block with its first use in a run, so a second
run of one optimizer with other constants, runs with rejected steps (which change the blocks' order)
and with bold updates (an accepted step that is not the best is what brings the third block in), and
residual / state counts around the 256-thread blocks of the reductions are held to the oracle.
Also the damped assembly at the odd panel sizes of its paired stores, and its two ways."""
import numpy as np
import pytest

from symforce_amd import _capi as capi
import oracle_wrap as ow
from test_optimizer_gpu import assert_same_trajectory

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


def with_values(p, values):
    return capi.Problem(p.letters, p.subs, p.supers, p.types, values, p.ftypes, p.fptr, p.fargs,
                        p.opt_keys, p.info)


def moved_constants(p, seed):
    """The 3-vectors of a localization problem (landmarks and measurements: constants), moved."""
    rng = np.random.default_rng(seed)
    v = p.values.copy()
    for o, t in zip(p.storage_offsets, p.types):
        if t == capi.TYPE_VECTOR3:
            v[o:o + 3] += 0.05 * rng.standard_normal(3)
    assert not np.array_equal(v, p.values)
    return v


@pytest.mark.parametrize("poses,lm,initial_lambda", [(5, 9, 1.0), (42, 9, 1e-6), (43, 20, 1e4),
                                                     (60, 40, 1e-6)])
def test_second_run_uses_its_own_constants(poses, lm, initial_lambda):
    prob = capi.gen_localization(poses, lm, 0.5, seed=poses)
    params = capi.default_params(iterations=12, initial_lambda=initial_lambda)
    opt = capi.HipOptimizer(prob, params)
    for values in (prob.values, moved_constants(prob, poses), prob.values):
        got = opt.optimize(values=values)
        ora = ow.OracleProblem(with_values(prob, values)).optimize(params)
        assert_same_trajectory(got, ora, rtol=1e-8)
        np.testing.assert_allclose(got["values"], ora["values"], rtol=0,
                                   atol=1e-8 * max(1.0, np.abs(ora["values"]).max()))


def moved_pixels(p, seed):
    """The pixel measurements of a bundle adjustment (constants), moved by a pixel or so."""
    rng = np.random.default_rng(seed)
    v = p.values.copy()
    for o, t in zip(p.storage_offsets, p.types):
        if t == capi.TYPE_VECTOR2:
            v[o:o + 2] += rng.standard_normal(2)
    assert not np.array_equal(v, p.values)
    return v


def steps(run):
    """A letter per step: r(ejected), a(ccepted), B(old: accepted without reducing the error)."""
    return "".join("r" if not it["update_accepted"] else "a" if it["relative_reduction"] > 0 else "B"
                   for it in run["iterations"] if it["iteration"] >= 0)


@pytest.mark.parametrize("solver", [capi.SOLVER_CHOLESKY, capi.SOLVER_SCHUR])
@pytest.mark.parametrize("cams,lam", [(4, capi.LAMBDA_STATIC), (4, capi.LAMBDA_DYNAMIC),
                                      (8, capi.LAMBDA_STATIC)])
def test_second_run_with_rejected_steps(cams, lam, solver):
    prob = capi.gen_ba_circle(cams, 8 * cams, seed=cams)
    params = capi.default_params(iterations=12, lambda_update_type=lam)
    opt = capi.HipOptimizer(prob, params, capi.solver_options(linear_solver=solver))
    for values in (prob.values, moved_pixels(prob, cams), prob.values):
        ora = ow.OracleProblem(with_values(prob, values)).optimize(params)
        assert "ra" in steps(ora), steps(ora)
        assert_same_trajectory(opt.optimize(values=values), ora, rtol=1e-8)


@pytest.mark.parametrize("solver", [capi.SOLVER_CHOLESKY, capi.SOLVER_SCHUR])
def test_second_run_with_bold_updates(solver):
    prob = capi.gen_ba_snavely(8, 160, 5)
    params = capi.default_params(iterations=11, enable_bold_updates=1)
    opt = capi.HipOptimizer(prob, params, capi.solver_options(linear_solver=solver))
    for values in (prob.values, moved_pixels(prob, 8), prob.values):
        ora = ow.OracleProblem(with_values(prob, values)).optimize(params)
        assert "B" in steps(ora), steps(ora)
        # A bold step is taken where the system is unstable: moving the oracle's start by 1e-13
        # moves its records by up to 1e-9. (The other run's pixels move the first one by 3e-4.)
        assert_same_trajectory(opt.optimize(values=values), ora, rtol=1e-7)


@pytest.mark.parametrize("n", [1, 2, 3, 5, 16, 17, 23, 65])
def test_assembly_of_odd_panels(n):
    """A band matrix, factored twice with different values on one handle: every panel entry is
    written again, zeros where the matrix has none."""
    rng = np.random.default_rng(n)
    chol = None
    for k in range(2):
        a = np.eye(n) * (4 + k) + np.diag(rng.uniform(-1, 1, n - 1), -1) if n > 1 else \
            np.eye(1) * (4.0 + k)
        full = np.tril(a) + np.tril(a, -1).T
        mask = np.abs(np.subtract.outer(np.arange(n), np.arange(n))) <= 1
        cols = [np.flatnonzero(mask[j:, j]) + j for j in range(n)]
        cp = np.concatenate([[0], np.cumsum([len(c) for c in cols])]).astype(np.int32)
        ri = np.concatenate(cols).astype(np.int32)
        v = np.concatenate([full[c, j] for j, c in enumerate(cols)])
        if chol is None:
            chol = capi.HipCholesky(n, cp, ri, ordering=capi.ORDERING_NATURAL)
        chol.factorize(v)
        b = rng.standard_normal(n)
        want = np.linalg.solve(full, b)
        # diagonally dominant: condition below (5 + 2) / (4 - 2); both solutions backward stable
        assert np.abs(chol.solve(b) - want).max() <= 4 * n * EPS * 3.5 * np.abs(want).max()


@pytest.mark.parametrize("damping", [dict(), dict(use_diagonal_damping=1)])
def test_assembly_by_list_and_by_scatter(damping):
    """Panels below and above the size from which the matrix is scattered into zeroed panels: one
    pose graph in two elimination orders, whose panels lie on either side, and the larger one
    twice on one optimizer (every panel entry is written again)."""
    prob = capi.gen_pose_graph(18500, 5550, 42)
    params = capi.default_params(iterations=4, early_exit_min_reduction=0.0, **damping)
    runs = []
    for ordering, small in ((capi.ORDERING_NESTED_DISSECTION, True),
                            (capi.ORDERING_MIN_DEGREE, False)):
        opt = capi.HipOptimizer(prob, params, capi.solver_options(ordering=ordering))
        assert (opt.solver_info()["panel"] <= 6 << 20) == small
        runs.append(opt.optimize())
    runs.append(opt.optimize(prob.values))
    for other in runs[1:]:
        assert_same_trajectory(other, runs[0], rtol=1e-8)
        np.testing.assert_allclose(other["values"], runs[0]["values"], rtol=0,
                                   atol=1e-8 * np.abs(runs[0]["values"]).max())
