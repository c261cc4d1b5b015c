"""The batched solve at the chain lengths where its elimination changes shape: the chain is cut at
its middle pose (odd and even lengths, one and two poses have no or one eliminated pose), a pose's
matching factors are dealt to 1, 2 or 4 lanes (more than 32, 17 to 32, up to 16 poses), and a pose
may have no matching factor or no odometry to the next. Held to the oracle's trajectory with
test_batch_gpu.py's tolerance; the FP32-Jacobian form, whose steps are its own, to the oracle's
minimum."""
import numpy as np
import pytest

from symforce_amd import _capi as capi
import oracle_wrap as ow
from test_optimizer_gpu import assert_same_trajectory

pytestmark = pytest.mark.gpu


def without(prob, drop):
    """The problem without the factors in `drop`."""
    keep = [f for f in range(prob.n_factors) if f not in drop]
    fptr, fargs = [0], []
    for f in keep:
        fargs.extend(prob.fargs[prob.fptr[f]:prob.fptr[f + 1]].tolist())
        fptr.append(len(fargs))
    return capi.Problem(prob.letters, prob.subs, prob.supers, prob.types, prob.values,
                        prob.ftypes[keep], fptr, fargs, prob.opt_keys, prob.info)


def check(probs, params):
    res = capi.HipBatch(probs, params).solve()["problems"]
    for prob, got in zip(probs, res):
        ora = ow.OracleProblem(prob).optimize(params)
        assert_same_trajectory(got, ora, rtol=1e-8)
        np.testing.assert_allclose(got["values"], ora["values"], rtol=0,
                                   atol=1e-8 * max(1.0, np.abs(ora["values"]).max()))


@pytest.mark.parametrize("poses", [1, 2, 3, 4, 5, 15, 16, 17, 31, 32, 33, 63, 64])
def test_chain_lengths(poses):
    probs = [capi.gen_localization(poses, lm, 0.3, seed=10 * poses + lm) for lm in (9, 21, 40)]
    check(probs, capi.default_params(iterations=20))


@pytest.mark.parametrize("poses", [1, 2, 16, 17, 32, 33, 64])
def test_chain_lengths_fp32(poses):
    probs = [capi.gen_localization(poses, lm, 0.3, seed=10 * poses + lm) for lm in (9, 21, 40)]
    params = capi.default_params(iterations=40, early_exit_min_reduction=0.0)
    res = capi.HipBatch(probs, params, precision=capi.PRECISION_F32_JAC).solve()["problems"]
    for prob, got in zip(probs, res):
        ora = ow.OracleProblem(prob).optimize(params)
        assert got["iterations"][0]["new_error"] == \
            pytest.approx(ora["iterations"][0]["new_error"], rel=1e-8)  # FP64 residuals
        best, want = (r["iterations"][r["best_index"]]["new_error"] for r in (got, ora))
        assert best == pytest.approx(want, rel=1e-8)


@pytest.mark.parametrize("poses", [2, 7, 16, 33])
def test_diagonal_damping(poses):
    probs = [capi.gen_localization(poses, 20, 0.3, seed=poses)]
    for keep in (0, 1):
        check(probs, capi.default_params(iterations=15, use_diagonal_damping=1,
                                         keep_max_diagonal_damping=keep))


@pytest.mark.parametrize("poses,gap", [(6, 0), (6, 2), (17, 8), (34, 17)])
def test_chain_with_a_gap(poses, gap):
    # no odometry from pose `gap` to the next: the coupling block between them is zero
    prob = capi.gen_localization(poses, 20, 0.5, seed=poses + gap)
    odo = np.flatnonzero(prob.ftypes == capi.FACTOR_ODOMETRY)
    check([without(prob, {int(odo[gap])})], capi.default_params(iterations=15))


def test_pose_without_matches():
    prob = capi.gen_localization(9, 20, 0.5, seed=3)
    poses = [int(prob.fargs[p]) for p in prob.fptr[:-1]]
    first = poses[int(np.flatnonzero(prob.ftypes == capi.FACTOR_ODOMETRY)[4])]
    drop = {f for f in range(prob.n_factors)
            if prob.ftypes[f] == capi.FACTOR_MATCHING and poses[f] == first}
    assert drop
    check([without(prob, drop)], capi.default_params(iterations=15))


@pytest.mark.parametrize("poses", [1, 2, 9, 33])
@pytest.mark.parametrize("damping", [dict(), dict(use_diagonal_damping=1, use_unit_damping=0)])
def test_infinite_damping(poses, damping):
    """lambda = inf: a step of exact zeros, at whose unchanged error the run ends (lambda has no
    bound to grow to); the oracle's linear error is inf * 0 and not compared."""
    prob = capi.gen_localization(poses, 20, 0.5, seed=poses)
    params = capi.default_params(iterations=5, initial_lambda=np.inf, lambda_upper_bound=np.inf,
                                 **damping)
    got = capi.HipBatch([prob], params).solve()["problems"][0]
    ora = ow.OracleProblem(prob).optimize(params)
    for k in ("status", "failure_reason", "best_index"):
        assert got[k] == ora[k], k
    assert [it["update_accepted"] for it in got["iterations"]] == \
        [it["update_accepted"] for it in ora["iterations"]]
    np.testing.assert_allclose([it["new_error"] for it in got["iterations"]],
                               [it["new_error"] for it in ora["iterations"]], rtol=1e-12)
    np.testing.assert_array_equal(got["values"], prob.values)
