"""The reduced camera system's pair sums at the pair counts where their batches of eight and work
items of 512 end: few cameras with few to many common points, the Schur path's run held to the
full-system LDL^T's (an independent assembly and factorization of the same Hessian). The FP32 form
(other strides, copies and reads) is held to itself with the landmarks in reverse order: every
observation's FP32 blocks are the same bits, the pair sums are FP64 and only their order differs, so
a pair that is lost or counted twice at a batch's or an item's end is another pair there."""
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


def reversed_landmarks(prob):
    """The same problem with its Vector3 landmarks stored, and so eliminated, in reverse order, and
    the storage places its values come from."""
    at = np.flatnonzero((prob.types == capi.TYPE_VECTOR3) & (prob.letters == ord("p")))
    other = np.arange(prob.n_keys)
    other[at] = at[::-1]
    place = np.arange(prob.values.size)
    for k in at:
        o, q = prob.storage_offsets[k], prob.storage_offsets[other[k]]
        place[q:q + 3] = np.arange(o, o + 3)
    return capi.Problem(prob.letters, prob.subs, prob.supers, prob.types, prob.values[place],
                        prob.ftypes, prob.fptr, other[prob.fargs], prob.opt_keys, prob.info), place


@pytest.mark.parametrize("gen", ["snavely", "circle"])  # camera nodes of 9 and of 6
@pytest.mark.parametrize("points", [7, 8, 9, 15, 16, 17, 31, 33, 511, 513, 1030])
def test_pair_counts_fp32(gen, points):
    prob = (capi.gen_ba_snavely if gen == "snavely" else capi.gen_ba_circle)(2, points, seed=points)
    back, place = reversed_landmarks(prob)
    assert not np.array_equal(place, np.arange(place.size))
    # one step: the next one's FP32 Jacobians would round the steps' last bits
    params = capi.default_params(iterations=1, initial_lambda=1.0)

    def run(p, precision):
        return capi.HipOptimizer(p, params, capi.solver_options(
            linear_solver=capi.SOLVER_SCHUR, precision=precision)).optimize()
    a, b, ref = (run(prob, capi.PRECISION_F32_JAC), run(back, capi.PRECISION_F32_JAC),
                 run(prob, capi.PRECISION_F64))
    assert_same_trajectory(a, b, rtol=1e-8)  # as above
    np.testing.assert_allclose(a["values"][place], b["values"], rtol=0,
                               atol=1e-7 * max(1.0, np.abs(b["values"]).max()))
    # and it is the FP64 step, to FP32 rounding (the FP32 form's tests' bound)
    e0, e64 = (it["new_error"] for it in ref["iterations"])
    assert a["iterations"][0]["new_error"] == e0
    assert abs(a["iterations"][1]["new_error"] - e64) <= 1e-2 * abs(e0 - e64)
