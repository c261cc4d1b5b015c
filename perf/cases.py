"""Performance cases: what programs built on this library spend their time in.

    listed()             the cases, as plain dicts
    draw(rng)            one more case of the same kinds, sizes spread over their ranges
    prepare(case, seed)  inputs and handles a program holds before the call
    run(state)           one pass through the public entry points, its outputs whole
    work(case)           bytes and flops one pass cannot do without
    exact(case, seed)    what run returns, by numpy in 64 bits (where that is practical)

A case's structure (who sees what, the loop closures) comes from the library's generators; the
seed moves the starting point of every optimized key, so another seed is another set of inputs to
the same plan. Optimizer passes run a fixed number of Levenberg-Marquardt iterations.
"""
from __future__ import annotations

import ctypes as C
import functools
import math

import numpy as np
import torch

from symforce_amd import _capi as capi


def listed():
    return [
        # The smallest optimizer call: the reference's ten-pose smoothing test and its twelve
        # iterations (a program that smooths a short window at frame rate: latency only).
        dict(name="chain_10", kind="chain", poses=10, iterations=12),
        # The repository's first configuration: 20 cameras around 1000 landmarks, the landmarks
        # kept in the sparse Cholesky path (a visual-odometry window).
        dict(name="circle_20x1000", kind="circle", cams=20, points=1000, iterations=6),
        # A mid-size reconstruction on the Schur path, odd sizes.
        dict(name="ba_137x9001", kind="ba", cams=137, points=9001, precision=0, pcg=0,
             iterations=10),
        # The headline configuration: 1000 cameras, 200 000 landmarks, ~1 M observations, FP64.
        dict(name="ba_1000x200000", kind="ba", cams=1000, points=200000, precision=0, pcg=0,
             iterations=10),
        # The same problem in the fast form: FP32 storage, truncated block-Jacobi PCG.
        dict(name="ba_1000x200000_f32_pcg", kind="ba", cams=1000, points=200000, precision=1,
             pcg=1, iterations=10),
        # Pose-graph SLAM at the size of one robot's session.
        dict(name="graph_2503", kind="graph", poses=2503, iterations=8),
        # Pose-graph SLAM at the repository's largest configuration.
        dict(name="graph_100000", kind="graph", poses=100000, iterations=5),
        # One small localization problem through the allocation-free batched entry: the latency of
        # a serving loop with a single robot.
        dict(name="batch_1", kind="batch", problems=1, precision=0),
        # A serving loop's batch, device-resident tables, the FP32-Jacobian form.
        dict(name="batch_499_f32", kind="batch", problems=499, precision=1),
        # The batched configuration: 4096 uneven problems, host results through the batch handle.
        dict(name="batch_host_4096", kind="batch_host", problems=4096, precision=0),
        # The linear-solver adapter a host Levenberg-Marquardt loop drives: factorize a Hessian of
        # host values, solve one right-hand side.
        dict(name="cholesky_1501", kind="cholesky", poses=1501),
        # Covariances at an estimate: factorize its Hessian, the dense inverse out.
        dict(name="covariance_151", kind="covariance", poses=151),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["chain", "circle", "ba", "ba", "ba", "graph", "graph", "batch", "batch",
                       "batch_host", "cholesky", "covariance"])
    if kind == "chain":
        return dict(kind=kind, poses=_log_int(rng, 4, 400), iterations=12)
    if kind == "circle":
        return dict(kind=kind, cams=rng.randint(6, 30), points=_log_int(rng, 100, 1500),
                    iterations=6)
    if kind == "ba":
        cams = _log_int(rng, 20, 900)
        fast = rng.random() < 0.3
        return dict(kind=kind, cams=cams, points=int(cams * rng.uniform(60, 200)),
                    precision=int(fast), pcg=int(fast), iterations=10)
    if kind == "graph":
        poses = _log_int(rng, 1500, 90000)  # shorter walks close no loop
        return dict(kind=kind, poses=poses, iterations=8 if poses < 20000 else 5)
    if kind == "batch":
        return dict(kind=kind, problems=_log_int(rng, 1, 500), precision=rng.randint(0, 1))
    if kind == "batch_host":
        return dict(kind=kind, problems=_log_int(rng, 256, 4000), precision=rng.randint(0, 1))
    if kind == "cholesky":
        return dict(kind=kind, poses=_log_int(rng, 150, 1500))
    return dict(kind=kind, poses=_log_int(rng, 15, 150))


# ---- prepare --------------------------------------------------------------------------------
_STRUCTURE_SEED = 42  # the seed the repository's tests and benchmark generate with
_POSES = dict(chain="P", covariance="P", circle="cp", ba="cp", graph="x", cholesky="x",
              batch="w")  # letters of the optimized Pose3 and Vector3 keys


@functools.lru_cache(maxsize=2)
def _structure(kind, *sizes):
    if kind in ("chain", "covariance"):
        return capi.gen_pose_smoothing(*sizes, _STRUCTURE_SEED)
    if kind == "circle":
        return capi.gen_ba_circle(*sizes, _STRUCTURE_SEED)
    if kind == "ba":
        return capi.gen_ba_snavely(*sizes, _STRUCTURE_SEED)
    if kind == "graph":
        return capi.gen_pose_graph(sizes[0], int(0.3 * sizes[0]), _STRUCTURE_SEED)
    return capi.gen_localization_batch(*sizes, _STRUCTURE_SEED)


def _moved(prob, seed, rotation, translation, point, letters):
    """The problem's values with the starting point of its optimized keys (their letters) moved by
    normal noise: Pose3 rotations (radians) and translations, Vector3 points."""
    rng = np.random.default_rng(seed)
    values = prob.values.copy()
    optimized = np.isin(prob.letters, [ord(c) for c in letters])
    at = prob.storage_offsets[optimized & (prob.types == capi.TYPE_POSE3)]
    d = rotation * rng.standard_normal((at.size, 3))
    q = values[at[:, None] + np.arange(4)]
    # q * exp(d): quaternions are x, y, z, w
    half = 0.5 * np.linalg.norm(d, axis=1, keepdims=True)
    e = 0.5 * d * np.sinc(half / np.pi)
    c, v, w = np.cos(half), q[:, :3], q[:, 3:]
    out = np.concatenate([w * e + c * v + np.cross(v, e),
                          c * w - (v * e).sum(1, keepdims=True)], axis=1)
    values[at[:, None] + np.arange(4)] = out / np.linalg.norm(out, axis=1, keepdims=True)
    values[at[:, None] + np.arange(4, 7)] += translation * rng.standard_normal((at.size, 3))
    at = prob.storage_offsets[optimized & (prob.types == capi.TYPE_VECTOR3)]
    values[at[:, None] + np.arange(3)] += point * rng.standard_normal((at.size, 3))
    return values


def _with_values(prob, values):
    return capi.Problem(prob.letters, prob.subs, prob.supers, prob.types, values, prob.ftypes,
                        prob.fptr, prob.fargs, prob.opt_keys, prob.info)


def _optimizer(prob, iterations, **options):
    """As bench.py builds them: dynamic damping, no early exit inside the fixed iterations."""
    params = capi.default_params(lambda_update_type=capi.LAMBDA_DYNAMIC, iterations=iterations,
                                 early_exit_min_reduction=0.0)
    return capi.HipOptimizer(prob, params, capi.solver_options(**options))


def _device(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


def _batch_problems(count, seed):
    probs = _structure("batch", count)
    return [_with_values(p, _moved(p, seed + i, 0.01, 0.02, 0.0, _POSES["batch"]))
            for i, p in enumerate(probs)]


def prepare(case, seed):
    kind = case["kind"]
    seed = int(seed) & 0x3FFFFFFF
    if kind == "chain":
        prob = _structure(kind, case["poses"])
        params = capi.default_params(iterations=case["iterations"])
        return dict(kind="optimize", opt=capi.HipOptimizer(prob, params),
                    values=_moved(prob, seed, 0.02, 0.02, 0.0, _POSES[kind]),
                    iterations=case["iterations"])
    if kind == "circle":
        prob = _structure(kind, case["cams"], case["points"])
        return dict(kind="optimize", opt=_optimizer(prob, case["iterations"]),
                    values=_moved(prob, seed, 0.01, 0.02, 0.02, _POSES[kind]),
                    iterations=case["iterations"])
    if kind == "ba":
        prob = _structure(kind, case["cams"], case["points"])
        more = dict(use_pcg=1, pcg_max_iters=20, pcg_rel_tol=3e-2) if case["pcg"] else {}
        opt = _optimizer(prob, case["iterations"], linear_solver=capi.SOLVER_SCHUR,
                         ordering=capi.ORDERING_NESTED_DISSECTION, precision=case["precision"],
                         **more)
        return dict(kind="optimize", opt=opt,
                    values=_moved(prob, seed, 1e-5, 1e-4, 1e-4, _POSES[kind]),
                    iterations=case["iterations"])
    if kind == "graph":
        prob = _structure(kind, case["poses"])
        opt = _optimizer(prob, case["iterations"], ordering=capi.ORDERING_NESTED_DISSECTION)
        return dict(kind="optimize", opt=opt,
                    values=_moved(prob, seed, 0.002, 0.01, 0.0, _POSES[kind]),
                    iterations=case["iterations"])
    if kind == "batch":
        probs = _batch_problems(case["problems"], seed)
        params = capi.default_params()
        host = capi.batch_pack(probs, params)
        names = ("pose_begin", "pose_soff", "match_ptr", "match_args", "odo_args", "values")
        dev = {k: _device(host[k]) for k in names}
        tables = capi.BatchTables(host["n_problems"], host["total_poses"], host["storage_size"],
                                  *[dev[k].data_ptr() for k in names])
        stats = torch.zeros((case["problems"], 4), dtype=torch.int32, device="cuda")
        return dict(kind="batch", tables=tables, dev=dev, params=params,
                    precision=case["precision"], epsilon=probs[0].info["epsilon"],
                    values=torch.zeros_like(dev["values"]), stats=stats)
    if kind == "batch_host":
        probs = _batch_problems(case["problems"], seed)
        batch = capi.HipBatch(probs, capi.default_params(), precision=case["precision"])
        batch.set_config(2)  # most poses first, as the tuner chooses for uneven problems
        return dict(kind="batch_host", batch=batch, values=np.zeros(sum(batch.sizes)),
                    stats=(capi.OptimizationStats * case["problems"])())
    if kind == "cholesky":
        prob = _structure("graph", case["poses"])
        hip = capi.HipProblem(prob)
        colptr, rowind = hip.hessian_structure()
        lin = hip.linearize(_moved(prob, seed, 0.002, 0.01, 0.0, _POSES[kind]))
        values = lin["hessian_values"]
        values[colptr[:-1]] += 1.0  # the damped diagonal (lambda = 1, unit damping)
        node_ptr = np.arange(0, hip.N + 1, 6, dtype=np.int32)
        chol = capi.HipCholesky(hip.N, colptr, rowind, node_ptr,
                                ordering=capi.ORDERING_NESTED_DISSECTION)
        return dict(kind="cholesky", chol=chol, values=values, b=lin["rhs"], colptr=colptr,
                    rowind=rowind)
    if kind == "covariance":
        prob = _structure(kind, case["poses"])
        hip = capi.HipProblem(prob)
        lin = hip.linearize(_moved(prob, seed, 0.02, 0.02, 0.0, _POSES[kind]))
        return dict(kind="covariance", problem=hip, hessian=lin["hessian_values"])
    raise ValueError(f"unknown kind {kind}")


# ---- run ------------------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    if kind == "optimize":
        r = state["opt"].optimize(state["values"], state["iterations"])
        return dict(values=r["values"], status=r["status"], best_index=r["best_index"],
                    error=r["iterations"][r["best_index"]]["new_error"])
    if kind == "batch":
        capi.batch_solve_noalloc(state["tables"], state["params"], state["precision"],
                                 state["epsilon"], state["values"].data_ptr(),
                                 state["stats"].data_ptr(), None,
                                 torch.cuda.current_stream().cuda_stream)
        return dict(values=state["values"], stats=state["stats"])
    if kind == "batch_host":
        batch = state["batch"]
        capi.check(capi.hip_lib().symhip_batch_solve(
            batch.h, capi.ptr(state["values"], C.c_double), state["stats"], None, None, None))
        return dict(values=state["values"], stats=np.frombuffer(state["stats"], np.int32))
    if kind == "cholesky":
        state["chol"].factorize(state["values"])
        return dict(x=state["chol"].solve(state["b"]))
    return dict(cov=capi.compute_full_covariance(state["problem"], state["hessian"]))


# ---- work -----------------------------------------------------------------------------------
# Flops per linearized factor (residual, Jacobian, its products) and sizes, counted from the
# factor bodies: a Snavely or linear-camera observation, a Pose3 between factor, a landmark match.
_OBS_FLOPS, _BETWEEN_FLOPS, _MATCH_FLOPS = 700, 2200, 500
_TRACK, _BAND = 5, 74  # observations per landmark; cameras covisible with one (the generators')
_BATCH_POSES, _BATCH_MATCHES, _BATCH_ITERATIONS = 27.5, 186, 9


def work(case):
    kind = case["kind"]
    if kind == "chain":
        n, it = case["poses"], 12
        return dict(bytes=8 * 7 * 2 * n, flops=it * n * (_BETWEEN_FLOPS + 3 * 6 ** 3))
    if kind == "circle":
        cams, pts, it = case["cams"], case["points"], case["iterations"]
        obs, nb = cams * pts, 6 * cams
        per = obs * (_OBS_FLOPS + 6 * 9) + pts * nb * nb * 3 + nb ** 3 / 3
        return dict(bytes=8 * (2 * 7 * cams + 2 * 3 * pts + 2 * obs), flops=it * per)
    if kind == "ba":
        cams, pts, it = case["cams"], case["points"], case["iterations"]
        obs, band = _TRACK * pts, min(_BAND, cams)
        pairs = obs * _TRACK
        chol = 9 * cams * (9 * band) ** 2 / (1 if cams > band else 3)
        # one exact solve an iteration, or the PCG's 20 products with S
        solve = 20 * 2 * 81 * cams * band if case["pcg"] else chol
        per = obs * (_OBS_FLOPS + 2 * 81) + pairs * 486 + solve
        return dict(bytes=8 * (2 * 10 * cams + 2 * 3 * pts + 2 * obs), flops=it * per)
    if kind == "graph":
        n, it = case["poses"], case["iterations"]
        edges = 1.2 * n
        per = edges * _BETWEEN_FLOPS + 9000 * n  # elimination: ~0.9 GFLOP at 100 000 nodes
        return dict(bytes=8 * (2 * 7 * n + 7 * edges), flops=it * per)
    if kind in ("batch", "batch_host"):
        n = case["problems"]
        storage = n * 8 * (7 * 2 * _BATCH_POSES + 3 * _BATCH_MATCHES + 100)
        per = (_BATCH_MATCHES * _MATCH_FLOPS + _BATCH_POSES * (_BETWEEN_FLOPS + 1200))
        return dict(bytes=2 * storage, flops=n * _BATCH_ITERATIONS * per)
    if kind == "cholesky":
        n = case["poses"]
        nnz = n * 6 * 10
        return dict(bytes=8 * (nnz + 12 * n), flops=9000 * n)
    n = 6 * case["poses"]
    return dict(bytes=8 * (n * n + n * 10), flops=2.0 * n * n * 36)


# ---- exact ----------------------------------------------------------------------------------
def _dense_lower(n, colptr, rowind, values):
    a = np.zeros((n, n))
    cols = np.repeat(np.arange(n), np.diff(colptr))
    a[rowind, cols] = values
    a[cols, rowind] = values
    return a


def exact(case, seed):
    # The optimizer passes are whole trajectories with no closed form in numpy: None.
    if case["kind"] == "cholesky":
        s = prepare(case, seed)  # its Hessian and right-hand side are the inputs
        a = _dense_lower(len(s["b"]), s["colptr"], s["rowind"], s["values"])
        return dict(x=np.linalg.solve(a, s["b"]))
    if case["kind"] == "covariance":
        s = prepare(case, seed)
        colptr, rowind = s["problem"].hessian_structure()
        return dict(cov=np.linalg.inv(_dense_lower(s["problem"].N, colptr, rowind, s["hessian"])))
    return None
