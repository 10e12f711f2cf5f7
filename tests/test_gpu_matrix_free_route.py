"""The matrix-free solver's change of operator: once a PCG solve has shown
that it pays, the product runs over the explicit reduced matrix, whose
structure and term lists are built on the device from the problem's edges.

Checked over the forms the edges take (fixed poses and landmarks among the
others, a pose without observations, rig edges with several observations,
lenses, observations given in any order), in both precisions, against the
oracle's matrix-free solver with the bars of the other parity tests: FP64 final
cost within 1e-9 relative, mixed 1e-6, camera centres within 1e-6 of the
extent. The PCG solves run to a relative residual of 1e-9 and may not stop
short of it: a solve that takes the iterate at its cap stays on the edges."""
import numpy as np
import pytest

import oracle
import vba
from vba import abi

pytestmark = pytest.mark.gpu


def loop(cams=60, lms=5000, seed=3):
    return vba.synthesize(abi.SYNTH_LOOP, num_cameras=cams, num_landmarks=lms, seed=seed, scene_scale=cams / 6.0)


def options(precision, policy=abi.PCG_MAXIT_REJECT, iterations=5, **kw):
    o = dict(linear_solver=abi.SOLVER_MATRIX_FREE, max_iterations=iterations, max_pcg_iterations=1000,
             pcg_relative_tolerance=1e-9, robust_kernel=abi.KERNEL_HUBER, robust_scale=1.0, precision=precision,
             pcg_maxit_policy=policy)
    o.update(kw)
    return vba.default_options(**o)


def solve_on_both_operators(device, problem, o):
    """The solve, with the launches of the edge product and of the matrix
    product counted: both must have run."""
    pp = device.prepare(problem, o)
    device.profile(True)
    out = pp.solve(o)
    device.profile(False, reset=False)
    assert out.status == abi.OK, out.message
    assert device.profile_query("schur_apply")["launches"] > 0
    assert device.profile_query("explicit_apply")["launches"] > 0
    state = pp.state()
    # timing or not, again or not: the same solve bit for bit
    again = pp.solve(o)
    assert again.iterations == out.iterations
    p, l = pp.state()
    assert np.array_equal(p, state[0]) and np.array_equal(l, state[1])
    pp.free()
    return out, state


def compare(device, problem, extent, o, solve=solve_on_both_operators):
    out, (poses, _) = solve(device, problem, o)
    ro = vba.default_options()
    for f, _ in abi.Options._fields_:
        setattr(ro, f, getattr(o, f))
    ro.precision = abi.PRECISION_FP64
    ref = oracle.optimize(problem, ro)
    assert out.accepted == ref.accepted
    rel = abs(out.result.final_cost - ref.result.final_cost) / ref.result.final_cost
    assert rel <= (1e-9 if o.precision == abi.PRECISION_FP64 else 1e-6), rel
    d = np.linalg.norm(vba.camera_centres(poses) - vba.camera_centres(ref.poses), axis=1).max()
    assert d <= 1e-6 * extent, d


@pytest.mark.parametrize("precision", [abi.PRECISION_FP64, abi.PRECISION_MIXED])
def test_loop(device, precision):
    s = loop()
    compare(device, s.problem, s.scene_extent, options(precision))


@pytest.mark.parametrize("precision", [abi.PRECISION_FP64, abi.PRECISION_MIXED])
def test_fixed_and_unobserved(device, precision):
    s = loop(cams=70, lms=6000, seed=5)
    p = s.problem.copy()
    p.pose_fixed[[7, 8, 33, 64]] = 1           # across bitmap words
    p.landmark_fixed[::11] = 1
    keep = p.obs_pose_ids != p.pose_ids[40]    # no observation of pose 40
    p.obs_pose_ids, p.obs_landmark_ids, p.obs_xy = p.obs_pose_ids[keep], p.obs_landmark_ids[keep], p.obs_xy[keep]
    order = np.random.default_rng(1).permutation(len(p.obs_xy))
    p.obs_pose_ids, p.obs_landmark_ids, p.obs_xy = p.obs_pose_ids[order], p.obs_landmark_ids[order], p.obs_xy[order]
    p.pose_fixed[40] = 1
    # (damped enough for every system to reach its residual)
    compare(device, p, s.scene_extent, options(precision, iterations=30, initial_lambda=0.1, min_lambda=0.1))


def test_rig_edges(device):
    s = vba.synthesize(abi.SYNTH_STEREO_WINDOW, num_cameras=36, num_landmarks=4000, seed=9)
    compare(device, s.problem, s.scene_extent,
            options(abi.PRECISION_FP64, robust_kernel=abi.KERNEL_CAUCHY))


def test_lenses_per_camera(device):
    s = vba.synthesize(abi.SYNTH_CITY, num_cameras=60, num_landmarks=27000, seed=4)
    o = options(abi.PRECISION_MIXED, robust_scale=2.0)
    compare(device, s.problem, s.scene_extent, o)


def solve_on_the_edges(device, problem, o):
    pp = device.prepare(problem, o)
    device.profile(True)
    out = pp.solve(o)
    device.profile(False, reset=False)
    assert out.status == abi.OK, out.message
    assert device.profile_query("schur_apply")["launches"] > 0
    assert device.profile_query("explicit_apply")["launches"] == 0
    state = pp.state()
    pp.free()
    return out, state


@pytest.mark.parametrize("precision", [abi.PRECISION_FP64, abi.PRECISION_MIXED])
@pytest.mark.parametrize("policy", [abi.PCG_MAXIT_ACCEPT_ITERATE, abi.PCG_MAXIT_REJECT])
def test_long_tracks_stay_on_the_edges(device, precision, policy):
    """Every landmark in every camera: more terms an edge than the lists may
    take, so the product stays on the edges. (A second fixed camera holds the
    scale, along which the precisions would part.)"""
    s = vba.synthesize(abi.SYNTH_CIRCLE, num_cameras=40, num_landmarks=2000, seed=2)
    p = s.problem.copy()
    p.pose_fixed[[0, 13]] = 1
    o = options(precision, policy, iterations=12, robust_kernel=abi.KERNEL_HUBER)
    compare(device, p, s.scene_extent, o, solve_on_the_edges)


@pytest.mark.parametrize("precision", [abi.PRECISION_FP64, abi.PRECISION_MIXED])
def test_the_iterate_at_the_cap_stays_on_the_edges(device, precision):
    s = loop()
    compare(device, s.problem, s.scene_extent, options(precision, abi.PCG_MAXIT_ACCEPT_ITERATE), solve_on_the_edges)


@pytest.mark.parametrize("cams,lms", [(3, 60), (31, 2000), (32, 2000), (33, 2000), (65, 4000)])
def test_explicit_solver_on_the_device_lists(device, cams, lms):
    """Row bitmaps at their words' edges, short rows and lists: one LM step
    against the oracle's dense solve of the same system. PCG to 1e-12 and a
    condition number up to some 1e7 leave steps 1e-5 apart at most."""
    s = vba.synthesize(abi.SYNTH_LOOP, num_cameras=cams, num_landmarks=lms, seed=cams, scene_scale=max(4.0, cams / 6.0))
    o = options(abi.PRECISION_FP64, iterations=1, linear_solver=abi.SOLVER_PCG_EXPLICIT, pcg_relative_tolerance=1e-12,
                max_pcg_iterations=5000, initial_lambda=1e-2)
    got = device.optimize(s.problem, o)
    o.linear_solver = abi.SOLVER_DENSE
    ref = oracle.optimize(s.problem, o)
    assert got.status == ref.status == abi.OK, got.message
    assert got.accepted == ref.accepted
    a, b = got.iterations[0], ref.iterations[0]
    assert abs(a["max_pose_step"] - b["max_pose_step"]) <= 1e-5 * b["max_pose_step"]
    assert abs(a["cost_after"] - b["cost_after"]) <= 1e-5 * b["cost_after"]
    assert np.abs(got.poses - ref.poses).max() <= 1e-5 * b["max_pose_step"]
