"""A matrix-free solve that changes to the stored reduced matrix against the
same solve over the edges throughout.

The second is had one LM iteration at a time: a solve of one iteration ends
before its first PCG solve could show that the matrix pays, and the next one
starts from its state and damping. The matrix replaces the product alone and
holds the same operator, so both solves are the same up to FP64 rounding: with
every step a converged one (REJECT at the cap of 100, relative residual 1e-4,
the workloads' setting) 110 scenes ended within 2.6e-8 of each other; the bar
is 1e-6. Where the iterate at the cap is taken as it is (ACCEPT_ITERATE), the
answer hangs on the operator's rounding, and the whole solve stays on the edges:
bit for bit the same."""
import numpy as np
import pytest

import vba
from vba import abi, workloads

pytestmark = pytest.mark.gpu


def one_iteration_at_a_time(device, problem, o):
    """(poses, landmarks, accept vector): the LM loop over the edges."""
    step = abi.Options.from_buffer_copy(o)
    step.max_iterations = 1
    poses, landmarks, accepted, lam = problem.poses, problem.landmarks, [], o.initial_lambda
    for _ in range(o.max_iterations):
        step.initial_lambda = lam
        out = device.optimize(problem.with_state(poses, landmarks), step)
        assert out.status == abi.OK, out.message
        it, = out.iterations
        accepted.append(bool(it["step_accepted"]))
        if accepted[-1]:
            poses, landmarks = out.poses, out.landmarks
            lam = max(lam * o.lambda_decrease_factor, o.min_lambda)
        else:
            lam = min(lam * o.lambda_increase_factor, o.max_lambda)
        if out.result.converged:
            break
    return poses, landmarks, accepted


def launches(device, problem, o):
    """The whole solve: its output and the products it ran over (edges, matrix)."""
    device.profile(True)
    out = device.optimize(problem, o)
    device.profile(False, reset=False)
    assert out.status == abi.OK, out.message
    return out, device.profile_query("schur_apply")["launches"], device.profile_query("explicit_apply")["launches"]


def scene(cameras, landmarks, seed):
    return vba.synthesize(abi.SYNTH_LOOP, num_cameras=cameras, num_landmarks=landmarks, seed=seed,
                          scene_scale=200.0 * cameras / 1200.0).problem


def relative(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("precision", [abi.PRECISION_FP64, abi.PRECISION_MIXED])
@pytest.mark.parametrize("cameras,landmarks,seed,iterations", [(141, 11276, 1579, 9), (114, 11423, 1527, 15)])
def test_the_matrix_is_the_edges_operator(device, precision, cameras, landmarks, seed, iterations):
    problem = scene(cameras, landmarks, seed)
    o = workloads.loop_options(precision, abi.PCG_MAXIT_REJECT, max_iterations=iterations)
    out, over_edges, over_matrix = launches(device, problem, o)
    assert over_edges > 0 and over_matrix > 0
    poses, lms, accepted = one_iteration_at_a_time(device, problem, o)
    assert out.accepted == accepted and any(accepted)
    assert relative(out.poses, poses) <= 1e-6
    assert relative(out.landmarks, lms) <= 1e-6


@pytest.mark.parametrize("precision", [abi.PRECISION_FP64, abi.PRECISION_MIXED])
@pytest.mark.parametrize("cameras,landmarks,seed,iterations", [(163, 40009, 7003, 15), (114, 11423, 1527, 15)])
def test_capped_iterates_keep_their_operator(device, precision, cameras, landmarks, seed, iterations):
    problem = scene(cameras, landmarks, seed)
    o = workloads.loop_options(precision, abi.PCG_MAXIT_ACCEPT_ITERATE, max_iterations=iterations)
    out, over_edges, over_matrix = launches(device, problem, o)
    assert any(it["pcg_iterations"] == o.max_pcg_iterations for it in out.iterations)
    assert over_edges > 0 and over_matrix == 0
    poses, lms, accepted = one_iteration_at_a_time(device, problem, o)
    assert out.accepted == accepted
    assert np.array_equal(out.poses, poses) and np.array_equal(out.landmarks, lms)


def test_a_solve_does_not_depend_on_those_before_it(device):
    """Short solves, whose few iterations left do not pay for the matrix, then
    a long one on the same handle: as on a handle of its own. One of the short
    ones passes the cost of the lists and fails that of the blocks."""
    problem = scene(300, 60000, 41)
    o = workloads.loop_options(abi.PRECISION_MIXED, abi.PCG_MAXIT_REJECT, max_iterations=15)
    handle = device.prepare(problem, o)
    want = handle.solve(o)
    state = handle.state()
    handle.free()
    for iterations in range(2, 9):
        handle = device.prepare(problem, o)
        short = abi.Options.from_buffer_copy(o)
        short.max_iterations = iterations
        assert handle.solve(short).status == abi.OK
        device.profile(True)
        got = handle.solve(o)
        device.profile(False, reset=False)
        assert device.profile_query("explicit_apply")["launches"] > 0
        assert got.iterations == want.iterations
        assert all(np.array_equal(a, b) for a, b in zip(handle.state(), state))
        handle.free()
