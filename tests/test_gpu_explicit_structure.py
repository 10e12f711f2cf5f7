"""The explicit reduced matrix's structure beyond the device build's limits, and
the memory it keeps."""
import ctypes as C

import numpy as np
import pytest

import vba
from vba import abi

pytestmark = pytest.mark.gpu


def scene(cameras, landmarks, seed=4):
    return vba.synthesize(abi.SYNTH_LOOP, num_cameras=cameras, num_landmarks=landmarks, seed=seed,
                          scene_scale=200.0 * cameras / 1200.0).problem


def options(solver, **kw):
    o = dict(linear_solver=solver, max_iterations=8, max_pcg_iterations=500, pcg_relative_tolerance=1e-8,
             initial_lambda=1.0, robust_kernel=abi.KERNEL_HUBER, robust_scale=1.0)
    o.update(kw)
    return vba.default_options(**o)


def free_bytes(device):
    free, total = C.c_size_t(), C.c_size_t()
    assert device.lib.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def matrix_sizes(problem):
    """(terms, stored blocks) of the reduced matrix, all poses but the fixed ones."""
    slot = {int(i): k for k, i in enumerate(problem.pose_ids)}
    pose = np.array([slot[int(i)] for i in problem.obs_pose_ids])
    keep = problem.pose_fixed[pose] == 0
    order = np.lexsort((pose[keep], problem.obs_landmark_ids[keep]))
    pose, lm = pose[keep][order], problem.obs_landmark_ids[keep][order]
    n = len(problem.pose_ids)
    pairs, terms, d = [], 0, 0
    while True:  # pairs of a landmark's observations d places apart
        same = lm[d:] == lm[:len(lm) - d]
        if not same.any():
            break
        terms += int(same.sum())
        pairs.append(np.unique(pose[:len(pose) - d][same] * n + pose[d:][same]))
        d += 1
    upper = np.unique(np.concatenate(pairs))
    return terms, 2 * len(upper) - int((upper // n == upper % n).sum())


def test_the_lists_scratch_is_given_back(device):
    """What the explicit solver adds to a handle is its lists and blocks, not
    the row bitmaps (32 MB at 16,000 poses) that the lists were built from."""
    problem = scene(16000, 24000)
    handle = device.prepare(problem, options(abi.SOLVER_MATRIX_FREE))
    assert handle.solve(options(abi.SOLVER_MATRIX_FREE, max_iterations=1)).status == abi.OK
    before = free_bytes(device)
    assert handle.solve(options(abi.SOLVER_PCG_EXPLICIT, max_iterations=1)).status == abi.OK
    used = before - free_bytes(device)
    handle.free()
    terms, blocks = matrix_sizes(problem)
    lists = 12 * terms + blocks * (4 + 288) + (blocks + 16000) / 2 * 20 + 16000 * 60
    # the rest is the allocations' granularity and what the runtime takes for itself, 8 MB at a time (11 to 19 MB
    # seen; 44 with the bitmaps)
    assert used <= 1.02 * lists + (24 << 20)


def test_structure_built_on_the_host(device):
    """More poses than the device build takes: the explicit solver's lists come
    from the host, and its steps are those of the product over the edges. A
    matrix-free solve does not take such a structure over."""
    problem = scene(16400, 12000)
    free, explicit = options(abi.SOLVER_MATRIX_FREE), options(abi.SOLVER_PCG_EXPLICIT)
    handle = device.prepare(problem, free)
    a = handle.solve(free)
    poses, landmarks = handle.state()
    b = handle.solve(explicit)
    p, l = handle.state()
    assert a.status == b.status == abi.OK and a.accepted == b.accepted and any(a.accepted)
    # both solve each system to 1e-8 at a damping of 1 and more
    assert np.linalg.norm(p - poses) <= 1e-7 * np.linalg.norm(poses)
    assert np.linalg.norm(l - landmarks) <= 1e-7 * np.linalg.norm(landmarks)
    assert b.result.total_pcg_iterations > 0
    device.profile(True)
    again = handle.solve(free)
    device.profile(False, reset=False)
    assert device.profile_query("explicit_apply")["launches"] == 0
    assert again.iterations == a.iterations
    handle.free()


@pytest.mark.parametrize("precision", [abi.PRECISION_FP64, abi.PRECISION_MIXED])
@pytest.mark.parametrize("cameras,landmarks", [(65, 200), (66, 3000), (3000, 6000), (3001, 6000), (3003, 120000)])
def test_few_and_many_rows_short_and_long_lists(device, cameras, landmarks, precision):
    """Products with four waves a row (up to 3,000 rows) and with one, lists of
    up to 40 terms a block summed by eight lanes and longer ones by a wave, the
    last work-group not full: the steps are those of the product over the edges
    (both to 1e-8, at a damping that lets CG get there)."""
    problem = scene(cameras, landmarks)
    kw = dict(precision=precision, max_iterations=3, initial_lambda=1e4, max_lambda=1e10,
              pcg_maxit_policy=abi.PCG_MAXIT_ACCEPT_ITERATE)
    a = device.optimize(problem, options(abi.SOLVER_MATRIX_FREE, **kw))
    b = device.optimize(problem, options(abi.SOLVER_PCG_EXPLICIT, **kw))
    assert a.status == b.status == abi.OK and a.accepted == b.accepted
    step = np.linalg.norm(a.poses - problem.poses)
    for x, y in zip(a.iterations, b.iterations):
        assert 0 < x["pcg_iterations"] < 500 and 0 < y["pcg_iterations"] < 500
        assert abs(x["max_pose_step"] - y["max_pose_step"]) <= 1e-6 * x["max_pose_step"]
    assert np.linalg.norm(a.poses - b.poses) <= 1e-6 * max(step, 1e-3)


def test_fixed_poses_do_not_count_against_the_lists(device):
    """Six landmarks seen by 16,000 fixed poses and 4 variable ones: 768M pairs
    of observations, more than the lists can hold, but 60 terms, as fixed poses
    have no part in the matrix."""
    rng = np.random.default_rng(7)
    n = 16004
    centres = np.stack([rng.uniform(-1, 1, n), rng.uniform(-1, 1, n), np.zeros(n)], 1)
    points = np.stack([rng.uniform(-1, 1, 6), rng.uniform(-1, 1, 6), rng.uniform(5, 7, 6)], 1)
    rel = points[None] - centres[:, None]
    xy = 500.0 * rel[..., :2] / rel[..., 2:] + np.array([320.0, 240.0]) + rng.normal(0, 0.3, (n, 6, 2))
    poses = np.concatenate([np.tile([1.0, 0, 0, 0], (n, 1)), -centres], 1)
    poses[-4:, 4:] += 0.05
    fixed = np.ones(n, np.uint8)
    fixed[-4:] = 0
    problem = vba.BundleProblem(
        camera=vba.camera(abi.CAMERA_PINHOLE, [500.0, 500.0, 320.0, 240.0], 640, 480),
        pose_ids=np.arange(n), poses=poses, pose_fixed=fixed, landmark_ids=np.arange(6), landmarks=points + 0.02,
        landmark_fixed=np.zeros(6, np.uint8), obs_pose_ids=np.repeat(np.arange(n), 6),
        obs_landmark_ids=np.tile(np.arange(6), n), obs_xy=xy.reshape(-1, 2))
    a = device.optimize(problem, options(abi.SOLVER_PCG_EXPLICIT, initial_lambda=1e-3, max_iterations=3))
    assert a.status == abi.OK, a.message
    b = device.optimize(problem, options(abi.SOLVER_DENSE, initial_lambda=1e-3, max_iterations=3))
    assert a.accepted == b.accepted and any(a.accepted)
    assert abs(a.result.final_cost - b.result.final_cost) <= 1e-9 * b.result.final_cost
    assert np.abs(a.poses - b.poses).max() <= 1e-7


@pytest.mark.parametrize("cameras,landmarks", [(40, 12000), (300, 40000)])
def test_two_builds_give_the_same_bits(device, cameras, landmarks):
    """The term lists' order, and so every sum's, is that of the edges: a
    structure built again, on a new handle, gives the same solve (a block's
    terms are some 200 neighbouring edges of its row here, so most of a wave's
    lanes add to the same lists)."""
    problem = scene(cameras, landmarks)
    o = options(abi.SOLVER_PCG_EXPLICIT, initial_lambda=1e-3, max_iterations=4)
    outs = [device.optimize(problem, o) for _ in range(4)]
    assert outs[0].status == abi.OK and any(outs[0].accepted)
    for out in outs[1:]:
        assert out.iterations == outs[0].iterations
        assert np.array_equal(out.poses, outs[0].poses) and np.array_equal(out.landmarks, outs[0].landmarks)
