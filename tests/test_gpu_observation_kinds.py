"""Linearization and cost by the kinds of observations a problem holds: one
camera, several pixel sensors, or stereo among them (an instantiation each),
against the oracle's first LM step, around the 256 edges of a work-group.

Bar: the costs are compensated FP64 sums of the same residuals, each within a
few roundings of pixel coordinates of up to 1e3 against residuals of about
0.1 to 1, so 1e4 x 2.2e-16 x a few: 1e-10 relative leaves a margin. The step
solves a damped system of condition number below 1e6 from sums in another
order, at most 1e6 x 64 x 2.2e-16 = 1.6e-8 relative: 1e-7. The stereo scene is
a loop of 40 cameras, whose slow modes take the condition number to some 1e7,
and whose first steps are rejected until the damping suits it: six iterations
and 1e-6."""
import numpy as np
import pytest

import oracle
import vba
from vba import abi, workloads

from test_gpu_stereo import loop_with_stereo

pytestmark = pytest.mark.gpu


def problem(kind, size):
    if kind == "one_camera":
        return vba.synthesize(abi.SYNTH_CIRCLE, num_cameras=4, num_landmarks=size, seed=size).problem
    if kind == "sensors":
        return workloads.window_problem((5, size, size)).problem
    return loop_with_stereo(seed=size)[0]


@pytest.mark.parametrize("kind,size", [("one_camera", 63), ("one_camera", 64), ("one_camera", 65), ("sensors", 25),
                                       ("sensors", 64), ("sensors", 301), ("stereo", 3), ("stereo", 7)])
def test_observation_kinds(device, kind, size):
    p = problem(kind, size)
    o = vba.default_options(linear_solver=abi.SOLVER_DENSE, max_iterations=6 if kind == "stereo" else 1,
                            robust_kernel=abi.KERNEL_HUBER, robust_scale=1.0)
    got, ref = device.optimize(p, o), oracle.optimize(p, o)
    assert got.status == ref.status == abi.OK, got.message
    assert got.accepted == ref.accepted and any(ref.accepted)
    assert abs(got.result.initial_cost - ref.result.initial_cost) <= 1e-10 * ref.result.initial_cost
    assert abs(got.result.final_cost - ref.result.final_cost) <= 1e-7 * ref.result.final_cost
    step = np.linalg.norm(ref.poses - p.poses)
    assert np.linalg.norm(got.poses - ref.poses) <= (1e-6 if kind == "stereo" else 1e-7) * step
