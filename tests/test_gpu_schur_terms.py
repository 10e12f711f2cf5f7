"""The Schur blocks' term sums (one wave per 6x6 block) at list lengths around
the wave's 64 lanes, in the dense and the explicit reduced solve, against the
oracle's first LM step from the same problem.

Bar: every camera sees every landmark, so each block sums as many terms as
there are landmarks. The step solves a system whose condition number stays
below 1e6 here (one camera fixed, wide baselines, lambda 1e-3), so FP64 sums
in another order move it by at most about 1e6 x 64 x 2.2e-16 = 1.6e-8
relative; 1e-7 leaves a margin."""
import numpy as np
import pytest

import oracle
import vba
from vba import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("landmarks", [9, 63, 64, 65, 127, 129, 257])
@pytest.mark.parametrize("solver", [abi.SOLVER_DENSE, abi.SOLVER_PCG_EXPLICIT])
def test_term_lists_around_a_wave(device, landmarks, solver):
    s = vba.synthesize(abi.SYNTH_CIRCLE, num_cameras=6, num_landmarks=landmarks, seed=landmarks)
    o = vba.default_options(linear_solver=solver, max_iterations=1, max_pcg_iterations=200,
                            pcg_relative_tolerance=1e-13)
    got = device.optimize(s.problem, o)
    assert got.status == abi.OK, got.message
    o.linear_solver = abi.SOLVER_DENSE
    ref = oracle.optimize(s.problem, o)
    assert got.accepted == ref.accepted == [True]
    step = np.linalg.norm(ref.poses - s.problem.poses)
    assert np.linalg.norm(got.poses - ref.poses) <= 1e-7 * step
    lstep = np.linalg.norm(ref.landmarks - s.problem.landmarks)
    assert np.linalg.norm(got.landmarks - ref.landmarks) <= 1e-7 * lstep
