"""The one-work-group dense solve (at most 256 unknowns, 16-column tiles held
in registers, 47 panel rows per wave) at sizes around its tiles, its waves'
rows and its limit, and windows around that limit in a batch.

Bar: spd(n) below has a condition number under 6, so a backward stable
Cholesky solve errs by at most about 6 n^1.5 eps relative (5.5e-12 at 256);
the LU systems have a condition number of 4 and 1e-10 as the other LU tests."""
import numpy as np
import pytest

import oracle
import vba
from vba import abi

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 15, 16, 17, 31, 33, 63, 64, 65, 110, 112, 200, 255, 256]


def spd(n):
    rng = np.random.default_rng(n)
    a = rng.standard_normal((n, n))
    return a @ a.T + n * np.eye(n), rng.standard_normal(n)


@pytest.mark.parametrize("n", SIZES)
def test_cholesky(device, n):
    h, b = spd(n)
    st, x = device.dense_solve(h, b)
    assert st == abi.OK
    ref = np.linalg.solve(h, b)
    assert np.abs(x - ref).max() <= 6 * n ** 1.5 * 2.3e-16 * np.abs(ref).max()


@pytest.mark.parametrize("n", [16, 17, 255, 256])
@pytest.mark.parametrize("at", ["first", "last"])
def test_lu_fallback_on_a_bad_pivot(device, n, at):
    """A negative pivot in the first or only in the last column: LU with
    partial pivoting on the system as given."""
    h, b = spd(n)
    k = 0 if at == "first" else n - 1
    h[k, k] = -h[k, k]
    st, x = device.dense_solve(h, b)
    ref = np.linalg.solve(h, b)
    assert st == abi.OK
    assert np.abs(x - ref).max() <= 1e-10 * np.abs(ref).max()


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_non_finite_pivots_end(device, bad):
    """A non-finite pivot fails the Cholesky as before; the LU then runs on
    the same system and the call ends, with a result or singular."""
    h, b = spd(40)
    h[21, 21] = bad
    st, x = device.dense_solve(h, b)
    assert st in (abi.OK, abi.ERR_SINGULAR_SYSTEM)


def test_windows_around_the_limit_equal_single_solves(device):
    """42 variable poses (252 unknowns) stay in registers, 43 and more use the
    factor in global memory; one batch holds both."""
    o = vba.default_options(linear_solver=abi.SOLVER_DENSE, max_iterations=3, robust_kernel=abi.KERNEL_CAUCHY,
                            robust_scale=1.0)
    scenes = [vba.synthesize(abi.SYNTH_STEREO_WINDOW, num_cameras=k, num_landmarks=900, seed=40 + k)
              for k in (43, 44, 12)]
    batch = device.optimize_batch([s.problem for s in scenes], o)
    assert batch.status == abi.OK, batch.message
    for s, got in zip(scenes, batch.windows):
        ref = oracle.optimize(s.problem, o)
        assert got.accepted == ref.accepted
        assert abs(got.result.final_cost - ref.result.final_cost) <= 1e-9 * ref.result.final_cost
        d = np.linalg.norm(vba.camera_centres(got.poses) - vba.camera_centres(ref.poses), axis=1).max()
        assert d <= 1e-6 * s.scene_extent
