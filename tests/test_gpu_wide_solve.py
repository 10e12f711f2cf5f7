"""The device-wide dense solve (beyond 256 unknowns: 64-column panels, the
previous panel's update in the same launch, a back substitution per panel) at
sizes around its panels and 16-row tiles, odd sizes (rows that are not
16-byte aligned) among them.

Bar: spd(n) has a condition number under 6, so a backward stable Cholesky
solve errs by at most about 6 n^1.5 eps relative; the LU systems 1e-10 as the
other LU tests."""
import numpy as np
import pytest

import vba
from vba import abi

pytestmark = pytest.mark.gpu


def spd(n):
    rng = np.random.default_rng(n)
    a = rng.standard_normal((n, n))
    return a @ a.T + n * np.eye(n), rng.standard_normal(n)


@pytest.mark.parametrize("n", [257, 271, 272, 273, 319, 320, 321, 383, 385, 450, 511, 513, 640, 1025])
def test_cholesky(device, n):
    h, b = spd(n)
    h[np.triu_indices(n, 1)] = 1e3  # only the lower triangle is read
    st, x = device.dense_solve(h, b)
    assert st == abi.OK
    h = np.tril(h) + np.tril(h, -1).T
    ref = np.linalg.solve(h, b)
    assert np.abs(x - ref).max() <= 6 * n ** 1.5 * 2.3e-16 * np.abs(ref).max()


@pytest.mark.parametrize("n", [257, 320, 321])
@pytest.mark.parametrize("at", [0, 63, 64, -1])
def test_lu_fallback_on_a_bad_pivot(device, n, at):
    """A negative pivot in the first, a panel's last, the next panel's first
    or only in the last column."""
    h, b = spd(n)
    h[at, at] = -h[at, at]
    st, x = device.dense_solve(h, b)
    ref = np.linalg.solve(h, b)
    assert st == abi.OK
    assert np.abs(x - ref).max() <= 1e-10 * np.abs(ref).max()


@pytest.mark.parametrize("n", [257, 700])
def test_noalloc_equals_the_allocating_solve(device, n):
    h, b = spd(n)
    st, x = device.dense_solve(h, b)
    st2, x2 = device.dense_solve(h, b, noalloc=True)
    assert st == st2 == abi.OK
    assert np.array_equal(x, x2)
