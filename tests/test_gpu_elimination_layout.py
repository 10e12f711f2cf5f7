"""vba_reduced_eliminate_row_major (what Device.reduced_eliminate calls) against
vba_reduced_eliminate (column-major blocks, nalgebra's layout): bit for bit, in
every block the caller passes or gets, at list lengths around the four terms
that a block's wave loads together. The struct's reserved word means nothing: a
caller that left it unset gets the same."""
import ctypes as C

import numpy as np
import pytest

import scenes
import vba
from vba import abi

pytestmark = pytest.mark.gpu


def column_major(device, el, reserved):
    view, keep = el.view()
    view.reserved = reserved
    runs = np.zeros((max(1, len(el.run_edges)), 36))
    m = el.coarse_aggregates()
    coarse = np.zeros((max(1, m * m), 36))
    st = device.lib.vba_reduced_eliminate(device.ctx, C.byref(view), runs.ctypes.data_as(abi.P64),
                                          coarse.ctypes.data_as(abi.P64))
    assert st == abi.OK, device.last_error()
    del keep
    runs = np.swapaxes(runs[:len(el.run_edges)].reshape(-1, 6, 6), -1, -2)
    return runs, np.swapaxes(coarse[:m * m].reshape(m, m, 6, 6), -1, -2) if m else None


@pytest.mark.parametrize("reserved", [0, 0xdeadbeef])
@pytest.mark.parametrize("nodes,points", [(5, 3), (8, 40), (60, 500), (150, 4000)])
def test_row_major_equals_column_major(device, nodes, points, reserved):
    el = scenes.elimination_problem(n=nodes, n_points=points, seed=nodes, extras=2, cluster=4, coarse_group=4)
    runs, coarse = column_major(device, el, reserved)
    got = device.reduced_eliminate(el)
    assert got is not None, device.last_error()
    assert np.array_equal(got[0], runs)
    assert np.array_equal(got[1], coarse)
