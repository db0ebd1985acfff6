"""Plans of the one-launch panels (csrc/panel_kernels.hip), on the host.

A workgroup may overwrite a message of two columns ago only because it waits for
the current column first, so no workgroup may find itself with nothing to wait
for.  Orders 64 k + 1, whose last column has a single row below it, are the ones
where that can happen.
"""
import ctypes

import pytest

from bse_amd import _abi


@pytest.mark.parametrize("workgroups", [256, 304, 64, 10])
def test_every_workgroup_waits_in_every_column(workgroups):
    lib = ctypes.CDLL(str(_abi.LIB_PATH))
    lib.bse_panel_unawaited.restype = ctypes.c_int64
    lib.bse_panel_first.restype = ctypes.c_int
    orders = [*range(2, 340), 385, 449, 641, 1407, 1409, 1473, 2050, 2049, 2817, 3009]
    taken = [n for n in orders if lib.bse_panel_first(n, workgroups) < n]
    assert len(taken) == len(orders)            # the last panels of every order run in one launch
    assert {n: lib.bse_panel_unawaited(n, workgroups) for n in taken} == dict.fromkeys(taken, 0)
