"""Band reduction of matrices whose panels are nearly dependent, from well
conditioned to numerically singular (where the Cholesky form gives way to the
tree of Householder factors).

The reduction is a unitary similarity transform, so eigenvalues are good to
1e-13 sqrt(n) of the norm however dependent the columns are.
"""
import numpy as np
import pytest

import bse_amd
from bse_amd import _abi
from bse_amd.lattice import KGrid

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx2():
    mp = pytest.MonkeyPatch()
    mp.setenv("BSE_TWO_STAGE", "1")
    c = _abi.Context(0)
    mp.undo()
    yield c
    c.close()


@pytest.mark.parametrize("grid", [(16, 32), (24, 24), (25, 41), (32, 33)])
def test_smooth_interaction(ctx2, grid):
    s = bse_amd.honeycomb_plain(6, gap=2.1).with_params(grid=KGrid(*grid))
    print(f"band panels, grid {grid}", flush=True)
    ctx2.set_system(s).build("fp64")
    ref = np.linalg.eigvalsh(ctx2.matrix())
    ctx2.eigh(4)
    assert np.abs(ctx2.eigenvalues() - ref).max() < 1e-13 * s.n_bse ** 0.5 * np.abs(ref).max()


@pytest.mark.parametrize("n,width", [(200, 3.0), (200, 6.0), (200, 10.0), (200, 16.0), (200, 40.0), (321, 16.0), (321, 40.0)])
def test_smooth_kernel(ctx2, n, width):
    i = np.arange(n)
    d = (i[:, None] - i[None, :]) / width
    a = np.exp(-d * d + 0.3j * d) + np.diag(0.5 + i / n)
    print(f"band panels n={n} width {width}", flush=True)
    ev, z = ctx2.eigh_dense(a, "fp64", 4)
    ref = np.linalg.eigvalsh(a)
    tol = 1e-13 * n ** 0.5 * np.abs(ref).max()
    assert np.abs(ev - ref).max() < tol
    assert np.abs(a @ z - z * ev[None, :4]).max() < 10 * tol


@pytest.mark.parametrize("one_stage", [False, True])
@pytest.mark.parametrize("n", [66, 70, 100])
def test_rank_one(ctx2, monkeypatch, n, one_stage):
    """Reflectors of what rounding leaves of a vanished column, and of that in
    turn: norms whose squares can no longer be formed."""
    if one_stage:
        monkeypatch.setenv("BSE_TWO_STAGE", "0")
        ctx2 = _abi.Context(0)
    a = np.ones((n, n), dtype=complex)
    ev, z = ctx2.eigh_dense(a, "fp64", 4)
    assert np.abs(ev - np.r_[np.zeros(n - 1), n]).max() < 1e-13 * n ** 1.5
    assert np.abs(a @ z - z * ev[None, :4]).max() < 1e-12 * n ** 1.5
    if one_stage:
        ctx2.close()
