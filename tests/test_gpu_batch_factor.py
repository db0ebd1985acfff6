"""The batched sweep's product with the reduction's orthogonal factor, one
workgroup per vector: orders around its 32-reflector panels, the 512 rows of a
half workgroup and the 1024 of a whole one, against the single-system path.

FP64 on both sides, so they differ by rounding: 1e-10 of the largest
eigenvalue and of the spectrum's norm, as for the sweep's other results.
"""
import numpy as np
import pytest

import bse_amd
from bse_amd import _abi
from bse_amd.lattice import KGrid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grids", [[(1, 2), (1, 3), (31, 1), (4, 8), (3, 11), (2, 17)], [(7, 9), (8, 8), (5, 13)],
                                   [(16, 32), (27, 19), (32, 33), (41, 25)]])
@pytest.mark.parametrize("refine", [False, True])
def test_against_single(grids, refine):
    base = bse_amd.honeycomb_plain(6, gap=2.1)
    systems = [base.with_params(grid=KGrid(*g)) for g in grids]
    k = min(8, min(s.n_bse for s in systems))
    om = base.omegas()
    print(f"batch factor grids {grids} refine {refine}", flush=True)
    c = _abi.Context(0)
    c.batch_prepare(systems, precision="fp64", n_lowest=k, refine=refine, omegas=om, eta=base.eta)
    for _ in range(2):
        c.batch_run()
        ev, eps = c.batch_results()
    for i, s in enumerate(systems):
        c.set_system(s).build("fp64").eigh(k)
        ref, re = c.eigenvalues(), c.spectrum(om, base.eta)
        assert np.abs(ev[i] - ref[:k]).max() < 1e-10 * np.abs(ref).max()
        assert np.linalg.norm(eps[i] - re) < 1e-10 * np.linalg.norm(re)
    c.close()
