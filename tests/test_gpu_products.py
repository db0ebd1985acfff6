"""Matrix-free products and derivative products in both forms (tiles on matrix
cores, the general one) at the edges of their blocks of k-points and vectors.

All FP64 sums of at most N terms: 1e-12 of the matrix norm per entry for the
products, and 1e-10 of the largest entry between the two forms' gradients
(sums over N^2 products, eigenvectors of the same matrix).
"""
import numpy as np
import pytest

import bse_amd
from bse_amd import _abi
from bse_amd.lattice import KGrid

pytestmark = pytest.mark.gpu


def _context(form):
    mp = pytest.MonkeyPatch()
    if form:
        mp.setenv("BSE_ASSEMBLY", form)
    c = _abi.Context(0)
    mp.undo()
    return c


@pytest.fixture(scope="module")
def general():
    c = _context("valu")
    yield c
    c.close()


@pytest.fixture(scope="module")
def tiles():
    c = _context(None)
    yield c
    c.close()


PLAIN = [((1, 2), 1), ((31, 1), 2), ((4, 8), 16), ((3, 11), 17), ((5, 13), 31), ((8, 16), 32), ((7, 19), 33),
         ((25, 41), 16)]


@pytest.mark.parametrize("grid,k", PLAIN)
def test_general_product(general, grid, k):
    print(f"general product grid {grid} k={k}", flush=True)
    s = bse_amd.honeycomb_plain(6).with_params(grid=KGrid(*grid))
    general.set_system(s).build("fp64")
    H = general.matrix()
    rng = np.random.default_rng(k)
    x = rng.normal(size=(s.n_bse, k)) + 1j * rng.normal(size=(s.n_bse, k))
    y = general.apply(x)
    assert np.abs(y - H @ x).max() < 1e-12 * np.abs(H).sum(axis=1).max() * np.abs(x).max()


SYSTEMS = [(lambda: bse_amd.random_multiorbital(2), 16), (lambda: bse_amd.random_multiorbital(3), 17),
           (lambda: bse_amd.honeycomb_magnetic(4), 33), (lambda: bse_amd.honeycomb_magnetic(5), 1),
           (lambda: bse_amd.honeycomb_magnetic(3).with_params(nv=1, nc=2), 5),
           (lambda: bse_amd.random_multiorbital(3).with_params(nv=2, nc=3), 32)]
IDS = ["4v4c_2", "4v4c_3", "2v2c_4", "2v2c_5", "1v2c_3", "2v3c_3"]


@pytest.mark.parametrize("make,k", SYSTEMS, ids=IDS)
def test_gradients_of_both_forms(general, tiles, make, k):
    s = make()
    print(f"gradients {s.name} N={s.n_bse} k={k}", flush=True)
    om = s.omegas()[::16]
    out = []
    for c in (general, tiles):
        c.set_system(s).build("fp64").eigh(-1)
        eps = c.spectrum(om, s.eta)
        L, dL = c.grad_spectrum(om, s.eta, 0.5 * eps.imag)
        out.append((c.eigenvalues(), c.grad_energies(min(k, s.n_bse)), L, dL))
    (e, g, L, dL), (e2, g2, L2, dL2) = out
    # a derivative of one state is defined where its energy is not degenerate
    gap = np.minimum(np.diff(e, prepend=-np.inf), np.diff(e, append=np.inf))[:g.shape[0]]
    ok = gap > 1e-4 * np.abs(e).max()
    assert np.abs(e - e2).max() < 1e-12 * np.abs(e).max()
    assert np.abs(g - g2)[ok].max(initial=0.0) < 1e-10 * max(np.abs(g).max(), 1.0)
    assert abs(L - L2) < 1e-10 * L
    assert np.abs(dL - dL2).max() < 1e-9 * np.abs(dL).max()
