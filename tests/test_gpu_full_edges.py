"""The full BSE's factorisation and triangular solves at the edges of their 64-row
tiles: order 2 N of one tile, one tile and a few rows, the change of sign
inside a tile (N not a multiple of 64) and at its edge, and one vector to all.

Checked against the oracle's Hamiltonian: H x = E x and x^H s3 x = 1 to the
tolerances of the other full-BSE tests (1e-10 of the largest energy, 1e-9).
"""
import numpy as np
import pytest

import bse_amd
from bse_amd import _abi
from bse_amd.lattice import KGrid
import bse_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = _abi.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("grid,k", [((1, 3), -1), ((5, 6), 1), ((4, 8), -1), ((3, 11), 32), ((7, 9), 17), ((8, 8), -1),
                                    ((5, 13), 65), ((8, 12), -1), ((12, 16), 64)])
def test_orders(ctx, grid, k):
    s = bse_amd.honeycomb_plain(6).with_params(grid=KGrid(*grid))
    n = s.n_bse
    print(f"full BSE order {2 * n}, {k} vectors", flush=True)
    p = O.problem_from_system(s)
    sol = O.solve_full(p)
    ctx.set_system(s).build_full().eigh_full(k)
    E = ctx.eigenvalues()
    k = n if k < 0 else k
    x = ctx.eigenvectors(k)
    scale = np.abs(sol["E"]).max()
    assert np.abs(E - sol["E"]).max() < 1e-10 * scale
    s3 = np.concatenate([np.ones(n), -np.ones(n)])
    assert np.abs(sol["H"] @ x - x * E[None, :k]).max() < 1e-10 * scale
    assert np.abs(x.conj().T @ (s3[:, None] * x) - np.eye(k)).max() < 1e-9
    eps = ctx.spectrum(p.omegas, p.eta)
    assert np.linalg.norm(eps - sol["eps"]) < 1e-9 * np.linalg.norm(sol["eps"] - 1.0)


@pytest.mark.parametrize("gap", [1e-100, 1e-300, 1e-309, 1e-315])
def test_tiny_pivots(ctx, gap):
    """Flat bands without interaction, whose M is the gap times the identity: a
    positive pivot factors whatever its size, subnormal ones included."""
    from dataclasses import replace
    s = bse_amd.honeycomb_plain(6)
    s = s.with_params(model=replace(s.model, h_r=np.zeros_like(s.model.h_r)), grid=KGrid(5, 7), scissor=gap,
                      direct_scale=0.0, exchange_scale=0.0)
    ctx.set_system(s).build_full().eigh_full(-1)
    # (a few units of the last place of a subnormal number)
    assert np.abs(ctx.eigenvalues() - gap).max() <= 1e-12 * gap + 2e-323
