"""States at given k: every padded order of the Jacobi kernel (1-2, 3-4, 5-8,
9-16 orbitals) at its edges, k counts around one wave's and one workgroup's
matrices, and exactly degenerate bands, against numpy in FP64.

Energies are those of a Hermitian matrix known to rounding: 1e-13 of its norm
(a few ulp per orbital); vectors through the residual, the orthonormality and
the fixed gauge.
"""
import numpy as np
import pytest

import bse_amd
from bse_amd import _abi
from bse_amd import tight_binding as tb

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = _abi.Context(0)
    yield c
    c.close()


def _check(model, k, e, u):
    h = model.hk(k)
    ref = np.linalg.eigvalsh(h)
    scale = np.abs(ref).max()
    n = model.norb
    assert np.abs(e - ref).max() < 1e-13 * scale
    z = np.swapaxes(u, 1, 2)
    assert np.abs(h @ z - z * e[:, None, :]).max() < 1e-13 * n * scale
    assert np.abs(np.swapaxes(z.conj(), 1, 2) @ z - np.eye(n)).max() < 1e-13 * n
    top = np.take_along_axis(z, np.argmax(np.abs(z), axis=1)[:, None, :], axis=1)
    assert np.all(top.real > 0) and np.abs(top.imag).max() < 1e-14


@pytest.mark.parametrize("norb", [1, 2, 3, 4, 5, 7, 8, 9, 12, 15, 16])
@pytest.mark.parametrize("nk", [1, 3, 17, 65, 259])
def test_every_order(ctx, norb, nk):
    print(f"states of {norb} orbitals at {nk} k", flush=True)
    model = tb.random_square(norb, seed=100 * norb + nk)
    k = np.random.default_rng(nk).uniform(-2, 2, size=(3, nk))
    _check(model, k, *ctx.tb_states_at(k, model=model))


@pytest.mark.parametrize("scale", [1e-140, 1e140])
def test_scale(ctx, scale):
    """Units in which the sums of squares that decide on convergence are still
    normal numbers, but nothing of higher order is."""
    m = tb.random_square(6, seed=3)
    from dataclasses import replace
    big = replace(m, h_r=m.h_r * scale)
    k = np.random.default_rng(0).uniform(-2, 2, size=(3, 9))
    e, u = ctx.tb_states_at(k, model=big)
    e1, _ = ctx.tb_states_at(k, model=m)
    assert np.abs(e / scale - e1).max() < 1e-12 * np.abs(e1).max()
    _check(m, k, e / scale, u)


@pytest.mark.parametrize("norb", [2, 6, 16])
def test_degenerate(ctx, norb):
    """A scalar Hamiltonian (all bands equal) and two equal blocks."""
    m = tb.random_square(norb // 2, seed=5)
    from dataclasses import replace
    h = np.kron(m.h_r, np.eye(2))
    two = replace(m, h_r=h, tau=np.repeat(m.tau, 2, axis=0))
    k = np.random.default_rng(1).uniform(-2, 2, size=(3, 5))
    e, u = ctx.tb_states_at(k, model=two)
    ref = np.linalg.eigvalsh(two.hk(k))
    assert np.abs(e - ref).max() < 1e-13 * np.abs(ref).max()
    z = np.swapaxes(u, 1, 2)
    assert np.abs(np.swapaxes(z.conj(), 1, 2) @ z - np.eye(norb)).max() < 1e-13 * norb
    flat = replace(two, h_r=np.zeros_like(h))
    e, u = ctx.tb_states_at(k, model=flat)
    assert np.all(e == 0.0)


@pytest.mark.parametrize("norb", [2, 3, 5, 16])
def test_phase_that_is_no_number(ctx, norb):
    """A k point so far out that its phase overflows: its own energies are NaN (no
    others in their place), those of the other points in its wave are right."""
    print(f"states of {norb} orbitals, one k point out of range", flush=True)
    model = tb.random_square(norb, seed=norb)
    k = np.random.default_rng(norb).uniform(-2, 2, size=(3, 9))
    k[:, 4] = [1.5e308, 1.5e308, 0.0]
    e, u = ctx.tb_states_at(k, model=model)
    assert np.all(np.isnan(e[4])) and np.all(np.isnan(u[4]).any(axis=-1))
    ok = np.delete(np.arange(9), 4)
    _check(model, k[:, ok], e[ok], u[ok])
