"""Many eigenvectors through the two-stage reduction: the bulge chase's
reflectors applied to the tridiagonal vectors, at the edges of their 32-sweep
blocks, of the 128 sweeps of a pass and of the column strips (16 columns).

Vectors of a unitary similarity transform in FP64: residual and orthogonality
to 1e-12 sqrt(n) of the norm, as for the other back-transforms.
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


def _herm(n):
    rng = np.random.default_rng(n)
    a = rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))
    return 0.5 * (a + a.conj().T)


KEPT = dict(reduction="two stages, reflectors kept", panels="none", chase="resident", reason=0)


@pytest.mark.parametrize("n", [21, 31, 32, 33, 34, 35, 63, 64, 65, 66, 97, 98, 128, 129, 130, 161, 258, 290, 545])
@pytest.mark.parametrize("nvec", [21, -1])
def test_orders(ctx2, n, nvec):
    print(f"many vectors n={n} nvec={nvec}", flush=True)
    a = _herm(n)
    ev, z = ctx2.eigh_dense(a, "fp64", nvec)
    assert ctx2.reduction_info() == KEPT
    ref = np.linalg.eigvalsh(a)
    k, tol = z.shape[1], 1e-12 * n ** 0.5
    assert np.abs(ev - ref).max() < tol * np.abs(ref).max()
    assert np.abs(a @ z - z * ev[None, :k]).max() < tol * np.abs(ref).max()
    assert np.abs(z.conj().T @ z - np.eye(k)).max() < tol


@pytest.mark.parametrize("n", [2, 3, 5])
def test_smallest(ctx2, n):
    print(f"many vectors n={n}", flush=True)
    a = _herm(n)
    ev, z = ctx2.eigh_dense(a, "fp64", -1)
    assert np.abs(a @ z - z * ev[None, :]).max() < 1e-13 * n * max(np.abs(ev).max(), 1.0)


def test_chosen_by_order():
    """An order beyond the line of the automatic choice, with 33 passes of 128
    sweeps and a last strip of two columns."""
    n = 4130
    print(f"many vectors n={n}", flush=True)
    a = _herm(n)
    with _abi.Context(0) as c:
        ev, z = c.eigh_dense(a, "fp64", -1)
        assert c.reduction_info() == KEPT
    pick = np.unique(np.r_[np.arange(0, n, 41), n - 33:n])
    zp = z[:, pick]
    tol = 1e-12 * n ** 0.5
    assert np.abs(a @ zp - zp * ev[None, pick]).max() < tol * np.abs(ev).max()
    g = z.conj().T @ zp
    g[pick, np.arange(pick.size)] -= 1.0
    assert np.abs(g).max() < tol


@pytest.mark.parametrize("make", [lambda: np.diag(np.arange(1.0, 71.0)), lambda: np.zeros((70, 70)),
                                  lambda: np.kron(np.eye(7), _herm(10)), lambda: np.ones((66, 66))],
                         ids=["diagonal", "zero", "blocks", "rank1"])
def test_vanishing_reflectors(ctx2, make):
    a = make().astype(complex)
    n = a.shape[0]
    ev, z = ctx2.eigh_dense(a, "fp64", -1)
    scale = max(np.abs(ev).max(), 1.0)
    assert np.abs(a @ z - z * ev[None, :]).max() < 1e-11 * scale
    assert np.abs(z.conj().T @ z - np.eye(n)).max() < 1e-10


@pytest.mark.parametrize("scale", [1e-129, 1e-140, 1e-147])
@pytest.mark.parametrize("n", [70, 200])
def test_small_scale(ctx2, n, scale):
    """The same matrix in small units, plain and graded over ten decades: columns
    of the chase whose squares leave the range of normal numbers count in full.
    Errors relative to the norm as in test_orders.  (Below 1e-135 the inverse
    iteration's own squares overflow, and at 1e-147 squares of the graded
    matrix's small entries underflow in the tridiagonal's split.)"""
    print(f"many vectors n={n} scale={scale}", flush=True)
    g = np.logspace(0, -5, n)
    for a in [_herm(n)] + ([_herm(n) * g[:, None] * g[None, :]] if scale > 1e-145 else []):
        ref = np.linalg.eigvalsh(a)
        ev, z = ctx2.eigh_dense(a * scale, "fp64", -1)
        ev = ev / scale
        tol = 1e-12 * n ** 0.5 * np.abs(ref).max()
        assert np.abs(ev - ref).max() < tol
        if scale > 1e-135:
            assert np.abs(a @ z - z * ev[None, :]).max() < tol
            assert np.abs(z.conj().T @ z - np.eye(n)).max() < 1e-12 * n ** 0.5


@pytest.mark.parametrize("scale", [1.0, 1e-129])
@pytest.mark.parametrize("nvec", [16, -1])
def test_numerically_rank_one(ctx2, nvec, scale):
    """What rounding leaves of a rank-one matrix is graded down to nothing."""
    n = 300
    print(f"rank one n={n} nvec={nvec} scale={scale}", flush=True)
    v = np.random.default_rng(5).uniform(0.5, 1.5, n)
    a = np.outer(v, v).astype(complex)
    ev, z = ctx2.eigh_dense(a * scale, "fp64", nvec)
    ev, k = ev / scale, z.shape[1]
    tol = 1e-12 * n ** 0.5
    assert np.abs(ev[:-1]).max() < tol * (v @ v) and abs(ev[-1] - v @ v) < tol * (v @ v)
    assert np.abs(a @ z - z * ev[None, :k]).max() < tol * (v @ v)
    assert np.abs(z.conj().T @ z - np.eye(k)).max() < tol


def test_without_the_resident_chase(ctx2, monkeypatch):
    """The general chase keeps no reflectors: the one-stage reduction serves."""
    a = _herm(200)
    monkeypatch.setenv("BSE_CHASE", "tasks")
    ev, z = ctx2.eigh_dense(a, "fp64", -1)
    assert ctx2.reduction_info()["reduction"] == "one stage"
    assert np.abs(a @ z - z * ev[None, :]).max() < 1e-11 * np.abs(ev).max()


@pytest.mark.parametrize("n", [21, 40, 200, 545])
def test_refused(ctx2, monkeypatch, n):
    """The chase leaves as if not resident: the matrix, by then a band matrix, is
    taken from its copy and reduced in one stage."""
    print(f"many vectors refused n={n}", flush=True)
    a = _herm(n)
    monkeypatch.setenv("BSE_RESIDENT_REFUSE", "chase")
    ev, z = ctx2.eigh_dense(a, "fp64", -1)
    assert ctx2.reduction_info() == dict(reduction="one stage", panels="ran", chase="one stage after refusal", reason=2)
    ref = np.linalg.eigvalsh(a)
    tol = 1e-12 * n ** 0.5
    assert np.abs(ev - ref).max() < tol * np.abs(ref).max()
    assert np.abs(a @ z - z * ev[None, :]).max() < tol * np.abs(ref).max()
    assert np.abs(z.conj().T @ z - np.eye(n)).max() < tol


@pytest.mark.parametrize("grid", [(5, 7), (8, 13), (11, 12)])
def test_problem_and_full_form(ctx2, grid):
    """With a dipole vector and an offset first vector (the full BSE's positive
    branch), against the one-stage reduction."""
    s = bse_amd.honeycomb_plain(6, gap=2.2).with_params(grid=KGrid(*grid))
    om = s.omegas()
    print(f"many vectors grid {grid}", flush=True)
    mp = pytest.MonkeyPatch()
    mp.setenv("BSE_TWO_STAGE", "0")
    c1 = _abi.Context(0)
    mp.undo()
    res = []
    for c in (c1, ctx2):
        c.set_system(s).build("fp64").eigh(-1)
        tda = (c.eigenvalues(), c.spectrum(om, s.eta))
        c.build_full().eigh_full(-1)
        x, E = c.eigenvectors(s.n_bse), c.eigenvalues()
        res.append(tda + (E, c.spectrum(om, s.eta)))
        s3 = np.concatenate([np.ones(s.n_bse), -np.ones(s.n_bse)])
        assert np.abs(x.conj().T @ (s3[:, None] * x) - np.eye(s.n_bse)).max() < 1e-8
    c1.close()
    for a, b in zip(*res):
        assert np.linalg.norm(a - b) < 1e-10 * np.linalg.norm(a)
