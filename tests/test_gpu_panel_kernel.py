"""One-stage reduction with a panel per launch (resident workgroups) against
LAPACK and against the per-column launches: orders around the 32-column panels
and 64-row tiles, the change from one tile per workgroup (up to 22
tile rows) to two, three and four, both storage types, matrices whose reflectors
vanish, and a panel that is refused.

Eigenvalues of a unitary similarity transform computed in FP64 are good to a
modest multiple of eps ||A||: 1e-13 sqrt(n) of the norm, as for the per-column
launches; FP32 storage rounds the matrix once per panel (6e-8 of the norm each).
"""
import numpy as np
import pytest

from bse_amd import _abi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    mp = pytest.MonkeyPatch()
    mp.setenv("BSE_TWO_STAGE", "0")
    c = _abi.Context(0)
    mp.undo()
    yield c
    c.close()


def _herm(n, seed):
    rng = np.random.default_rng(seed)
    a = rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))
    return 0.5 * (a + a.conj().T)


RAN = dict(reduction="one stage", panels="ran", chase="none", reason=0)


def _check(a, ev, z, ref, tol):
    n = a.shape[0]
    scale = max(np.abs(ref).max(), 1e-300)
    assert np.abs(ev - ref).max() < tol * scale * n ** 0.5
    assert np.abs(a @ z - z * ev[None, :]).max() < 10 * tol * scale * n ** 0.5
    assert np.abs(z.conj().T @ z - np.eye(n)).max() < 1e-10


@pytest.mark.parametrize("n", [2, 3, 31, 32, 33, 34, 63, 64, 65, 66, 95, 97, 127, 128, 129, 130, 193, 257, 333, 600])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_orders(ctx, n, prec):
    print(f"panel kernel n={n} {prec}", flush=True)
    a = _herm(n, n)
    ev, z = ctx.eigh_dense(a, prec)
    assert ctx.reduction_info() == RAN
    _check(a, ev, z, np.linalg.eigvalsh(a), 1e-13 if prec == "fp64" else 2e-6)


@pytest.mark.parametrize("n", [1407, 1409, 1441, 1500, 2050, 2500, 2830])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_against_column_launches(ctx, monkeypatch, n, prec):
    print(f"panel kernel n={n} {prec}", flush=True)
    a = _herm(n, n)
    ev, z = ctx.eigh_dense(a, prec, 8)
    assert ctx.reduction_info() == RAN
    monkeypatch.setenv("BSE_TRD_PANEL", "0")
    ev2, _ = ctx.eigh_dense(a, prec, 8)
    assert ctx.reduction_info()["panels"] == "none"
    scale = np.abs(ev2).max()
    assert np.abs(ev - ev2).max() < (1e-13 if prec == "fp64" else 2e-7) * scale * n ** 0.5
    tol = 1e-12 if prec == "fp64" else 1e-5
    assert np.abs(a @ z - z * ev[None, :8]).max() < tol * scale * n ** 0.5


@pytest.mark.parametrize("n", [2, 70, 333, 1500, 2960])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_refused(ctx, monkeypatch, n, prec):
    """The last panel leaves as if not resident: the matrix, changed by the panels
    before it, is taken from its copy and reduced by columns."""
    print(f"panel kernel refused n={n} {prec}", flush=True)
    a = _herm(n, n)
    monkeypatch.setenv("BSE_RESIDENT_REFUSE", "panel")
    ev, z = ctx.eigh_dense(a, prec, min(n, 8))
    assert ctx.reduction_info() == dict(RAN, panels="repeated", reason=2)
    monkeypatch.delenv("BSE_RESIDENT_REFUSE")
    monkeypatch.setenv("BSE_TRD_PANEL", "0")
    ev2, z2 = ctx.eigh_dense(a, prec, min(n, 8))
    assert np.array_equal(ev, ev2) and np.array_equal(z, z2)      # the same launches


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_vanishing_reflectors(ctx, prec):
    tol = 1e-13 if prec == "fp64" else 2e-6
    n = 150
    d = np.diag(np.linspace(-3.0, 5.0, n)).astype(complex)
    ev, z = ctx.eigh_dense(d, prec)
    _check(d, ev, z, np.linspace(-3.0, 5.0, n), tol)
    t = np.zeros((n, n), complex)
    i = np.arange(n - 1)
    t[i + 1, i] = 1j
    t[i, i + 1] = -1j                    # tridiagonal, imaginary: a phase per reflector
    ev, z = ctx.eigh_dense(t, prec)
    _check(t, ev, z, np.linalg.eigvalsh(t), tol)
    b = np.zeros((n, n), complex)
    b[:70, :70] = _herm(70, 1)
    b[70:, 70:] = _herm(n - 70, 2)       # two blocks: a column that is zero below its diagonal
    ev, z = ctx.eigh_dense(b, prec)
    _check(b, ev, z, np.linalg.eigvalsh(b), tol)


@pytest.mark.parametrize("scale", [1e-140, 1e-129, 1e-105, 1e-60, 1e60, 1e101, 1e120, 1e140])
@pytest.mark.parametrize("n", [70, 200, 1500])
def test_scale(ctx, n, scale):
    """The same matrix in other units: x^H A x is of third order in them.  (Below
    1e-135 the inverse iteration's own squares overflow.)"""
    print(f"panel kernel n={n} scale={scale}", flush=True)
    a = _herm(n, n)
    ref = np.linalg.eigvalsh(a)
    ev, z = ctx.eigh_dense(a * scale, "fp64", 16)
    ev = ev / scale
    assert np.abs(ev - ref).max() < 1e-13 * np.abs(ref).max() * n ** 0.5
    if scale > 1e-135:
        assert np.abs(a @ z - z * ev[None, :16]).max() < 1e-12 * np.abs(ref).max() * n ** 0.5
        assert np.abs(z.conj().T @ z - np.eye(16)).max() < 1e-10


def test_two_contexts_at_once():
    import threading
    mats = [_herm(500, 11), _herm(460, 12)]
    out = [None, None]

    def work(i):
        with _abi.Context(0) as c:
            out[i] = [c.eigh_dense(mats[i], "fp64")[0] for _ in range(3)]

    th = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join(timeout=60)
    for i in range(2):
        with _abi.Context(0) as c:
            ref = c.eigh_dense(mats[i], "fp64")[0]
        for r in out[i]:
            assert np.array_equal(r, ref)
