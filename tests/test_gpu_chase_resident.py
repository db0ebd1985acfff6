"""Bulge chase with the band resident in LDS against the form with one wave
per sweep, at the edges of its 32-row blocks (one block, a block of one row,
full blocks, one row more), and the vector y it carries.

Both forms are unitary similarity transforms of the same band matrix, so
their eigenvalues differ by rounding alone: 1e-13 ||A|| sqrt(n) (a few ulp of
the norm for each of the O(sqrt(n)) statistically independent sweeps).
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


RESIDENT = dict(reduction="two stages", panels="none", chase="resident", reason=0)


@pytest.mark.parametrize("n", [2, 3, 31, 32, 33, 34, 35, 63, 64, 65, 66, 67, 97, 98, 129, 258, 290, 545])
def test_same_eigenvalues(ctx2, monkeypatch, n):
    print(f"resident chase n={n}", flush=True)
    rng = np.random.default_rng(n)
    a = rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))
    a = 0.5 * (a + a.conj().T)
    ev, _ = ctx2.eigh_dense(a, "fp64", 0)
    assert ctx2.reduction_info() == RESIDENT
    monkeypatch.setenv("BSE_CHASE", "tasks")
    ev2, _ = ctx2.eigh_dense(a, "fp64", 0)
    assert ctx2.reduction_info() == dict(RESIDENT, chase="tasks")
    ref = np.linalg.eigvalsh(a)
    tol = 1e-13 * np.abs(ref).max() * n ** 0.5
    assert np.abs(ev - ev2).max() < tol
    assert np.abs(ev - ref).max() < 10 * tol


@pytest.mark.parametrize("grid", [(1, 2), (3, 11), (2, 17), (5, 13), (6, 11), (8, 12), (10, 13), (14, 23)])
def test_same_oscillator_strengths(ctx2, monkeypatch, grid):
    """Q^H rho: the spectrum is the resolvent on rho, so it does not see the
    free choices of the two forms."""
    s = bse_amd.honeycomb_plain(6).with_params(grid=KGrid(*grid))
    om = s.omegas()
    print(f"resident chase y, grid {grid}", flush=True)
    ctx2.set_system(s).build("fp64").eigh(1)
    assert ctx2.reduction_info() == RESIDENT
    e, eps = ctx2.eigenvalues(), ctx2.spectrum(om, s.eta)
    monkeypatch.setenv("BSE_CHASE", "tasks")
    ctx2.set_system(s).build("fp64").eigh(1)
    e2, eps2 = ctx2.eigenvalues(), ctx2.spectrum(om, s.eta)
    assert np.abs(e - e2).max() < 1e-12 * np.abs(e2).max()
    assert np.linalg.norm(eps - eps2) < 1e-11 * np.linalg.norm(eps2 - 1)


@pytest.mark.parametrize("grid", [(1, 2), (5, 13), (14, 23)])
def test_refused(ctx2, monkeypatch, grid):
    """The resident chase leaves as if not resident, with the band and y untouched:
    one wave per sweep serves, with its own results bit for bit."""
    s = bse_amd.honeycomb_plain(6).with_params(grid=KGrid(*grid))
    om = s.omegas()
    print(f"resident chase refused, grid {grid}", flush=True)
    res = []
    for name, value, chase in (("BSE_RESIDENT_REFUSE", "chase", "tasks after refusal"),
                               ("BSE_CHASE", "tasks", "tasks")):
        with pytest.MonkeyPatch.context() as mp:
            mp.setenv(name, value)
            ctx2.set_system(s).build("fp64").eigh(1)
        info = ctx2.reduction_info()
        assert info["chase"] == chase and info["reason"] == (2 if "after" in chase else 0)
        res.append((ctx2.eigenvalues(), ctx2.spectrum(om, s.eta), ctx2.eigenvectors(1)))
    for a, b in zip(*res):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("two_stage", ["0", "1"])
def test_two_contexts_at_once(monkeypatch, two_stage):
    """Contexts on two threads launch resident kernels (the chase, the one-stage
    panels) on one device: the launches follow one another, and each result is
    its own.  Without the run-time search over kernels, whose choice follows
    the load and changes the order of sums, they are the same bit for bit."""
    import threading
    monkeypatch.setenv("BSE_TWO_STAGE", two_stage)
    monkeypatch.setenv("BSE_AUTOTUNE", "0")
    systems = [bse_amd.honeycomb_plain(24), bse_amd.honeycomb_plain(25, gap=2.0)]
    out = [None, None]

    def work(i):
        c = _abi.Context(0)
        try:
            res = []
            for _ in range(3):
                c.set_system(systems[i]).build("fp64").eigh(4)
                res.append(c.eigenvalues())
            out[i] = res
        finally:
            c.close()

    th = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join(timeout=60)
    for i in range(2):
        c = _abi.Context(0)
        c.set_system(systems[i]).build("fp64").eigh(4)
        ref = c.eigenvalues()
        c.close()
        for r in out[i]:
            assert np.array_equal(r, ref), np.abs(r - ref).max()
