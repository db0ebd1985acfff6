"""Back-transform of the one-stage reduction on both sides of its rules: up to 16
vectors, from 17, and from order 256 four panels per pass (orders around a group
of 128 reflectors; a group of one column; few vectors and all).

Vectors of a unitary similarity transform in FP64: residual and orthogonality
to 1e-12 sqrt(n) of the norm.
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


@pytest.mark.parametrize("n", [40, 255, 256, 257, 258, 289, 385, 386, 520])
@pytest.mark.parametrize("nvec", [16, 17, 33, -1])
def test_vectors(ctx, n, nvec):
    print(f"back-transform n={n} nvec={nvec}", flush=True)
    rng = np.random.default_rng(n)
    a = rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))
    a = 0.5 * (a + a.conj().T)
    ev, z = ctx.eigh_dense(a, "fp64", nvec)
    k = z.shape[1]
    tol = 1e-12 * n ** 0.5
    assert np.abs(a @ z - z * ev[None, :k]).max() < tol * np.abs(ev).max()
    assert np.abs(z.conj().T @ z - np.eye(k)).max() < tol
