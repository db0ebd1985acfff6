"""Eigensolves with little device memory: what the faster reductions keep beyond the
solve's own buffers (the matrix's copy behind the one-launch panels, the chase's
reflectors) never makes a solve fail that fits without.

The memory that a solve needs at least is found with those paths off; with them
on, the same limit has to do.
"""
import numpy as np
import pytest

from bse_amd import _abi

pytestmark = pytest.mark.gpu

N, STEP = 600, 64 * 1024


def _matrix():
    rng = np.random.default_rng(N)
    a = rng.normal(size=(N, N)) + 1j * rng.normal(size=(N, N))
    return 0.5 * (a + a.conj().T)


def _solve(env, limit, first, nvec, prec):
    """Two solves in one context, the second one under the limit."""
    a = _matrix()
    with pytest.MonkeyPatch.context() as mp:
        for k, v in env.items():
            mp.setenv(k, v)
        with _abi.Context(0) as c:
            if first:
                c.eigh_dense(a, prec, first)
            mp.setenv("BSE_MEMORY_LIMIT", str(limit))
            ev, z = c.eigh_dense(a, prec, nvec)
            return ev, z, c.reduction_info()


def _least(env, first, nvec, prec):
    lo, hi = 0, 1 << 30                   # lo fails, hi does
    while hi - lo > STEP:
        mid = (lo + hi) // 2
        try:
            _solve(env, mid, first, nvec, prec)
            hi = mid
        except _abi.BSEError as e:
            assert "hipMalloc" in str(e)
            lo = mid
    return hi


@pytest.mark.parametrize("two_stage", ["0", "1"])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("first", [0, 21])
def test_least_memory(two_stage, prec, first):
    plain = dict(BSE_TWO_STAGE="0", BSE_TRD_PANEL="0", BSE_AUTOTUNE="0")
    least = _least(plain, first, -1, prec)
    print(f"two_stage={two_stage} {prec} first={first}: {least} bytes", flush=True)
    env = dict(BSE_TWO_STAGE=two_stage, BSE_AUTOTUNE="0")
    a = _matrix()
    ref = np.linalg.eigvalsh(a)
    tol = (1e-12 if prec == "fp64" else 1e-5) * N ** 0.5
    routes = set()
    for limit in [least + f * N * N // 2 for f in (0, 2, 4, 8, 12, 16, 24)] + [1 << 31]:
        ev, z, info = _solve(env, limit, first, -1, prec)
        routes.add((info["reduction"], info["panels"]))
        assert np.abs(ev - ref).max() < tol * np.abs(ref).max()
        assert np.abs(a @ z - z * ev[None, :]).max() < 10 * tol * np.abs(ref).max()
    # from the plain path, without room, to the fast one
    assert ("one stage", "none") in routes
    assert (("two stages, reflectors kept", "none") if two_stage == "1" and prec == "fp64" else ("one stage", "ran")) in routes
