"""Work that a program asks of this package, as measurable cases.

Each case is one use of the Python entry points (``_abi.Context`` and
``autograd``) with its sizes: a band path, small and large Tamm-Dancoff
problems in every precision, one with its eigenvectors, the matrix-free
product, the full BSE, the parameter gradients, the batched sweep and the
dense eigensolver.  ``prepare`` makes what the program holds beforehand (a
context with the problem uploaded, or a recorded sweep), ``run`` is one pass,
``exact`` the same results from numpy in 64 bits.  Load it with the repository's root as the working
folder.
"""
from __future__ import annotations

import importlib.util
import math
import pathlib
import sys

import numpy as np


def _package():
    if "bse_amd" not in sys.modules:
        d = pathlib.Path.cwd() / "bethe-salpeter-equation_amd"
        spec = importlib.util.spec_from_file_location("bse_amd", d / "__init__.py",
                                                      submodule_search_locations=[str(d)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["bse_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["bse_amd"]


def _abi():
    _package()
    return importlib.import_module("bse_amd._abi")


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # the smallest call: energies and states of an 8-orbital model along a band path
        dict(name="band_path", kind="bands", norb=8, nk=257),
        # one small exciton problem from matrix to spectrum, as in a fit or a convergence scan: N = 144
        dict(name="tda_small", kind="tda", model="plain", n1=12, n2=12, precision="fp64", n_vec=-1),
        # the spinful magnetic honeycomb on its usual grid, the zheevd replacement: N = 3600
        dict(name="tda_magnetic", kind="tda", model="magnetic", n1=30, n2=30, precision="fp64", n_vec=-1),
        # every eigenvector in FP64 of a multi-band problem on an uneven grid: N = 8096
        dict(name="tda_all_vectors", kind="tda", model="random", n1=23, n2=22, precision="fp64", n_vec=-1),
        # the lowest excitons in FP64 with their vectors and the whole spectrum: N = 6720
        dict(name="tda_lowest", kind="tda", model="random", n1=21, n2=20, precision="fp64", n_vec=16),
        # mixed precision (compensated BF16 assembly, FP32 storage, FP64 refinement), ragged order: N = 4624
        dict(name="mixed_odd", kind="tda", model="random", n1=17, n2=17, precision="bf16x2", n_vec=16),
        # the package's headline workload: mixed precision at N = 20736
        dict(name="mixed_large", kind="tda", model="random", n1=36, n2=36, precision="bf16x2", n_vec=16),
        # matrix-free H X on a block of vectors, as a program's own iterative solver calls it: N = 10816
        dict(name="apply_block", kind="apply", n1=26, n2=26, k=16),
        # beyond Tamm-Dancoff: coupling block, structure-preserving solve, spectrum: order 2 x 1296
        dict(name="full_bse", kind="full", model="magnetic", n1=18, n2=18),
        # forward and backward of a parameter fit: energies, spectrum misfit and both gradients: N = 2304
        dict(name="gradients", kind="grad", n1=12, n2=12),
        # one launch of a recorded sweep of uneven honeycomb systems (FP32 storage, FP64 refinement)
        dict(name="sweep", kind="sweep", systems=64, lo=12, hi=40, grids=4),
        # a program's own Hermitian matrix on the host, every eigenpair (eig_sym): n = 777
        dict(name="dense", kind="dense", n=777, precision="fp64", n_vec=-1),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, lo, hi):
    """Two grid sides whose product is spread over the logarithm of [lo, hi]."""
    nk = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    n1 = max(2, int(round(math.sqrt(nk * rng.uniform(0.7, 1.4)))))
    n2 = max(2, int(nk / n1))
    return n1, n2


def draw(rng):
    kind = rng.choice(["bands", "tda", "tda", "tda", "apply", "full", "grad", "sweep", "dense"])
    if kind == "bands":
        return dict(kind=kind, norb=rng.choice([2, 3, 5, 8, 12, 16]), nk=_log_int(rng, 20, 4000))
    if kind == "tda":
        model = rng.choice(["plain", "magnetic", "random"])
        per_k = {"plain": 1, "magnetic": 4, "random": 16}[model]
        precision = rng.choice(["fp64", "fp64", "fp32", "bf16x2"])
        n_vec = 16 if precision != "fp64" else rng.choice([-1, 16])
        lo, hi = 100, 9000 if n_vec < 0 else 16000
        n1, n2 = _grid(rng, max(8, lo / per_k), min(hi / per_k, 3000))
        if n1 * n2 * per_k < 24:
            n1 = n2 = 5
        return dict(kind=kind, model=model, n1=n1, n2=n2, precision=precision, n_vec=n_vec)
    if kind == "apply":
        n1, n2 = _grid(rng, 16, 1200)
        return dict(kind=kind, n1=n1, n2=n2, k=rng.randint(1, 24))
    if kind == "full":
        model = rng.choice(["plain", "magnetic"])
        n1, n2 = _grid(rng, 36, 1600 if model == "plain" else 400)
        return dict(kind=kind, model=model, n1=n1, n2=n2)
    if kind == "grad":
        n1, n2 = _grid(rng, 9, 256)
        return dict(kind=kind, n1=n1, n2=n2)
    if kind == "sweep":
        lo = rng.randint(6, 20)
        return dict(kind=kind, systems=_log_int(rng, 4, 64), lo=lo, hi=rng.randint(lo + 2, 40),
                    grids=rng.randint(1, 1000))
    return dict(kind=kind, n=_log_int(rng, 24, 1500), precision=rng.choice(["fp64", "fp64", "fp32"]),
                n_vec=rng.choice([-1, 16]))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _rng(seed, tag):
    return np.random.Generator(np.random.PCG64([int(seed), tag]))


def _system(case, seed):
    """The exciton problem of a case: grid and bands from the case, the model's
    own parameters and the screening from the seed."""
    pkg = _package()
    tb = pkg.tight_binding
    r = _rng(seed, 1)
    model = case.get("model", "random")
    grid = pkg.lattice.KGrid(case["n1"], case["n2"])
    if model == "plain":
        return pkg.BSESystem(tb.honeycomb_two_band(gap=float(r.uniform(2.0, 4.0))), grid, n_occ=1, nv=1, nc=1,
                             r0=float(r.uniform(5, 30)), eps_env=float(r.uniform(1, 5)), g_cut=6.0)
    if model == "magnetic":
        return pkg.BSESystem(tb.honeycomb_spinful(gap=float(r.uniform(2.5, 4.0)),
                                                  exchange=float(r.uniform(0.05, 0.2)),
                                                  rashba=float(r.uniform(0.01, 0.05))),
                             grid, n_occ=2, nv=2, nc=2, r0=float(r.uniform(5, 30)),
                             eps_env=float(r.uniform(1, 5)), g_cut=6.0)
    # the repository's multi-orbital model, at the hopping scale and screening of one point of a scan
    m = tb.random_square(8).scaled(hopping_scale=float(r.uniform(0.9, 1.1)))
    return pkg.BSESystem(m, grid, n_occ=4, nv=4, nc=4, r0=float(r.uniform(10, 20)),
                         eps_env=float(r.uniform(1, 2)), g_cut=4.5)


def _size(case):
    per_k = {"plain": 1, "magnetic": 4, "random": 16}[case.get("model", "random")]
    return case["n1"] * case["n2"] * per_k


def _path_points(case, seed):
    pkg = _package()
    model = pkg.tight_binding.random_square(case["norb"], seed=int(_rng(seed, 2).integers(1, 1 << 30)))
    corner = [np.zeros(3), np.array([0.5, 0.0, 0.0]), np.array([0.5, 0.5, 0.0]), np.zeros(3)]
    n = case["nk"]
    parts = [n // 3, n // 3, n - 2 * (n // 3)]
    # the points keep off the symmetry points themselves (band path with open ends)
    k = np.concatenate([np.outer(a, 1 - t) + np.outer(b, t) for a, b, m in zip(corner, corner[1:], parts)
                        for t in [(np.arange(m) + 0.5) / m]], axis=1)
    return model, model.lattice.reciprocal @ k


def _block(case, seed):
    r = _rng(seed, 3)
    n = _size(case)
    x = r.standard_normal((n, case["k"])) + 1j * r.standard_normal((n, case["k"]))
    return np.asfortranarray(x / np.linalg.norm(x, axis=0))


def _matrix(case, seed):
    r = _rng(seed, 4)
    n = case["n"]
    a = r.standard_normal((n, n)) + 1j * r.standard_normal((n, n))
    return np.asfortranarray((a + a.conj().T) / (2 * math.sqrt(n)))


def _sweep_systems(case, seed):
    """Grids from the case (so that every seed asks for the same work), model
    parameters from the seed."""
    pkg = _package()
    g = np.random.Generator(np.random.PCG64(case["grids"]))
    sides = g.integers(case["lo"], case["hi"] + 1, size=(case["systems"], 2))
    r = _rng(seed, 5)
    return [pkg.BSESystem(pkg.tight_binding.honeycomb_two_band(gap=float(r.uniform(1.5, 4.0))),
                          pkg.lattice.KGrid(int(a), int(b)), n_occ=1, nv=1, nc=1, r0=float(r.uniform(5, 30)),
                          eps_env=float(r.uniform(1, 5)), g_cut=6.0) for a, b in sides]


def _theta(case, seed, base):
    """Parameters of one step of a fit: hopping scale, scissor, r0, eps, field."""
    r = _rng(seed, 6)
    return np.array([float(r.uniform(0.97, 1.03)), float(r.uniform(0.5, 1.0)), base.r0, base.eps_env,
                     float(r.uniform(-0.02, 0.02))])


def _target(case, seed, base):
    om = base.omegas()
    r = _rng(seed, 7)
    c, w, a = r.uniform(1, 5, 6), r.uniform(0.1, 0.6, 6), r.uniform(0.2, 2, 6)
    return np.sum(a[:, None] * np.exp(-0.5 * ((om - c[:, None]) / w[:, None]) ** 2), axis=0)


def _n_low(case):
    return min(8, _size(case))


def prepare(case, seed):
    abi = _abi()
    ctx = abi.Context(0)
    st = dict(case=case, ctx=ctx)
    kind = case["kind"]
    if kind == "bands":
        model, st["k"] = _path_points(case, seed)
        st["model"] = model
    elif kind in ("tda", "full"):
        st["system"] = _system(case, seed)
        st["omega"] = st["system"].omegas()
        ctx.set_system(st["system"])
    elif kind == "apply":
        ctx.set_system(_system(case, seed)).build("fp64")
        st["x"] = _block(case, seed)
    elif kind == "grad":
        st["system"] = _system(case, seed)
        st["theta"] = _theta(case, seed, st["system"])
        st["target"] = _target(case, seed, st["system"])
        st["omega"] = st["system"].omegas()
    elif kind == "sweep":
        systems = _sweep_systems(case, seed)
        ctx.batch_prepare(systems, precision="fp32", n_lowest=_sweep_low(case), refine=True,
                          omegas=systems[0].omegas(), eta=systems[0].eta)
    else:
        st["a"] = _matrix(case, seed)
    return st


def _sweep_low(case):
    return 16


def _aligned(z):
    """Eigenvectors with their free phase fixed: the largest component of each
    column real and positive, as a program stores them."""
    i = np.argmax(np.abs(z), axis=0)
    p = z[i, np.arange(z.shape[1])]
    return z * (p.conj() / np.abs(p))


def run(state):
    case, ctx = state["case"], state["ctx"]
    kind = case["kind"]
    if kind == "bands":
        return ctx.tb_states_at(state["k"], model=state["model"])
    if kind == "tda":
        low = min(case["n_vec"], _size(case))
        ctx.build(case["precision"]).eigh(low, refine=case["precision"] != "fp64")
        out = [ctx.eigenvalues(), ctx.spectrum(state["omega"], state["system"].eta)]
        # the honeycomb models have degenerate levels, whose vectors are a free
        # choice; the random model has none
        if low > 0 and case["model"] == "random":
            out.append(_aligned(ctx.eigenvectors(low)))
        return out
    if kind == "full":
        ctx.build_full().eigh_full(-1)
        return [ctx.eigenvalues(), ctx.spectrum(state["omega"], state["system"].eta)]
    if kind == "apply":
        return ctx.apply(state["x"])
    if kind == "grad":
        ag = importlib.import_module("bse_amd.autograd")
        s = ag.apply_theta(state["system"], state["theta"])
        ctx.set_system(s).build("fp64").eigh(-1)
        e = ctx.eigenvalues()
        de = ctx.grad_energies(_n_low(case))
        misfit, dl = ctx.grad_spectrum(state["omega"], s.eta, state["target"])
        return [e, de, misfit, dl]
    if kind == "sweep":
        ctx.batch_run()
        return list(ctx.batch_results())
    e, z = ctx.eigh_dense(state["a"], case["precision"], case["n_vec"] if case["n_vec"] < 0
                          else min(case["n_vec"], case["n"]))
    return [e, _aligned(z)]


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

N_OMEGA = 2048


def _eig_flops(n, nvec):
    """Hermitian eigenproblem with LAPACK's counts: reduction 16/3 n^3, and 8 n^2
    per vector transformed back."""
    return 16.0 / 3.0 * n ** 3 + 8.0 * n * n * nvec


def _assembly_flops(nk, b):
    norb, bands = {1: (2, 1), 4: (4, 2), 16: (8, 4)}[b]
    return 4.0 * nk * nk * (bands ** 2 * norb * (norb + bands ** 2) + b * b * norb)   # lower half


def work(case):
    kind = case["kind"]
    if kind == "bands":
        m, nk = case["norb"], case["nk"]
        return dict(bytes=nk * (24 + 8 * m + 16 * m * m), flops=nk * (8.0 * m * m * 9 + _eig_flops(m, m)))
    if kind == "dense":
        n, nv = case["n"], case["n"] if case["n_vec"] < 0 else min(case["n"], case["n_vec"])
        return dict(bytes=16.0 * n * n + 16.0 * n * nv + 8 * n, flops=_eig_flops(n, nv))
    if kind == "sweep":
        g = np.random.Generator(np.random.PCG64(case["grids"]))
        ns = g.integers(case["lo"], case["hi"] + 1, size=(case["systems"], 2)).prod(axis=1).astype(float)
        return dict(bytes=case["systems"] * 16.0 * N_OMEGA,
                    flops=float(np.sum(16.0 / 3.0 * ns ** 3 + 8.0 * N_OMEGA * ns)))
    n = _size(case)
    b = {"plain": 1, "magnetic": 4, "random": 16}[case.get("model", "random")]
    nk = n // b
    if kind == "apply":
        return dict(bytes=32.0 * n * case["k"], flops=2 * _assembly_flops(nk, b) / 2 + 8.0 * n * n * case["k"])
    spec = 8.0 * n * N_OMEGA
    if kind == "tda":
        nv = n if case["n_vec"] < 0 else min(n, case["n_vec"])
        return dict(bytes=8.0 * n + 24.0 * N_OMEGA + (16.0 * n * nv if 0 < case["n_vec"] else 0),
                    flops=_assembly_flops(nk, b) + _eig_flops(n, nv) + spec)
    if kind == "full":
        # two blocks, Cholesky and L^H s L of order 2n, and the eigenproblem of order 2n
        return dict(bytes=8.0 * n + 24.0 * N_OMEGA,
                    flops=2 * _assembly_flops(nk, b) + 2 * 4.0 / 3.0 * (2 * n) ** 3 + _eig_flops(2 * n, n) + spec)
    # gradients: the eigenproblem with all vectors and the three N x N x N_OMEGA products
    return dict(bytes=8.0 * n + 16.0 * N_OMEGA,
                flops=_assembly_flops(nk, b) * 6 + _eig_flops(n, n) + 24.0 * n * n * N_OMEGA)


def tolerance(case):
    """About four times the largest difference from ``exact`` over the ranges of
    ``draw``.  Eigenvectors and gradients carry the rounding of the matrix over
    a level spacing, the mixed-precision vectors their refinement's stopping
    rule (residual 1e-7 ||H||) over it."""
    kind = case["kind"]
    if kind in ("bands", "apply"):
        return {"rel": 2e-14 if kind == "bands" else 5e-15}
    if kind == "dense":
        return {"rel": 5e-13 if case["precision"] == "fp64" else 1e-5}
    if kind == "sweep":
        return {"rel": 5e-10}
    if kind == "tda" and case["precision"] == "fp64":
        return {"rel": 1e-12}
    if kind == "tda":
        # levels from FP32 storage; the random model's vectors are among the outputs
        return {"rel": 4e-5 if case["model"] == "random" else 6e-7}
    return {"rel": 2e-12 if kind == "grad" else 8e-15}


# ---------------------------------------------------------------------------
# The same results from numpy in 64 bits
# ---------------------------------------------------------------------------

CHARGE = 1602.176634 / 8.8541878176          # e^2 / eps_0 in eV Angstrom


def _phased(u):
    p = np.take_along_axis(u, np.argmax(np.abs(u), axis=1)[:, None, :], axis=1)
    return u * (p.conj() / np.abs(p))


class _Reference:
    """The q -> 0 exciton problem of a 2D system, dense, k fastest in the basis
    (c, v, k); coefficient arrays are [k, band, orbital]."""

    def __init__(self, s):
        m = s.model
        self.s, self.tau = s, np.asarray(m.tau)
        a = np.asarray(m.lattice.bravais)
        self.recip = 2 * np.pi * np.linalg.inv(a).T
        self.area = float(np.linalg.norm(np.cross(a[:, 0], a[:, 1])))
        self.volume = float(abs(np.linalg.det(a)))
        self.rvec = (a @ np.asarray(m.r_cryst, float).T).T
        self.h_r = np.asarray(m.h_r)
        self.onsite = np.all(np.asarray(m.r_cryst) == 0, axis=1)
        n1, n2 = s.grid.n1, s.grid.n2
        self.n1, self.n2, self.nk = n1, n2, n1 * n2
        self.i1, self.i2 = (x.ravel() for x in np.meshgrid(np.arange(n1), np.arange(n2), indexing="ij"))
        sh = tuple(s.grid.shift) + (0.0, 0.0)
        self.k = self.recip @ np.stack([(self.i1 + sh[0]) / n1, (self.i2 + sh[1]) / n2, np.zeros(self.nk)])
        half = [int(s.g_cut / np.linalg.norm(self.recip[:, d])) for d in (0, 1)]
        self.g = np.array([i * self.recip[:, 0] + j * self.recip[:, 1] for i in range(-half[0], half[0] + 1)
                           for j in range(-half[1], half[1] + 1)])
        self.nc, self.nv, self.n = s.nc, s.nv, s.nv * s.nc * self.nk
        self.fs = 1.0 if m.spinful else 2.0
        kq = self.k - np.asarray(s.q_opt, float)[:, None]
        self.ek, self.uk = self.states(self.k)
        self.eq, self.uq = self.states(kq)
        self.kq = kq
        self.cidx = s.n_occ + np.arange(s.nc)
        self.vidx = s.n_occ - 1 - np.arange(s.nv)
        self.C, self.V = self.pick(self.uk, self.cidx), self.pick(self.uq, self.vidx)

    def hamiltonian(self, k, keep=None):
        keep = slice(None) if keep is None else keep
        return np.einsum("rk,rlm->klm", np.exp(1j * (self.rvec[keep] @ k)), self.h_r[keep])

    def states(self, k):
        """Ascending bands, each state's largest component real and positive."""
        e, u = np.linalg.eigh(self.hamiltonian(k))
        return e, _phased(u)

    @staticmethod
    def pick(u, idx):
        return np.ascontiguousarray(np.swapaxes(u[:, :, idx], 1, 2))

    def phases(self, q):
        """e^{i q.(tau_i - tau_j)} over the last two axes."""
        p = np.exp(1j * (q @ self.tau.T))
        return p[..., :, None] * p[..., None, :].conj()

    def table(self, potential, origin):
        """sum_G potential(|Q + G|) e^{i(Q+G).(tau_i - tau_j)} on the grid differences."""
        d1, d2 = np.arange(1 - self.n1, self.n1), np.arange(1 - self.n2, self.n2)
        q = (d1[:, None, None] / self.n1) * self.recip[:, 0] + (d2[None, :, None] / self.n2) * self.recip[:, 1]
        out = 0
        for g in self.g:
            x = q + g
            r = np.linalg.norm(x, axis=-1)
            near = r < 1e-12
            w = np.where(near, origin, potential(np.where(near, 1.0, r)))
            out = out + w[..., None, None] * self.phases(x)
        return out

    def screened(self, wrt=None):
        """W_ij(Q), or its derivative with respect to r0 or eps_env."""
        r0, eps = self.s.r0, self.s.eps_env
        da = (2 * np.pi) ** 2 / (self.area * self.nk)
        rad = math.sqrt(da / math.pi)
        w0 = math.pi * CHARGE / eps * math.log1p(r0 * rad) / (r0 * da)
        if wrt is None:
            return self.table(lambda r: 0.5 * CHARGE / (eps * r * (1 + r0 * r)), w0)
        if wrt == "eps_env":
            return self.table(lambda r: -0.5 * CHARGE / (eps ** 2 * r * (1 + r0 * r)), -w0 / eps)
        return self.table(lambda r: -0.5 * CHARGE / (eps * (1 + r0 * r) ** 2),
                          math.pi * CHARGE / (eps * da) * (rad / (r0 * (1 + r0 * rad))
                                                           - math.log1p(r0 * rad) / r0 ** 2))

    def bare(self):
        g = np.delete(self.g, len(self.g) // 2, axis=0)
        return np.einsum("g,gij->ij", 0.5 * CHARGE / np.linalg.norm(g, axis=1), self.phases(g))

    def direct(self, w, lc, rc, lv, rv):
        """-(1/A Nk) sum_ij conj(lc_ck,i) rc_c'k',i W_ij(k - k') lv_vk,j conj(rv_v'k',j)."""
        nk = self.nk
        out = np.empty((lc.shape[1], lv.shape[1], nk, rc.shape[1], rv.shape[1], nk), complex)
        for k in range(nk):
            wk = w[self.i1[k] - self.i1 + self.n1 - 1, self.i2[k] - self.i2 + self.n2 - 1]
            x = (lc[k].conj()[None, :, None, :] * rc[:, None]) .reshape(nk, -1, wk.shape[1]) @ wk
            y = (lv[k][None, :, None, :] * rv.conj()[:, None]).reshape(nk, -1, wk.shape[1])
            z = x @ np.swapaxes(y, 1, 2)
            z = z.reshape(nk, lc.shape[1], rc.shape[1], lv.shape[1], rv.shape[1])
            out[:, :, k] = np.transpose(z, (1, 3, 2, 4, 0))
        return (-self.s.direct_scale / (self.area * nk)) * out

    def pairs(self, c, v):
        return np.einsum("kci,kvi->cvki", c.conj(), v).reshape(-1, c.shape[2])

    def differences(self, ec, ev):
        return np.transpose(ec[:, :, None] - ev[:, None, :], (1, 2, 0)).ravel()

    def matrix(self):
        h = self.direct(self.screened(), self.C, self.C, self.V, self.V).reshape(self.n, self.n)
        p = self.pairs(self.C, self.V)
        h += (self.s.exchange_scale * self.fs / (self.area * self.nk)) * (p @ self.bare() @ p.conj().T)
        h[np.diag_indices(self.n)] += self.differences(self.ek[:, self.cidx] + self.s.scissor,
                                                       self.eq[:, self.vidx])
        return h

    def coupling(self):
        b = self.direct(self.screened(), self.C, self.V, self.V, self.C)     # [c, v, k, v', c', k']
        b = np.transpose(b, (0, 1, 2, 4, 3, 5)).reshape(self.n, self.n)
        p = self.pairs(self.C, self.V)
        return b + (self.s.exchange_scale * self.fs / (self.area * self.nk)) * (p @ self.bare() @ p.T)

    def dipole(self, c, v):
        return 1j * np.einsum("kci,i,kvi->cvk", c.conj(), self.tau[:, 0], v).ravel()

    def prefactor(self):
        return CHARGE / (self.volume * self.nk)

    def spectrum(self, e, f2, om, eta, both=False):
        out = np.empty(om.size, complex)
        for lo in range(0, om.size, 256):
            w = om[lo:lo + 256, None] + 1j * eta
            g = 1 / (w - e)
            if both:
                g = g - 1 / (w + e)
            out[lo:lo + 256] = g @ f2
        return 1 - self.prefactor() * out

    def perturbed(self, k, e, u, dh):
        """First-order change of energies and states (parallel transport)."""
        m = np.swapaxes(u.conj(), 1, 2) @ dh @ u
        gap = e[:, None, :] - e[:, :, None]
        i = np.arange(e.shape[1])
        gap[:, i, i] = 1.0
        c = m / gap
        c[:, i, i] = 0.0
        return np.real(m[:, i, i]), u @ c

    def derivative(self, name):
        """(dH, drho) with respect to one parameter of the fit."""
        zero = np.zeros(self.n, complex)
        if name == "scissor":
            return np.eye(self.n, dtype=complex), zero
        if name in ("r0", "eps_env"):
            return self.direct(self.screened(name), self.C, self.C, self.V, self.V).reshape(self.n, self.n), zero
        if name == "hopping_scale":
            dk, dq = self.hamiltonian(self.k, ~self.onsite), self.hamiltonian(self.kq, ~self.onsite)
        else:
            m = self.tau.shape[0]
            sz = np.diag(np.where(np.arange(m) % 2 == 0, 1.0, -1.0)).astype(complex)
            dk = dq = np.broadcast_to(sz, (self.nk, m, m))
        dek, duk = self.perturbed(self.k, self.ek, self.uk, dk)
        deq, duq = self.perturbed(self.kq, self.eq, self.uq, dq)
        dC, dV = self.pick(duk, self.cidx), self.pick(duq, self.vidx)
        w, C, V = self.screened(), self.C, self.V
        # the two terms with a changed primed factor are the adjoints of the other two
        half = (self.direct(w, dC, C, V, V) + self.direct(w, C, C, dV, V)).reshape(self.n, self.n)
        p, dp = self.pairs(C, V), self.pairs(dC, V) + self.pairs(C, dV)
        half += (self.s.exchange_scale * self.fs / (self.area * self.nk)) * (dp @ self.bare() @ p.conj().T)
        dh = half + half.conj().T
        dh[np.diag_indices(self.n)] += self.differences(dek[:, self.cidx], deq[:, self.vidx])
        return dh, self.dipole(dC, V) + self.dipole(C, dV)


PARAMETERS = ("hopping_scale", "scissor", "r0", "eps_env", "exchange_field")


def _exact_gradients(case, seed):
    base = _system(case, seed)
    th = _theta(case, seed, base)
    model = base.model.scaled(hopping_scale=th[0], exchange_field=th[4])
    s = base.with_params(model=model, scissor=th[1], r0=th[2], eps_env=th[3])
    ref = _Reference(s)
    e, z = np.linalg.eigh(ref.matrix())
    rho = ref.dipole(ref.C, ref.V)
    f = z.T @ rho.conj()                                   # rho^H A_m
    om, target = base.omegas(), _target(case, seed, base)
    r = ref.spectrum(e, np.abs(f) ** 2, om, s.eta).imag - target
    g = 1 / (om[None, :] + 1j * s.eta - e[:, None])        # (N, n_omega)
    right = z @ (g * f.conj()[:, None])                    # (z - H)^-1 rho
    left = z.conj() @ (g * f[:, None])                     # rho^H (z - H)^-1, as columns
    low = _n_low(case)
    de, dl = np.zeros((low, 5)), np.zeros(5)
    mix = (right * r) @ left.T                             # B with tr(dH B) the matrix part of dL
    for t, name in enumerate(PARAMETERS):
        dh, drho = ref.derivative(name)
        de[:, t] = np.real(np.einsum("rm,rm->m", z[:, :low].conj(), dh @ z[:, :low]))
        val = np.sum(dh * mix.T) + np.sum(r * (drho.conj() @ right + drho @ left))
        dl[t] = -2 * ref.prefactor() * np.imag(val)
    return [e, de, float(np.sum(r * r)), dl]


def exact(case, seed):
    kind = case["kind"]
    if kind == "bands":
        model, k = _path_points(case, seed)
        r = np.asarray(model.lattice.bravais) @ np.asarray(model.r_cryst, float).T
        e, u = np.linalg.eigh(np.einsum("rk,rlm->klm", np.exp(1j * (r.T @ k)), model.h_r))
        return e, np.swapaxes(_phased(u), 1, 2)
    if kind == "dense":
        e, z = np.linalg.eigh(_matrix(case, seed))
        return [e, _aligned(z if case["n_vec"] < 0 else z[:, :min(case["n_vec"], case["n"])])]
    if kind == "sweep":
        if case["systems"] * (case["hi"] / 40.0) ** 6 > 70:
            return None
        low, lowest, eps = _sweep_low(case), [], []
        for s in _sweep_systems(case, seed):
            ref = _Reference(s)
            e, z = np.linalg.eigh(ref.matrix())
            f2 = np.abs(z.T @ ref.dipole(ref.C, ref.V).conj()) ** 2
            lowest.append(e[:low])
            eps.append(ref.spectrum(e, f2, s.omegas(), s.eta))
        return [np.array(lowest), np.array(eps)]
    n = _size(case)
    if kind == "grad":
        return _exact_gradients(case, seed) if n <= 2400 else None
    if kind == "apply":
        if n > 11000:
            return None
        ref = _Reference(_system(case, seed))
        return ref.matrix() @ _block(case, seed)
    if n > (1400 if kind == "full" else 4700):
        return None
    s = _system(case, seed)
    ref = _Reference(s)
    rho = ref.dipole(ref.C, ref.V)
    if kind == "tda":
        e, z = np.linalg.eigh(ref.matrix())
        out = [e, ref.spectrum(e, np.abs(z.T @ rho.conj()) ** 2, s.omegas(), s.eta)]
        low = min(case["n_vec"], n)
        if low > 0 and case["model"] == "random":
            out.append(_aligned(z[:, :low]))
        return out
    a, b = ref.matrix(), ref.coupling()
    chol = np.linalg.cholesky(np.block([[a, b], [b.conj(), a.conj()]]))
    sign = np.concatenate([np.ones(n), -np.ones(n)])
    e, y = np.linalg.eigh(chol.conj().T @ (sign[:, None] * chol))
    e, y = e[n:], y[:, n:]
    f = y.T @ np.linalg.solve(chol, np.concatenate([rho, -rho.conj()])).conj()
    return [e, ref.spectrum(e, e * np.abs(f) ** 2, s.omegas(), s.eta, both=True)]
