"""Plans whose H(k) is real symmetric (equal atoms, no spin-orbit) run real
kernels: against the oracle, and against the complex kernels, which the same
material takes once an antisymmetric form factor of 1e-300 makes its atoms
unequal (H(k) changes by nothing that FP64 holds)."""
from __future__ import annotations

import copy

import numpy as np
import pytest

from ultimateepm_amd import api
from ultimateepm_amd.material import load

pytestmark = pytest.mark.gpu

# FP64: both reductions are backward stable, n eps ||H|| <= 448 * 2.2e-16 * 450 eV = 4.5e-11 eV
FP64_TOL = 1e-10
# precision form: Ritz values are second order in vectors good to ~3e-5 (FP32 rounding of
# ||H|| over the gap to the bands outside the Ritz space): ~1e-9 eV each
MIXED_TOL = 1e-8


def _plan(ctx, sym, G, flags, nb, general=False):
    m = load(sym)
    if general:
        m = copy.deepcopy(m)
        m.V_A = (1e-300, 0.0, 0.0, 0.0)
    return api.Plan(ctx, m, G, flags, nb)


def _reduction(plan, ks):
    plan.set_timing(True)
    dk = api.DeviceArray.from_host(plan._ctx, ks)
    de = api.DeviceArray(plan._ctx, (len(ks), plan.nb))
    plan.solve_device(dk.ptr, len(ks), de.ptr)
    names = list(plan.last_timing())
    plan.set_timing(False)
    return names[1]


def test_which_plans_are_real(gpu_ctx):
    """The rule: no antisymmetric form factor, equal non-local terms, no spin-orbit, and
    not the blocked reduction by request."""
    G = api.basis_vectors(6)
    ks = api.bz_sample(1, 8)

    def name(sym, flags, change=None, **cfg):
        m = copy.deepcopy(load(sym))
        if change:
            change(m)
        p = api.Plan(gpu_ctx, m, G, flags, 4)
        p._ctx = gpu_ctx
        p.set_config(**cfg)
        return _reduction(p, ks)

    for sym in ("Si", "Ge", "Sn"):
        assert name(sym, api.NONLOCAL) == "tridiag_real<f64>"
        assert name(sym, api.NONLOCAL | api.MIXED) == "tridiag_real<f32>"
    assert name("GaAs", api.NONLOCAL) == "tridiag_reg_kernel<c128>"
    assert not name("Ge", api.NONLOCAL | api.SOC).startswith("tridiag_real")
    assert name("Si", api.NONLOCAL, tridiag=1) == "tridiag_reg_kernel<c128>"
    assert name("Si", 0, lambda m: setattr(m, "V_A", (0.0, 1e-9, 0.0, 0.0))) == "tridiag_reg_kernel<c128>"
    for field in ("alpha_0_anion", "beta_0_cation", "R0_anion"):
        unequal = lambda m: setattr(m.non_local, field, 0.9 * getattr(m.non_local, field))  # noqa: E731
        assert name("Si", api.NONLOCAL, unequal) == "tridiag_reg_kernel<c128>"
        assert name("Si", 0, unequal) == "tridiag_real<f64>"  # local: the non-local terms do not enter


@pytest.mark.parametrize("sym", ["Si", "Ge", "Sn"])
def test_imaginary_parts_are_exactly_zero(gpu_ctx, sym):
    G = api.basis_vectors(9)
    ks = np.vstack([[0.0, 0.0, 0.0], [0.5, 0.5, 0.5], api.bz_sample(2, 6)])
    for flags in (0, api.NONLOCAL):
        p = api.Plan(gpu_ctx, load(sym), G, flags, 4)
        dk = api.DeviceArray.from_host(gpu_ctx, ks)
        dH = api.DeviceArray(gpu_ctx, (len(ks), p.dim, p.dim, 2))
        p.assemble_device(dk.ptr, len(ks), dH.ptr)
        gpu_ctx.synchronize()
        assert np.all(dH.numpy()[..., 1] == 0.0)


# sizes at the edges of the stages (row kernels 64 / 96 / 128, grids 160 .. 448), and the
# first sizes above the real kernels' range
@pytest.mark.parametrize("ng,mixed", [(1, False), (2, True), (17, False), (64, False), (65, False), (64, True), (65, True),
                                      (96, True), (97, False), (128, False), (129, True), (160, False), (161, True),
                                      (192, False), (193, False), (224, True), (225, False), (257, True), (288, False),
                                      (289, False), (320, False), (321, False), (289, True), (385, True), (448, True),
                                      (449, True)])
def test_real_matches_general(gpu_ctx, ng, mixed):
    print(f"case: real against general, Si, {ng} vectors, mixed {mixed}", flush=True)
    G = np.ascontiguousarray(api.basis_vectors(22)[:ng])
    nb = min(ng, 17 if ng % 2 else 6)
    flags = api.NONLOCAL | api.GRADIENTS | (api.MIXED if mixed else 0)
    ks = api.bz_sample(ng, 5)
    e, v, g = _plan(gpu_ctx, "Si", G, flags, nb).solve(ks, vectors=True)
    e2, v2, g2 = _plan(gpu_ctx, "Si", G, flags, nb, general=True).solve(ks, vectors=True)
    assert np.abs(e - e2).max() <= (MIXED_TOL if mixed else FP64_TOL)
    assert np.all(v.imag == 0.0)
    assert np.abs(v @ v.transpose(0, 2, 1) - np.eye(nb)).max() <= 1e-10
    # bands apart from their neighbours (and from band nb, unknown here): the same vectors up to
    # phase, and gradients; first order in the vectors' error over the gap
    gap = np.full(e.shape, np.inf)
    gap[:, 1:] = np.minimum(gap[:, 1:], np.diff(e, axis=1))
    gap[:, :-1] = np.minimum(gap[:, :-1], np.diff(e, axis=1))
    ok = gap > 0.05
    ok[:, -1] = ng == nb
    tol = 1e-3 if mixed else 1e-8  # 1e-10 eV (FP32: 3e-5) over 0.05 eV
    over = np.abs(np.einsum("kbi,kbi->kb", v.conj(), v2))
    assert np.abs(over - 1.0)[ok].max(initial=0.0) <= tol * tol + 1e-12
    scale = np.abs(g2).max()
    assert np.abs(g - g2)[ok].max(initial=0.0) <= tol * scale


@pytest.mark.parametrize("sym,n,flags,nb", [("Si", 12, api.NONLOCAL | api.VECTORS, 12), ("Ge", 9, api.NONLOCAL, 16),
                                            ("Sn", 8, api.NONLOCAL | api.MIXED, 24), ("Si", 16, 0, 8),
                                            ("Si", 16, api.MIXED, 8)])
def test_real_matches_the_oracle(gpu_ctx, oracle, sym, n, flags, nb):
    print(f"case: real against the oracle, {sym} n={n} flags {flags}", flush=True)
    G = api.basis_vectors(n)
    # high-symmetry points (degenerate levels) and general ones
    ks = np.vstack([[0.0, 0.0, 0.0], [1.0, 0.0, 0.0], [0.5, 0.5, 0.5], api.bz_sample(4, 9)])
    p = _plan(gpu_ctx, sym, G, flags, nb)
    e, v, _ = p.solve(ks)
    w, _, _ = oracle.solve(load(sym), G, flags & api.NONLOCAL, nb, ks, nthreads=8)
    # the oracle's radial integrals lose digits where two |k + G| nearly meet
    tol = max(1e-4 if flags & api.MIXED else 1e-9, *[6.0 * 2.0e-6 / oracle.min_norm_gap(load(sym), G, k) for k in ks]) \
        if flags & api.NONLOCAL else (1e-4 if flags & api.MIXED else 1e-9)
    assert np.abs(e - w).max() <= tol
    if v is not None:
        for i, k in enumerate(ks):
            H = oracle.assemble(load(sym), G, k, nl=bool(flags & api.NONLOCAL), soc=False)
            X = v[i].T
            assert np.linalg.norm(H @ X - X * e[i], axis=0).max() <= 1e-8
            assert np.abs(X.conj().T @ X - np.eye(nb)).max() <= 1e-10
