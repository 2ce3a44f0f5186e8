"""Spin-orbit plans of equal atoms run quaternion kernels (one vector per Kramers
pair): against the oracle, and against the complex kernels, which the same
material takes once an antisymmetric form factor of 1e-300 makes its atoms
unequal (H(k) changes by nothing that FP64 holds)."""
from __future__ import annotations

import copy

import numpy as np
import pytest

from ultimateepm_amd import api
from ultimateepm_amd.material import load

pytestmark = pytest.mark.gpu

# FP64: both reductions are backward stable, n eps ||H|| <= 400 * 2.2e-16 * 450 eV = 4e-11 eV
FP64_TOL = 1e-10
# precision form: second order in vectors good to ~3e-5, ~1e-9 eV each
MIXED_TOL = 1e-8


def _plan(ctx, sym, G, flags, nb, change=None):
    m = copy.deepcopy(load(sym))
    if change:
        change(m)
    return api.Plan(ctx, m, G, flags | api.SOC, nb)


def _general(m):
    m.V_A = (1e-300, 0.0, 0.0, 0.0)


def test_which_plans_are_quaternion(gpu_ctx):
    """The rule: no antisymmetric form factor, equal non-local and spin-orbit terms, spin-orbit on,
    and not the blocked reduction by request."""
    G = api.basis_vectors(6)
    ks = api.bz_sample(1, 8)

    def name(sym, flags, change=None, **cfg):
        p = _plan(gpu_ctx, sym, G, flags, 4, change)
        p.set_config(**cfg)
        p.set_timing(True)
        dk = api.DeviceArray.from_host(gpu_ctx, ks)
        de = api.DeviceArray(gpu_ctx, (len(ks), 4))
        p.solve_device(dk.ptr, len(ks), de.ptr)
        return list(p.last_timing())[1]

    for sym in ("Si", "Ge"):
        assert name(sym, api.NONLOCAL) == "tridiag_quaternion<f64>"
        assert name(sym, api.NONLOCAL | api.MIXED) == "tridiag_quaternion<f32>"
    general = "tridiag_reg_kernel<c128>"
    assert name("GaAs", api.NONLOCAL) == general
    assert name("Ge", api.NONLOCAL, tridiag=1) == general
    assert name("Ge", api.NONLOCAL, _general) == general
    assert name("Ge", api.NONLOCAL, lambda m: setattr(m.non_local, "A2_cation", 0.2)) == general
    assert name("Ge", 0, lambda m: setattr(m.spin_orbit, "alpha", 1.1)) == general
    assert name("Ge", 0, lambda m: setattr(m.spin_orbit, "period_anion", 3)) == general
    assert name("Ge", 0, lambda m: setattr(m.spin_orbit, "radial_extent_cation", 5.0)) == general


# numbers of plane waves at the edges of the grids (64 .. 192), of the back-transform's waves, and
# the first ones above the quaternion kernels' range; odd and even band counts
@pytest.mark.parametrize("ng,nb,mixed", [(1, 2, False), (1, 1, True), (2, 3, False), (17, 7, True), (64, 9, False),
                                         (65, 8, False), (64, 24, True), (65, 23, True), (96, 4, False), (97, 35, False),
                                         (128, 5, True), (129, 6, False), (129, 6, True), (144, 6, False), (144, 5, True),
                                         (145, 6, False), (145, 6, True), (160, 7, False), (161, 6, False),
                                         (161, 16, True), (192, 11, True), (193, 12, True)])
def test_quaternion_matches_general(gpu_ctx, ng, nb, mixed):
    print(f"case: quaternion against general, Ge, {ng} vectors, {nb} bands, mixed {mixed}", flush=True)
    G = np.ascontiguousarray(api.basis_vectors(14)[:ng])
    flags = api.NONLOCAL | api.GRADIENTS | (api.MIXED if mixed else 0)
    ks = api.bz_sample(ng, 5)
    e, v, g = _plan(gpu_ctx, "Ge", G, flags, nb).solve(ks, vectors=True)
    e2, v2, g2 = _plan(gpu_ctx, "Ge", G, flags, nb, _general).solve(ks, vectors=True)
    assert np.abs(e - e2).max() <= (MIXED_TOL if mixed else FP64_TOL)
    if ng <= (192 if mixed else 160):  # the quaternion kernels' range: each Kramers pair's level twice
        assert np.array_equal(e[:, 0:nb - nb % 2:2], e[:, 1::2])
    assert np.abs(np.einsum("kbi,kci->kbc", v.conj(), v) - np.eye(nb)).max() <= 1e-10
    # whole pairs more than 50 meV from the next level (the last one: unknown) span the same space, and
    # their mean gradient is the same; first order in the vectors' error over the gap
    tol = 1e-3 if mixed else 1e-8
    scale = np.abs(g2).max()
    for i in range(len(ks)):
        for b in range(0, nb - 1, 2):
            near = [abs(e[i, b] - e[i, c]) for c in (b - 2, b + 2) if 0 <= c < nb]
            if (b + 2 >= nb and nb < 2 * ng) or min(near, default=1.0) < 0.05:
                continue
            s = np.linalg.svd(v[i, b:b + 2].conj() @ v2[i, b:b + 2].T, compute_uv=False)
            assert np.abs(s - 1.0).max() <= tol * tol + 1e-11, (i, b)
            assert np.abs(g[i, b:b + 2].mean(axis=0) - g2[i, b:b + 2].mean(axis=0)).max() <= tol * scale


@pytest.mark.parametrize("sym,n,flags,nb", [("Ge", 10, api.VECTORS, 16), ("Ge", 8, api.VECTORS | api.MIXED, 15),
                                            ("Si", 9, 0, 8), ("Ge", 12, api.MIXED, 20)])
def test_quaternion_matches_the_oracle(gpu_ctx, oracle, sym, n, flags, nb):
    print(f"case: quaternion against the oracle, {sym} n={n} flags {flags}", flush=True)
    G = api.basis_vectors(n)
    ks = np.vstack([[0.0, 0.0, 0.0], [1.0, 0.0, 0.0], [0.5, 0.5, 0.5], api.bz_sample(4, 5)])
    e, v, _ = _plan(gpu_ctx, sym, G, flags | api.NONLOCAL, nb).solve(ks)
    w, _, _ = oracle.solve(load(sym), G, api.NONLOCAL | api.SOC, nb, ks, nthreads=8)
    noise = max(6.0 * 2.0e-6 / oracle.min_norm_gap(load(sym), G, k) for k in ks)  # the oracle's square-well integrals
    assert np.abs(e - w).max() <= max(1e-4 if flags & api.MIXED else 1e-9, noise if sym == "Si" else 0.0)
    if v is not None:
        res = 1e-3 if flags & api.MIXED else 1e-8
        for i, k in enumerate(ks):
            H = oracle.assemble(load(sym), G, k, nl=True, soc=True)
            X = v[i].T
            assert np.linalg.norm(H @ X - X * e[i], axis=0).max() <= res
            assert np.abs(X.conj().T @ X - np.eye(nb)).max() <= 1e-10
