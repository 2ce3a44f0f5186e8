"""Bases whose reciprocal vectors are far from the origin or far from each other:
H(k) depends on k + G and on G - G' alone, for every int32 G."""
from __future__ import annotations

import numpy as np
import pytest

from ultimateepm_amd import api
from ultimateepm_amd.material import load

pytestmark = pytest.mark.gpu


def _assemble(ctx, mat, G, flags, ks):
    p = api.Plan(ctx, mat, np.ascontiguousarray(G, dtype=np.int32), flags, 4)
    dk = api.DeviceArray.from_host(ctx, np.ascontiguousarray(ks))
    dH = api.DeviceArray(ctx, (len(ks), p.dim, p.dim, 2))
    p.assemble_device(dk.ptr, len(ks), dH.ptr)
    ctx.synchronize()
    H = dH.numpy()
    p.close()
    return (H[..., 0] + 1j * H[..., 1]).transpose(0, 2, 1)  # column-major on the device


def _kpoints(nk):
    """Points whose coordinates are multiples of 2^-20, so that k - s and k - s + G are exact."""
    return np.round(api.bz_sample(17, nk) * 2.0**20) / 2.0**20


@pytest.mark.parametrize("sym,flags", [("Si", api.NONLOCAL), ("GaAs", api.NONLOCAL), ("InP", api.NONLOCAL),
                                       ("Ge", api.NONLOCAL | api.SOC), ("GaAs", api.NONLOCAL | api.SOC)])
@pytest.mark.parametrize("shift", [(600, -700, 0), (511, 512, -513), (-513, 0, 1025), (100003, -200001, 70000)])
def test_shifted_basis(gpu_ctx, oracle, sym, flags, shift):
    """G + s at k - s is the same H(k) as G at k."""
    print(f"case: {sym} flags {flags}, basis shifted by {shift}", flush=True)
    mat = load(sym)
    G = api.basis_vectors(8)
    ks = _kpoints(3)
    s = np.array(shift)
    H0 = _assemble(gpu_ctx, mat, G, flags, ks)
    H1 = _assemble(gpu_ctx, mat, G + s, flags, ks - s)
    if flags & api.SOC:
        # the spin-orbit phases of the two bases differ by a common one: some ulp of sin and cos
        assert np.abs(H1 - H0).max() <= 16 * 2.3e-16 * np.abs(H0).max()
    else:
        assert np.array_equal(H1, H0)
    for i, k in enumerate(ks):
        H = oracle.assemble(mat, G, k, nl=True, soc=bool(flags & api.SOC))
        tol = max(1e-9, 2.0e-6 / oracle.min_norm_gap(mat, G, k))  # its radial integrals lose digits where norms meet
        assert np.abs(H1[i] - H).max() <= tol


@pytest.mark.parametrize("apart", [(600, 0, 0), (0, 1024, 0), (1024, 1024, 1024), (-512, 512, 3)])
@pytest.mark.parametrize("sym", ["Si", "GaAs"])
def test_two_clusters_of_vectors(gpu_ctx, oracle, sym, apart):
    """A basis of two copies far apart: the local potential joins none of one to any of the other."""
    print(f"case: {sym} local, two copies {apart} apart", flush=True)
    mat = load(sym)
    G0 = api.basis_vectors(6)
    n = len(G0)
    G = np.vstack([G0, G0 + np.array(apart)])
    ks = _kpoints(2)
    H = _assemble(gpu_ctx, mat, G, 0, ks)
    assert np.all(H[:, :n, n:] == 0.0) and np.all(H[:, n:, :n] == 0.0)
    off = ~np.eye(n, dtype=bool)
    for i, k in enumerate(ks):
        ref = oracle.assemble(mat, G0, k, nl=False, soc=False)
        assert np.abs(H[i, :n, :n] - ref).max() <= 1e-9
        assert np.abs((H[i, n:, n:] - ref)[off]).max() <= 1e-9


def test_eigenvalues_of_a_shifted_basis(gpu_ctx, oracle):
    print("case: solve with a basis shifted by (600, -700, 0)", flush=True)
    G = api.basis_vectors(8)
    ks = _kpoints(5)
    s = np.array([600, -700, 0])
    for sym, flags, nb in (("Si", api.NONLOCAL, 8), ("GaAs", api.NONLOCAL, 8), ("Ge", api.NONLOCAL | api.SOC, 8)):
        mat = load(sym)
        e, _, _ = api.Plan(gpu_ctx, mat, np.ascontiguousarray(G + s, dtype=np.int32), flags, nb).solve(ks - s)
        w, _, _ = oracle.solve(mat, G, flags, nb, ks, nthreads=8)
        tol = max(1e-9, *[6.0 * 2.0e-6 / oracle.min_norm_gap(mat, G, k) for k in ks])
        assert np.abs(e - w).max() <= tol
