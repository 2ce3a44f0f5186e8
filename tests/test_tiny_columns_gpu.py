"""Reductions of matrices whose off-diagonal elements are tiny or zero (form factors
scaled down): a column under the grids' smallest is no reflector, everything above it
is, and the eigenvalues and vectors are LAPACK's either way.  Complex, real and
quaternion chains."""
from __future__ import annotations

import copy

import numpy as np
import pytest

from ultimateepm_amd import api
from ultimateepm_amd.material import load

pytestmark = pytest.mark.gpu

MIXED_TOL = 1e-4  # eV, the precision form's bar against FP64


@pytest.mark.parametrize("sym", ["GaAs", "Si"])
@pytest.mark.parametrize("f", [0.0, 1e-162, 1e-148, 1e-144, 1e-120, 1e-30, 1e-17, 1e-16, 1e-15, 1e-14, 1e-12, 1e-8, 1e-4])
def test_scaled_form_factors(gpu_ctx, oracle, sym, f):
    print(f"case: {sym}, form factors x {f}", flush=True)
    m = copy.deepcopy(load(sym))
    m.V_S = tuple(f * v for v in m.V_S)
    m.V_A = tuple(f * v for v in m.V_A)
    G = api.basis_vectors(10)
    nb = 12
    ks = np.vstack([[0.0, 0.0, 0.0], api.bz_sample(3, 4)])
    for soc in (0, api.SOC):
        # LAPACK's eigenvalues of the oracle's H: the oracle's own reduction underflows at 1e-162
        w = np.array([np.linalg.eigvalsh(oracle.assemble(m, G, k, nl=False, soc=bool(soc)))[:nb] for k in ks])
        for flags, tol, res in ((0, 1e-9, 1e-8), (api.MIXED, MIXED_TOL, 1e-3)):
            e, v, _ = api.Plan(gpu_ctx, m, G, flags | soc | api.VECTORS, nb).solve(ks, vectors=True)
            assert np.abs(e - w).max() <= tol
            for i, k in enumerate(ks):
                H = oracle.assemble(m, G, k, nl=False, soc=bool(soc))
                X = v[i].T
                assert np.linalg.norm(H @ X - X * e[i], axis=0).max() <= res
                assert np.abs(X.conj().T @ X - np.eye(nb)).max() <= 1e-10
