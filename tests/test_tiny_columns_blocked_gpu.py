"""The LDS-blocked reduction on matrices whose off-diagonal elements are tiny or zero
(form factors scaled down), alone and ahead of the register grids: a column too small
for its squared norm takes no reflector; eigenvalues and vectors are LAPACK's."""
from __future__ import annotations

import copy

import numpy as np
import pytest

from ultimateepm_amd import api
from ultimateepm_amd.material import load

pytestmark = pytest.mark.gpu

MIXED_TOL = 1e-4  # eV, the precision form's bar against FP64


@pytest.mark.parametrize("dim,mixed,blocked_alone", [(200, False, False), (259, False, False), (100, True, True),
                                                     (330, True, True), (392, True, False)])
@pytest.mark.parametrize("f", [0.0, 1e-170, 1e-162, 1e-156, 1e-148, 1e-144, 1e-120, 1e-42, 1e-39, 1e-37, 1e-30, 1e-16, 1e-14,
                               1e-8])
def test_scaled_form_factors(gpu_ctx, oracle, dim, mixed, blocked_alone, f):
    print(f"case: GaAs local, dim {dim}, mixed {mixed}, blocked alone {blocked_alone}, form factors x {f}", flush=True)
    m = copy.deepcopy(load("GaAs"))
    m.V_S = tuple(f * v for v in m.V_S)
    m.V_A = (f * m.V_A[0], f * m.V_A[1], f * m.V_A[2], f * m.V_A[3] or 1e-300)  # complex kernels at f = 0 too
    G = np.ascontiguousarray(api.basis_vectors(20)[:dim])
    nb = 10
    ks = np.vstack([[0.0, 0.0, 0.0], api.bz_sample(3, 3)])
    p = api.Plan(gpu_ctx, m, G, api.VECTORS | (api.MIXED if mixed else 0), nb)
    if blocked_alone:
        p.set_config(tridiag=1)
    e, v, _ = p.solve(ks, vectors=True)
    p.close()
    for i, k in enumerate(ks):
        H = oracle.assemble(m, G, k, nl=False, soc=False)
        w = np.linalg.eigvalsh(H)[:nb]
        assert np.abs(e[i] - w).max() <= (MIXED_TOL if mixed else 1e-9)
        X = v[i].T
        assert np.linalg.norm(H @ X - X * e[i], axis=0).max() <= (1e-3 if mixed else 1e-8)
        assert np.abs(X.conj().T @ X - np.eye(nb)).max() <= 1e-10
