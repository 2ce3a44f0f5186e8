"""The 16 x 16-lane complex grids (complex64 blocks up to 160, complex128 up to 128) at
the edges of their blocks, first in the chain and after a larger grid, against LAPACK."""
from __future__ import annotations

import numpy as np
import pytest

from ultimateepm_amd import api
from ultimateepm_amd.material import load

pytestmark = pytest.mark.gpu

MIXED_TOL = 1e-4  # eV, the precision form's bar against FP64


@pytest.mark.parametrize("mixed", [True, False])
@pytest.mark.parametrize("dim", [65, 79, 80, 81, 95, 96, 97, 112, 113, 127, 128, 129, 144, 145, 159, 160, 161, 192])
def test_complex_grids(gpu_ctx, oracle, dim, mixed):
    print(f"case: GaAs, dim {dim}, mixed {mixed}", flush=True)
    mat = load("GaAs")
    G = np.ascontiguousarray(api.basis_vectors(13)[:dim])
    nb = 10
    ks = np.vstack([[0.0, 0.0, 0.0], api.bz_sample(dim, 3)])
    e, v, _ = api.Plan(gpu_ctx, mat, G, (api.MIXED if mixed else 0) | api.VECTORS, nb).solve(ks, vectors=True)
    for i, k in enumerate(ks):
        H = oracle.assemble(mat, G, k, nl=False, soc=False)
        X = v[i].T
        assert np.abs(e[i] - np.linalg.eigvalsh(H)[:nb]).max() <= (MIXED_TOL if mixed else 1e-9)
        assert np.linalg.norm(H @ X - X * e[i], axis=0).max() <= (1e-3 if mixed else 1e-8)
        assert np.abs(X.conj().T @ X - np.eye(nb)).max() <= 1e-10
