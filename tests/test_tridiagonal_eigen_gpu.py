"""The eigen-stage (multisection by principal minors, inverse iteration by blocks of
rows) at its edges: orders around the row blocks, every width of the band groups,
degenerate levels at high-symmetry points, against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

from ultimateepm_amd import api
from ultimateepm_amd.material import load

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ng,nb", [(1, 1), (2, 2), (7, 7), (8, 8), (9, 9), (15, 15), (16, 16), (17, 17), (24, 16), (32, 32),
                                   (33, 33), (65, 16), (65, 17), (65, 32), (65, 33), (65, 64), (65, 65), (89, 80), (181, 70)])
def test_eigen_stage(gpu_ctx, oracle, ng, nb):
    print(f"case: FP64 GaAs, {ng} vectors, {nb} bands", flush=True)
    mat = load("GaAs")
    G = np.ascontiguousarray(api.basis_vectors(12)[:ng])
    ks = np.vstack([[0.0, 0.0, 0.0], [1.0, 0.0, 0.0], [0.5, 0.5, 0.5], api.bz_sample(ng, 4)])
    e, v, _ = api.Plan(gpu_ctx, mat, G, api.VECTORS, nb).solve(ks, vectors=True)  # local terms: no integrals between the two
    assert np.all(np.diff(e, axis=1) >= -1e-12)
    w, _, _ = oracle.solve(mat, G, 0, nb, ks, nthreads=8)
    assert np.abs(e - w).max() <= 1e-9
    for i, k in enumerate(ks):
        H = oracle.assemble(mat, G, k, nl=False, soc=False)
        X = v[i].T
        assert np.linalg.norm(H @ X - X * e[i], axis=0).max() <= 1e-8
        assert np.abs(X.conj().T @ X - np.eye(nb)).max() <= 1e-10
