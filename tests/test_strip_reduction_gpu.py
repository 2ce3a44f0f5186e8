"""The strip kernel (complex64 reduction above the register grids, dims 289 to 384)
at the edges of its block columns, and after the blocked reduction above 384,
against the oracle; III-V compounds (complex H(k)), with and without spin-orbit."""
from __future__ import annotations

import numpy as np
import pytest

from ultimateepm_amd import api
from ultimateepm_amd.material import load

pytestmark = pytest.mark.gpu

MIXED_TOL = 1e-8  # eV, the precision form's bar


@pytest.mark.parametrize("dim,soc", [(289, False), (290, True), (303, False), (304, False), (305, False), (320, True),
                                     (321, False), (336, True), (352, False), (353, False), (367, False), (368, True),
                                     (369, False), (383, False), (384, True), (385, False), (386, True), (400, False)])
def test_strip_kernel(gpu_ctx, oracle, dim, soc):
    print(f"case: mixed GaAs, dim {dim}, soc {soc}", flush=True)
    mat = load("GaAs")
    G = np.ascontiguousarray(api.basis_vectors(24)[: dim // 2 if soc else dim])
    flags = api.SOC if soc else 0  # local terms otherwise: no radial integrals between the two
    plan = api.Plan(gpu_ctx, mat, G, flags | api.MIXED | api.VECTORS, 12)
    assert plan.dim == dim
    ks = np.vstack([[0.0, 0.0, 0.0], api.bz_sample(dim, 3)])
    e, v, _ = plan.solve(ks, vectors=True)
    w, _, _ = oracle.solve(mat, G, flags, 12, ks, nthreads=8)
    assert np.abs(e - w).max() <= MIXED_TOL
    for i, k in enumerate(ks):
        X = v[i].T
        H = oracle.assemble(mat, G, k, nl=False, soc=soc)
        assert np.linalg.norm(H @ X - X * e[i], axis=0).max() <= 1e-3
        assert np.abs(X.conj().T @ X - np.eye(12)).max() <= 1e-10
