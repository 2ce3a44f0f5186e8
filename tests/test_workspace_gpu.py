"""Workspace of a k-point: a region (a server's slot, the no-allocation array) that took a
plan with the complex kernels takes it with the real and quaternion ones."""
from __future__ import annotations

import numpy as np
import pytest

from ultimateepm_amd import api
from ultimateepm_amd.material import load

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flags", [0, api.VECTORS, api.MIXED, api.MIXED | api.VECTORS])
@pytest.mark.parametrize("sym,soc,top", [("Si", 0, 448), ("Ge", api.SOC, 192)])
def test_symmetric_plans_take_no_more_than_complex_ones(gpu_ctx, sym, soc, top, flags):
    print(f"case: workspace of {sym} plans, flags {flags | soc}", flush=True)
    basis = api.basis_vectors(24)
    for N in [1, 2, 3, 16, 31, 32, 33, 64, 65, 96, 97, 128, 129, 144, 145, 160, 161, 192, 193, 224, 225, 256, 257, 288, 289,
              296, 320, 321, 384, 385, 448]:
        dim = 2 * N if soc else N
        if N > top:
            continue
        for nb in (1, min(dim, 12), min(dim, 24)):
            p = api.Plan(gpu_ctx, load(sym), np.ascontiguousarray(basis[:N]), flags | soc, nb)
            auto = p.workspace_bytes(1)
            p.set_config(tridiag=1)
            assert auto <= p.workspace_bytes(1), (N, nb)
            p.close()


@pytest.mark.parametrize("dim", [289, 320, 384, 385, 400, 450, 512, 576])
@pytest.mark.parametrize("nb", [1, 12, 24])
def test_hand_over_of_large_complex64_reductions(gpu_ctx, dim, nb):
    """Above dim 288 the reduction's own workspace is the larger of two hand-over blocks
    (256 and 224 rows) and the blocked kernel's columns, beside H, the reflectors and
    what the later stages hold."""
    print(f"case: workspace of a mixed GaAs plan, dim {dim}, {nb} bands", flush=True)
    p = api.Plan(gpu_ctx, load("GaAs"), np.ascontiguousarray(api.basis_vectors(26)[:dim]), api.MIXED, nb)
    auto = p.workspace_bytes(1)
    p.set_config(tridiag=1)
    blocked = p.workspace_bytes(1)
    p.close()
    nbr = nb + 4
    held = 24 * dim * dim + 40 * dim + (8 + 56 * dim) * nbr + 4
    assert auto - held <= max(8 * (256 * 256 + 224 * 224), blocked - held)
