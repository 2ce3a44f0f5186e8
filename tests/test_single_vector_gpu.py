"""A basis of one vector, down to H(k) = 0 at the zone centre: the smallest solve that an
entry point takes.  The eigenvector is a unit vector and no k-point fails, however small
H(k) is, in every form and with every kind of crystal."""
from __future__ import annotations

import numpy as np
import pytest

from ultimateepm_amd import api
from ultimateepm_amd.material import load

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sym", ["Si", "GaAs"])
@pytest.mark.parametrize("soc", [0, api.SOC])
@pytest.mark.parametrize("mixed", [0, api.MIXED])
def test_one_vector(gpu_ctx, sym, soc, mixed):
    print(f"case: {sym}, G = 0 alone, soc {bool(soc)}, mixed {bool(mixed)}", flush=True)
    x = np.array([0.0, 1e-160, 1e-153, 1e-120, 1e-85, 1e-30, 1e-8, 1e-3, 0.5])
    ks = np.stack([x, 0.0 * x, -2.0 * x], axis=1)
    nb = 2 if soc else 1
    p = api.Plan(gpu_ctx, load(sym), np.zeros((1, 3), dtype=np.int32), soc | mixed | api.GRADIENTS, nb)
    e, v, g = p.solve(ks, vectors=True)
    assert p.status() == (0, -1)
    dk = api.DeviceArray.from_host(gpu_ctx, ks)
    dH = api.DeviceArray(gpu_ctx, (len(ks), p.dim, p.dim, 2))
    p.assemble_device(dk.ptr, len(ks), dH.ptr)
    gpu_ctx.synchronize()
    H = dH.numpy()[..., 0]
    d = np.einsum("kii->ki", H)
    assert np.all(H[:, ~np.eye(nb, dtype=bool)] == 0.0) and np.all(d[0] == 0.0)
    # one or two equal diagonal elements: rounding of the bisection (2 eps) or of the Ritz
    # step, and 200 sweeps' worth of a bracket at the smallest
    assert np.all(np.abs(e - d) <= 8 * 2.3e-16 * d + 1e-150)
    assert np.abs(v @ v.conj().transpose(0, 2, 1) - np.eye(nb)).max() <= 1e-12
    assert np.all(np.isfinite(g)) and np.all(g[0] == 0.0)
    p.close()
