"""FP64 eigenvalues of a tridiagonal matrix to their own rounding: with every form
factor zero H(k) is diagonal, no column takes a reflector and T is H's diagonal, so
each level is one diagonal element and the bisection alone sets its error, however
far below ||H|| it lies."""
from __future__ import annotations

import copy

import numpy as np
import pytest

from ultimateepm_amd import api
from ultimateepm_amd.material import load

pytestmark = pytest.mark.gpu

KS = np.array([[1e-6, 2e-6, 3e-6], [1e-9, 0.0, 0.0], [1e-4, -1e-4, 1e-4], [0.0, 0.0, 0.0], [0.25, 0.125, -0.5],
               [1.0, 0.0, 0.0], [1.0 - 1e-7, 1.0, 1e-7]])


@pytest.mark.parametrize("n,nb", [(6, 8), (8, 12), (8, 30), (8, 64), (10, 16)])
@pytest.mark.parametrize("route", ["real", "complex", "quaternion"])
@pytest.mark.parametrize("vectors", [False, True])
def test_levels_of_the_empty_lattice(gpu_ctx, n, nb, route, vectors):
    print(f"case: empty lattice, n={n}, {nb} bands, {route}, vectors {vectors}", flush=True)
    m = copy.deepcopy(load("Si"))
    m.V_S = m.V_A = (0.0, 0.0, 0.0, 0.0)
    m.spin_orbit.mu = 0.0
    flags = (api.SOC if route == "quaternion" else 0) | (api.VECTORS if vectors else 0)
    p = api.Plan(gpu_ctx, m, api.basis_vectors(n), flags, nb)
    if route == "complex":
        p.set_config(tridiag=1)
    dk = api.DeviceArray.from_host(gpu_ctx, KS)
    dH = api.DeviceArray(gpu_ctx, (len(KS), p.dim, p.dim, 2))
    p.assemble_device(dk.ptr, len(KS), dH.ptr)
    gpu_ctx.synchronize()
    d = np.sort(np.einsum("kii->ki", dH.numpy()[..., 0]), axis=1)[:, :nb]
    e, _, _ = p.solve(KS)
    # a bracket of 2 eps |E| is final and its middle is returned: eps |E|, and rounding; at
    # zero itself the bracket closes by halves and fifths for 200 sweeps
    assert np.all(np.abs(e - d) <= 4 * 2.3e-16 * np.abs(d) + 1e-40)
    p.close()


@pytest.mark.parametrize("f", [1e-9, 1e-10, 1e-12])
@pytest.mark.parametrize("route", ["real", "complex"])
def test_level_behind_a_tiny_coupling(gpu_ctx, f, route):
    """Form factors scaled to 1e-9: T's first diagonal element is H's, its coupling to the
    rest under the rounding of ||T||, so second-order perturbation theory gives the lowest
    level near the zone centre to its own digits (the next order is below 1e-15 of it)."""
    print(f"case: form factors x {f}, {route}", flush=True)
    m = copy.deepcopy(load("Si"))
    m.V_S = tuple(f * v for v in m.V_S)
    G = api.basis_vectors(8)
    G = np.ascontiguousarray(G[np.argsort((G * G).sum(1), kind="stable")])  # G = 0 first
    p = api.Plan(gpu_ctx, m, G, 0, 8)
    if route == "complex":
        p.set_config(tridiag=1)
    ks = np.array([[1e-6, 2e-6, 3e-6], [2e-7, 0.0, 1e-7], [1e-4, -1e-4, 1e-4]])
    dk = api.DeviceArray.from_host(gpu_ctx, ks)
    dH = api.DeviceArray(gpu_ctx, (len(ks), p.dim, p.dim, 2))
    p.assemble_device(dk.ptr, len(ks), dH.ptr)
    gpu_ctx.synchronize()
    h = dH.numpy()
    e, _, _ = p.solve(ks)
    for i in range(len(ks)):
        d = np.diag(h[i, :, :, 0])
        v2 = (h[i, 0, 1:] ** 2).sum(-1)
        w = d[0] - (v2 / (d[1:] - d[0])).sum()
        assert abs(e[i, 0] - w) <= 1e-12 * abs(w)
    p.close()
