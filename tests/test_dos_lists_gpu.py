"""The DOS kernel's lists of cutting (energy, tetrahedron) pairs at their edges: around
the block of tetrahedra, slices of more than one block, energies that cut every
tetrahedron or none, groups of energies that are not full, against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

from ultimateepm_amd import mesh

pytestmark = pytest.mark.gpu


def _soup(nt, seed):
    """nt separate tetrahedra of random corners, an energy and a gradient at each corner."""
    rng = np.random.default_rng(seed)
    xyz = rng.uniform(-1.0, 1.0, size=(4 * nt, 3)) * 1e10
    tet = np.arange(4 * nt, dtype=np.int32).reshape(nt, 4)
    v = np.einsum("ti,ti->t", xyz[1::4] - xyz[::4], np.cross(xyz[2::4] - xyz[::4], xyz[3::4] - xyz[::4]))
    tet[v < 0] = tet[v < 0][:, [0, 2, 1, 3]]
    E = rng.uniform(-1.0, 1.0, size=(4 * nt, 1))
    E[: 2 * nt : 4] -= 1.5  # half the tetrahedra: one corner well below zero, one well above, all cut there
    E[1 : 2 * nt : 4] += 1.5
    return xyz, tet, E, rng.uniform(0.5, 2.0, size=(4 * nt, 1, 3)) * 1e-10


@pytest.mark.parametrize("nt,points", [(1, 2), (1, 5), (255, 4), (256, 3), (1023, 9), (1024, 8), (1025, 2), (2049, 33),
                                       (4 * 1024, 6), (256 * 1024 + 1, 5)])
def test_lists(gpu_ctx, oracle, nt, points):
    print(f"case: tetra DOS, {nt} tetrahedra, {points} energies", flush=True)
    xyz, tet, E, G = _soup(nt, nt + points)
    m = mesh.MeshBZ.from_arrays(gpu_ctx, xyz, tet)
    m.set_bands(E, G)
    for lo, hi in ((-3.0, 3.0), (-0.2, 0.3), (5.0, 6.0)):
        _, dos = m.dos(0, points, lo, hi, 1.0, 2.0)
        _, dos_o = oracle.tetra_dos(xyz, tet, E, G, 0, points, lo, hi, 1.0, 2.0, nthreads=8)
        assert np.abs(dos - dos_o).max() <= 1e-10 * np.abs(dos_o).max()
        if nt > 1 and -1.0 < lo < 5.0:
            assert dos_o.max() > 0.0
        # an energy alone and in a grid: the same bits
        _, two = m.dos(0, 2, lo, hi, 1.0, 2.0)
        assert two[0] == dos[0]
    m.close()
