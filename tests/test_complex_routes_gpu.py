"""The complex kernels on compounds without an inversion centre (GaAs, GaP), whose plans
no real or quaternion kernel takes: every case names the reduction it means to run and
checks that the plan reports it, so that a change of the dispatch cannot empty it."""
from __future__ import annotations

import numpy as np
import pytest

from ultimateepm_amd import api
from ultimateepm_amd._abi import UEPM_ERR_NOT_CONVERGED, UepmError
from ultimateepm_amd.material import load

pytestmark = pytest.mark.gpu

MIXED_TOL = 1e-4  # eV: the precision form's bar against FP64

REG32 = "tridiag_reg_kernel<c64>"
STRIP32 = "tridiag_strip+reg_kernel<c64>"
BLOCKED_REG32 = "tridiag_blocked+reg_kernel<c64>"
BLOCKED32 = "tridiag_blocked_kernel<c64>"
REG64 = "tridiag_reg_kernel<c128>"
BLOCKED_REG64 = "tridiag_blocked+reg_kernel<c128>"


def _dev(ctx, a):
    return api.DeviceArray.from_host(ctx, np.ascontiguousarray(a))


def _basis(n):
    return np.ascontiguousarray(api.basis_vectors(22)[:n])


def _solve_device(ctx, p, ks, want_vec=False, want_grad=False):
    """(stage names, energies, vectors, gradients) of a device solve; the buffers start as zeros."""
    dk, de = _dev(ctx, ks), api.DeviceArray(ctx, (len(ks), p.nb))
    dv = api.DeviceArray(ctx, (len(ks), p.nb, p.dim, 2)) if want_vec else None
    dg = api.DeviceArray(ctx, (len(ks), p.nb, 3)) if want_grad else None
    for b in (de, dv, dg):
        if b:
            b.zero()
    p.set_timing(True)
    p.solve_device(dk.ptr, len(ks), de.ptr, dv.ptr if dv else 0, dg.ptr if dg else 0)
    p.set_timing(False)
    v = dv.numpy() if dv else None
    return (list(p.last_timing()), de.numpy(), v[..., 0] + 1j * v[..., 1] if dv else None, dg.numpy() if dg else None)


@pytest.mark.parametrize("sym,n,soc,flags,nb,route,cfg", [
    ("GaAs", 59, 0, 0, 8, REG64, {}),  # row kernel alone
    ("GaAs", 89, 0, api.GRADIENTS, 8, REG64, {}),
    ("GaAs", 181, 0, api.GRADIENTS, 10, REG64, {}),
    ("GaAs", 259, 0, api.GRADIENTS, 8, BLOCKED_REG64, {}),  # blocked, then the compact-WY back-transform
    ("GaAs", 137, api.SOC, api.GRADIENTS, 16, BLOCKED_REG64, {}),
    ("GaAs", 137, api.SOC, 0, 16, BLOCKED_REG64, {}),
    ("GaAs", 59, 0, api.MIXED, 8, REG32, {}),  # one wave alone
    ("GaP", 89, 0, api.MIXED | api.VECTORS, 12, REG32, {}),
    ("GaAs", 137, api.SOC, api.MIXED | api.GRADIENTS, 16, REG32, {}),  # 288 grid, two-tile refinement
    ("GaAs", 307, 0, api.MIXED | api.VECTORS, 12, STRIP32, {}),
    ("GaAs", 181, api.SOC, api.MIXED | api.GRADIENTS, 20, STRIP32, {}),
    ("GaAs", 229, api.SOC, api.MIXED, 12, BLOCKED_REG32, {}),
    ("GaP", 89, 0, api.MIXED | api.VECTORS, 12, BLOCKED32, {"tridiag": 1}),
    ("GaAs", 181, 0, api.GRADIENTS, 10, REG64, {"bt_bands": 8}),
])
def test_non_finite_k(gpu_ctx, oracle, sym, n, soc, flags, nb, route, cfg):
    """NaN and infinite k-points in a device batch over two chunks and lanes: NaN results
    and a status for those, every other k-point as if alone."""
    print(f"case: NaN/inf k, {sym} N={n} flags {flags | soc} nb {nb} {cfg}", flush=True)
    mat, G = load(sym), _basis(n)
    ks = api.bz_sample(31, 40)
    bad = [5, 29, 30]
    ks[5, 0], ks[29, 1], ks[30, 2] = np.nan, np.inf, -np.inf
    good = np.setdiff1d(np.arange(len(ks)), bad)
    p = api.Plan(gpu_ctx, mat, G, flags | soc, nb)  # local terms: the oracle keeps its digits
    p.set_config(max_chunk=24, **cfg)
    vec, grad = bool(flags & (api.VECTORS | api.GRADIENTS)), bool(flags & api.GRADIENTS)
    names, e, v, g = _solve_device(gpu_ctx, p, ks, vec, grad)
    assert names[1] == route
    assert p.status() == (len(bad), bad[0])
    assert np.all(np.isnan(e[bad])) and np.all(np.isfinite(e[good]))
    w, _, _ = oracle.solve(mat, G, soc, nb, ks[good], nthreads=8)
    assert np.abs(e[good] - w).max() <= (MIXED_TOL if flags & api.MIXED else 1e-9)
    for out in (v, g):
        if out is not None:
            assert np.all(np.isnan(out[bad])) and np.all(np.isfinite(out[good]))
    _, e2, v2, g2 = _solve_device(gpu_ctx, p, ks[good], vec, grad)  # and the status is cleared
    assert p.status() == (0, -1)
    assert np.array_equal(e2, e[good])
    for a, b in ((v2, v), (g2, g)):
        if a is not None:
            assert np.array_equal(a, b[good])
    p.close()


@pytest.mark.parametrize("n,flags,route", [(89, 0, REG64), (259, 0, BLOCKED_REG64), (137, api.MIXED, REG32),
                                           (307, api.MIXED, STRIP32)])
def test_overflowing_k(gpu_ctx, n, flags, route):
    print(f"case: |k| = 1e160, GaAs N={n} flags {flags}", flush=True)
    p = api.Plan(gpu_ctx, load("GaAs"), _basis(n), api.NONLOCAL | api.GRADIENTS | flags, 8)
    ks = api.bz_sample(8, 6)
    assert _solve_device(gpu_ctx, p, ks)[0][1] == route
    ks[3] = (1e160, 0.0, 0.0)
    with pytest.raises(UepmError) as err:
        p.solve(ks, vectors=True)
    assert err.value.code == UEPM_ERR_NOT_CONVERGED and "first at index 3" in str(err.value)
    good = [0, 1, 2, 4, 5]
    for out in err.value.result:
        assert np.all(np.isnan(out[3])) and np.all(np.isfinite(out[good]))
    p.close()


@pytest.mark.parametrize("n,flags,route", [(137, api.NONLOCAL | api.VECTORS, REG64),
                                           (229, api.VECTORS, BLOCKED_REG64),
                                           (137, api.NONLOCAL | api.VECTORS | api.MIXED, REG32),
                                           (307, api.VECTORS | api.MIXED, STRIP32)])
def test_two_lanes_equal_one_lane(gpu_ctx, n, flags, route):
    """Alternate chunks on a second stream, each with its own workspace: the same bits."""
    print(f"case: lanes 2 vs 1, GaAs N={n} flags {flags}, 300 k in chunks of 64", flush=True)
    ks = api.bz_sample(13, 300)
    p = api.Plan(gpu_ctx, load("GaAs"), _basis(n), flags, 10)
    out = None
    for lanes in (1, 2, 0):
        p.set_config(max_chunk=64, lanes=lanes)
        names, e, v, _ = _solve_device(gpu_ctx, p, ks, True)
        assert names[1] == route
        if out:
            assert np.array_equal(e, out[0]) and np.array_equal(v, out[1])
        out = (e, v)
    p.close()


@pytest.mark.parametrize("dim,soc", [(200, 0), (224, 0), (225, 0), (240, 0), (256, 0), (257, 0), (259, 0), (280, api.SOC),
                                     (288, api.SOC), (288, 0)])
def test_wide_complex64_grids(gpu_ctx, oracle, dim, soc):
    """First blocks of the 224-, 256- and 288-wide complex64 grids and their edges."""
    print(f"case: mixed GaAs, dim {dim}, soc {bool(soc)}", flush=True)
    mat, G, nb = load("GaAs"), _basis(dim // 2 if soc else dim), 12
    p = api.Plan(gpu_ctx, mat, G, soc | api.MIXED | api.VECTORS, nb)
    ks = np.vstack([[0.0, 0.0, 0.0], [0.5, 0.5, 0.5], api.bz_sample(77, 6)])
    names, e, v, _ = _solve_device(gpu_ctx, p, ks, True)
    assert names[1] == REG32
    w, _, _ = oracle.solve(mat, G, soc, nb, ks, nthreads=8)
    assert np.abs(e - w).max() <= MIXED_TOL
    for i, k in enumerate(ks[:3]):
        H = oracle.assemble(mat, G, k, nl=False, soc=bool(soc))
        X = v[i].T
        assert np.abs(X.conj().T @ X - np.eye(nb)).max() <= 1e-10
        assert np.linalg.norm(H @ X - X * e[i], axis=0).max() <= 1e-3  # complex64 subspace
    p.close()


def _same_spaces(ev, v0, v1, tol):
    """Bands split into clusters at gaps above 50 meV: each cluster's two bases span the same space."""
    nb, checked = ev.shape[1], 0
    d = np.diff(ev, axis=1)
    for i in range(len(ev)):
        cuts = [0] + [b + 1 for b in range(nb - 1) if d[i, b] > 0.05]
        for a, b in zip(cuts[:-1], cuts[1:]):
            s = np.linalg.svd(v0[i, a:b].conj() @ v1[i, a:b].T, compute_uv=False)
            assert np.abs(s - 1.0).max() <= tol, (i, a, b, s)
            checked += b - a
    assert checked >= ev.size // 2


@pytest.mark.parametrize("n,soc,nb,route", [(259, 0, 12, REG32), (137, api.SOC, 16, REG32), (169, api.SOC, 24, STRIP32),
                                            (181, api.SOC, 20, STRIP32), (259, api.SOC, 16, BLOCKED_REG32), (137, 0, 24, REG32)])
def test_wy_back_transform_matches_per_reflector(gpu_ctx, n, soc, nb, route):
    """Precision form: the compact-WY back-transform (automatic above dim 192 or past 16
    Ritz vectors: one band tile, two, two passes of one at dim 518) against the
    reflector-by-reflector kernel: the same subspace to the Ritz step."""
    print(f"case: WY vs per-reflector, mixed GaAs N={n} soc {bool(soc)} nb {nb}", flush=True)
    p = api.Plan(gpu_ctx, load("GaAs"), _basis(n), api.MIXED | api.VECTORS | soc, nb)
    ks = api.bz_sample(808, 24)
    names, ev0, v0, _ = _solve_device(gpu_ctx, p, ks, True)
    assert names[1] == route
    p.set_config(bt_bands=16)
    _, ev1, v1, _ = _solve_device(gpu_ctx, p, ks, True)
    assert not np.array_equal(v0, v1)  # two kernels: their sums round differently
    assert np.abs(ev0 - ev1).max() <= 1e-8
    _same_spaces(ev1, v0, v1, 1e-5)
    p.close()


@pytest.mark.parametrize("n,soc,nb", [(137, api.SOC, 16), (411, 0, 24), (229, api.SOC, 12), (259, api.SOC, 16)])
def test_fp64_wy_back_transform_matches_per_reflector(gpu_ctx, n, soc, nb):
    """FP64 above dim 192: both back-transforms apply the same Q to the same vectors of T."""
    print(f"case: FP64 WY vs per-reflector, GaAs N={n} soc {bool(soc)} nb {nb}", flush=True)
    p = api.Plan(gpu_ctx, load("GaAs"), _basis(n), api.GRADIENTS | soc, nb)
    ks = api.bz_sample(909, 16)
    names, ev0, v0, g0 = _solve_device(gpu_ctx, p, ks, True, True)
    assert names[1] == BLOCKED_REG64
    p.set_config(bt_bands=16)
    _, ev1, v1, g1 = _solve_device(gpu_ctx, p, ks, True, True)
    assert np.array_equal(ev0, ev1) and not np.array_equal(v0, v1)
    assert np.abs(v0 - v1).max() <= 1e-11
    assert np.abs(g0 - g1).max() <= 1e-9 * max(1.0, np.abs(g1).max())
    assert np.abs(np.linalg.norm(v0, axis=2) - 1.0).max() <= 1e-12
    p.close()


@pytest.mark.parametrize("sym,n,nb,refine", [("GaAs", 137, 12, "refine_mfma_kernel"), ("GaAs", 137, 24, "refine_mfma2_kernel"),
                                             ("GaP", 89, 20, "refine_mfma2_kernel")])
def test_complex_refinement(gpu_ctx, oracle, sym, n, nb, refine):
    """One and two band tiles of the complex FP64 Rayleigh-Ritz step."""
    print(f"case: mixed {sym} N={n} nb {nb}", flush=True)
    mat, G = load(sym), _basis(n)
    p = api.Plan(gpu_ctx, mat, G, api.MIXED | api.GRADIENTS, nb)
    ks = np.vstack([[0.0, 0.0, 0.0], api.bz_sample(314, 20)])
    names, e, v, g = _solve_device(gpu_ctx, p, ks, True, True)
    assert names[1] == REG32 and names[4] == refine
    w, _, go = oracle.solve(mat, G, api.GRADIENTS, nb, ks, nthreads=8)
    assert np.abs(e - w).max() <= MIXED_TOL
    d = np.diff(w, axis=1)
    ok = np.ones(w.shape, dtype=bool)
    ok[:, :-1] &= d > 1e-3
    ok[:, 1:] &= d > 1e-3
    ok[:, -1] = False
    # gradients carry the Ritz vectors' accuracy (complex64 subspace, FP64 Ritz step)
    assert np.abs(g - go)[ok].max() <= 1e-4 * np.abs(go).max()
    assert np.abs(v @ v.conj().transpose(0, 2, 1) - np.eye(nb)).max() <= 1e-10
    p.close()


def test_tuned_plan_above_the_register_grids(gpu_ctx):
    """Above dim 288 the tuner times the strip and the LDS-blocked reduction alone, above
    384 the blocked one with and without the grids: one bar for every candidate."""
    for n, auto in ((169, STRIP32), (229, BLOCKED_REG32)):
        print(f"case: autotune GaAs SOC N={n} mixed, 96 k", flush=True)
        ks = api.bz_sample(11, 96)
        p = api.Plan(gpu_ctx, load("GaAs"), _basis(n), api.SOC | api.MIXED, 16)
        names, ev0, _, _ = _solve_device(gpu_ctx, p, ks)
        assert names[1] == auto
        dk = _dev(gpu_ctx, ks)
        chosen = p.tune(dk.ptr, len(ks))
        assert chosen["tridiag"] in (0, 1) and chosen["tri_block"] in (256, 512)
        _, ev1, _, _ = _solve_device(gpu_ctx, p, ks)
        assert np.abs(ev1 - ev0).max() <= 1e-8
        p.set_config(tridiag=1, tri_block=512, bt_bands=8)
        names, ev2, _, _ = _solve_device(gpu_ctx, p, ks)
        assert names[1] == BLOCKED32 and np.abs(ev2 - ev0).max() <= 1e-8
        p.close()


def test_batch_graph_over_complex_plans(gpu_ctx):
    """The strip, the blocked kernel, both compact-WY back-transforms and the complex
    refinement captured into one graph: every replay equals the plans' own solves, with
    eager work between the replays."""
    print("case: batch graph over 4 GaAs plans, 3 replays", flush=True)
    specs = [(137, api.SOC | api.GRADIENTS, 16, BLOCKED_REG64), (181, api.SOC | api.MIXED | api.VECTORS, 16, STRIP32),
             (89, api.NONLOCAL | api.GRADIENTS, 8, REG64), (137, api.MIXED | api.VECTORS, 12, REG32)]
    plans, ks, bufs, ref = [], [], [], []
    for i, (n, flags, nb, route) in enumerate(specs):
        p = api.Plan(gpu_ctx, load("GaAs"), _basis(n), flags, nb)
        k = api.bz_sample(300 + i, 60 + 20 * i)
        names, e, v, _ = _solve_device(gpu_ctx, p, k, True)
        assert names[1] == route
        ref.append((e, v))
        plans.append(p)
        ks.append(k)
        bufs.append((_dev(gpu_ctx, k), api.DeviceArray(gpu_ctx, (len(k), nb)), api.DeviceArray(gpu_ctx, (len(k), nb, p.dim, 2))))
    b = api.Batch(gpu_ctx, [(p, dk.ptr, len(k), de.ptr, dv.ptr) for p, k, (dk, de, dv) in zip(plans, ks, bufs)], branches=3)
    for replay in range(3):
        for _, de, dv in bufs:
            de.zero()
            dv.zero()
        b.launch()
        gpu_ctx.synchronize()
        for p, k in zip(plans, ks):
            p.solve(k[:5])
        for (_, de, dv), (e, v), spec in zip(bufs, ref, specs):
            got = dv.numpy()
            assert np.array_equal(de.numpy(), e), (replay, spec)
            assert np.array_equal(got[..., 0] + 1j * got[..., 1], v), (replay, spec)
    b.close()
    for p in plans:
        p.close()
