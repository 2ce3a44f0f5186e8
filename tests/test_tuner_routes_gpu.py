"""The autotuner times the routes that the plans take by themselves: the real and
quaternion kernels of crystals of equal atoms stay on, in both forms, and a knob that
a plan's kernels do not have is left automatic, not picked among equal timings."""
from __future__ import annotations

import numpy as np
import pytest

from ultimateepm_amd import api
from ultimateepm_amd.material import load

pytestmark = pytest.mark.gpu


def _reduction(ctx, plan, ks):
    plan.set_timing(True)
    dk = api.DeviceArray.from_host(ctx, ks)
    de = api.DeviceArray(ctx, (len(ks), plan.nb))
    plan.solve_device(dk.ptr, len(ks), de.ptr)
    plan.set_timing(False)
    return list(plan.last_timing())[1]


@pytest.mark.parametrize("sym,n,flags,nb,route", [
    ("Si", 8, api.NONLOCAL, 8, "tridiag_real<f64>"),
    ("Si", 12, api.NONLOCAL | api.VECTORS, 12, "tridiag_real<f64>"),
    ("Si", 14, api.NONLOCAL, 8, "tridiag_real<f64>"),
    ("Si", 12, api.NONLOCAL | api.MIXED, 12, "tridiag_real<f32>"),
    ("Si", 16, api.NONLOCAL | api.MIXED, 12, "tridiag_real<f32>"),
    ("Ge", 8, api.NONLOCAL | api.SOC, 16, "tridiag_quaternion<f64>"),
    ("Ge", 10, api.NONLOCAL | api.SOC | api.VECTORS, 16, "tridiag_quaternion<f64>"),
    ("Ge", 10, api.NONLOCAL | api.SOC | api.MIXED, 16, "tridiag_quaternion<f32>"),
    ("Ge", 11, api.NONLOCAL | api.SOC | api.MIXED, 16, "tridiag_quaternion<f32>"),
])
def test_symmetric_plans_keep_their_kernels(gpu_ctx, sym, n, flags, nb, route):
    print(f"case: tune {sym} n={n} flags {flags}", flush=True)
    ks = api.bz_sample(5, 96)
    dk = api.DeviceArray.from_host(gpu_ctx, ks)
    for before in ({}, {"tridiag": 1, "bt_bands": 8}):  # whatever the plan was configured to
        p = api.Plan(gpu_ctx, load(sym), api.basis_vectors(n), flags, nb)
        want, _, _ = p.solve(ks)
        p.set_config(max_chunk=64, **before)
        chosen = p.tune(dk.ptr, len(ks))
        assert chosen["tridiag"] != 1 and chosen["bt_bands"] == 0 and chosen["max_chunk"] == 64
        assert _reduction(gpu_ctx, p, ks) == route
        got, _, _ = p.solve(ks)
        assert np.array_equal(got, want)
        p.close()


@pytest.mark.parametrize("sym,n,flags,nb,route", [
    ("GaAs", 8, api.NONLOCAL, 8, "tridiag_reg_kernel<c128>"),
    ("GaAs", 14, api.NONLOCAL | api.VECTORS, 8, "tridiag_blocked+reg_kernel<c128>"),
    ("GaAs", 10, api.NONLOCAL | api.SOC, 16, "tridiag_blocked+reg_kernel<c128>"),
])
def test_a_choice_serves_the_other_route_of_its_dimension(gpu_ctx, sym, n, flags, nb, route):
    """An FP64 III-V plan is tuned without turning the automatic reduction off, so its
    choice given to a crystal of equal atoms leaves that one's kernels on too."""
    print(f"case: tune FP64 {sym} n={n} flags {flags}", flush=True)
    ks = api.bz_sample(6, 96)
    dk = api.DeviceArray.from_host(gpu_ctx, ks)
    p = api.Plan(gpu_ctx, load(sym), api.basis_vectors(n), flags, nb)
    want, vec, _ = p.solve(ks)
    chosen = p.tune(dk.ptr, len(ks))
    assert chosen["tridiag"] == 0
    if not flags & api.VECTORS:
        assert chosen["bt_bands"] == 0  # no back-transform runs
    assert _reduction(gpu_ctx, p, ks) == route
    got, _, _ = p.solve(ks)
    assert np.abs(got - want).max() <= 1e-10  # the blocked kernel's widths add in other orders
    q = api.Plan(gpu_ctx, load("Ge" if flags & api.SOC else "Si"), api.basis_vectors(n), flags, nb)
    q.set_config(**chosen)
    assert _reduction(gpu_ctx, q, ks).startswith("tridiag_quaternion" if flags & api.SOC else "tridiag_real")
    p.close()
    q.close()
