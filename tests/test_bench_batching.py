"""bench.py's batching leg, on stand-ins for the device: each plan gets a configuration
that was tuned on a plan of its own dimension and kind of crystal."""
from __future__ import annotations

import types

import numpy as np

import bench
from ultimateepm_amd import api


class _Array:
    def __init__(self, ctx, shape):
        self.ptr, self._shape = 1, shape

    @classmethod
    def from_host(cls, ctx, a):
        return cls(ctx, a.shape)

    def numpy(self):
        return np.zeros(self._shape)

    def free(self):
        pass


def test_choices_stay_with_their_kind_of_crystal(monkeypatch):
    plans = []

    class Plan:
        def __init__(self, ctx, mat, G, flags, nb):
            self.sym, self.dim = mat.name, len(G) * (2 if flags & api.SOC else 1)
            self.equal = mat.name in ("Si", "Ge", "Sn")
            self.form = bool(flags & api.MIXED)
            self.cfg = None
            plans.append(self)

        def workspace_bytes(self, nk):
            return 1 << 20

        def tune(self, ptr, nk):
            return {"tridiag": 0, "tri_block": 0, "bt_bands": 0, "lanes": 0, "from": (self.dim, self.equal, self.form)}

        def set_config(self, **cfg):
            self.cfg = cfg

        def solve_device(self, *a):
            pass

        def close(self):
            pass

    monkeypatch.setattr(api, "Plan", Plan)
    monkeypatch.setattr(api, "DeviceArray", _Array)
    monkeypatch.setattr(api, "Batch", lambda ctx, items, branches: types.SimpleNamespace(launch=lambda: None, close=lambda: None))
    out = bench.batching_leg(types.SimpleNamespace(synchronize=lambda: None), 4)
    assert len(plans) == 56
    for p in plans:
        assert p.cfg["from"] == (p.dim, p.equal, p.form), p.sym
    assert {k for k in out["mixed"]["tuned"] if k.startswith("dim274")} == {"dim274", "dim274_iii_v"}
