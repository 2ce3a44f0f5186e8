"""The band solves and their consumers that a program built on ultimateepm_amd runs, as measurable cases.

Each case goes through the public Python entry points (``api.Plan.solve``, ``api.Plan.solve_device``,
``mesh.MeshBZ.dos_device``, ``api.dielectric``).  Device buffers are torch tensors: ``solve_device`` and
``dos_device`` take plain device pointers, and torch's default stream is the null stream that they use by default.

Kinds of case:

* ``solve``: k-points and results resident on the device (the bulk form: BZ sampling, mesh vertices);
* ``host``: host arrays in and out (a band path, one k-point of a ``Hamiltonian``);
* ``dos``: tetrahedron density of states of a mesh whose bands are on the device;
* ``dielectric``: the epsilon(q, E) sums, two band solves per q included.

``out`` says what a solve is asked for besides the energies: ``e`` nothing, ``v`` eigenvectors, ``g`` gradients (and
vectors).  An eigenvector's phase is arbitrary, so the program fixes it (``_fix_phase``) in the FP64 form; the
precision form's vectors are accurate to about 1e-6, and the program keeps their plane-wave weights in single
precision (``_weights``).  Spin-orbit cases ask for energies: Kramers pairs leave the vectors of a level free.
"""
from __future__ import annotations

import math
import os

import numpy as np
import torch

import ultimateepm_amd
from ultimateepm_amd import api
from ultimateepm_amd.material import load
from ultimateepm_amd.mesh import MeshBZ

_PARAMS = os.path.join(os.path.dirname(ultimateepm_amd.__file__), "params")
_FILES = {"nonlocal": "materials.yaml", "local": "materials-local-cohen.yaml"}
# plane waves up to |G|^2 <= G2[n - 1] (the reference's shells) for n = 4 .. 16
_SIZE = {4: 27, 5: 51, 6: 59, 7: 65, 8: 89, 9: 113, 10: 137, 11: 169, 12: 181, 13: 229, 14: 259, 15: 283, 16: 307}
_SHELL_G2 = {4: 8, 5: 11, 6: 12, 7: 16, 8: 19, 9: 20, 10: 24, 11: 27, 12: 32, 13: 35, 14: 36, 15: 40, 16: 43}


def _solve(name, material, n, nk, nb, out="e", mixed=False, soc=False, nonlocal_=True, kind="solve"):
    return {"name": name, "kind": kind, "material": material, "n": n, "nonlocal": nonlocal_, "soc": soc,
            "mixed": mixed, "nb": nb, "nk": nk, "out": out}


def listed():
    return [
        # one k-point with vectors and gradients through host arrays: Hamiltonian::SetMatrix + Diagonalize, called in a
        # loop by a program that wants one point at a time; latency
        _solve("point_gaas", "GaAs", 10, 1, 12, out="g", kind="host"),
        # a band path: a few hundred points on straight segments, host arrays, energies only (BandStructure)
        _solve("path_si_local", "Si", 10, 240, 16, nonlocal_=False, kind="host"),
        # the headline workload's form: Si non-local, N = 181, 12 bands and their vectors over BZ samples
        _solve("si_mixed_vectors", "Si", 12, 16001, 12, out="v", mixed=True),
        _solve("si_fp64_vectors", "Si", 12, 6000, 12, out="v"),
        # bands and gradients at mesh vertices (BandsOnBZ): local, 20 levels
        _solve("mesh_si_gradients", "Si", 10, 4913, 20, out="g", nonlocal_=False),
        # a III-V compound (no inversion centre) at the headline's size
        _solve("gaas_mixed_vectors", "GaAs", 12, 8191, 12, out="v", mixed=True),
        # Ge with spin-orbit, dimension 274, 16 levels, in both forms
        _solve("ge_soc_mixed", "Ge", 10, 3000, 16, mixed=True, soc=True),
        _solve("ge_soc_fp64", "Ge", 10, 961, 16, soc=True),
        # a III-V compound with spin-orbit in a large basis (dimension 362)
        _solve("gaas_soc_large", "GaAs", 12, 700, 20, mixed=True, soc=True),
        # many k-points in a small basis, energies only
        _solve("inp_small_fp64", "InP", 6, 20001, 8),
        # density of states of four bands of a mesh of the size of the reference's
        {"name": "dos", "kind": "dos", "cells": 21, "bands": 4, "points": 500},
        # epsilon(q, E) of Si for two q
        {"name": "dielectric_si", "kind": "dielectric", "material": "Si", "n": 8, "nk": 1500, "nq": 2, "nb": 12,
         "energies": 1001},
    ]


def _log(rng, lo, hi):
    """A whole number, uniform in its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    what = rng.random()
    if what < 0.08:
        return {"kind": "dos", "cells": rng.randint(5, 21), "bands": rng.randint(1, 4), "points": _log(rng, 30, 500)}
    if what < 0.16:
        return {"kind": "dielectric", "material": rng.choice(["Si", "GaAs"]), "n": rng.choice([6, 7, 8]),
                "nk": _log(rng, 60, 1500), "nq": rng.randint(1, 2), "nb": rng.randint(6, 14),
                "energies": _log(rng, 60, 1001)}
    soc = rng.random() < 0.35
    material = rng.choice(["Si", "Ge", "GaAs", "GaP"] + ([] if soc else ["InP"]))
    n = rng.choice([6, 7, 8, 9, 10, 11, 12]) if soc else rng.choice(list(_SIZE))
    dim = _SIZE[n] * (2 if soc else 1)
    mixed = rng.random() < 0.5
    out = "e" if soc else rng.choice("eev" if mixed else "evg")
    host = rng.random() < 0.15
    # as many k-points as cost the largest listed case's time, at most
    most = max(8, int((1.2e10 if mixed else 5e9) / (dim**3 + 3e5)))
    nk = _log(rng, 1, 300) if host else _log(rng, 32, 16001)
    return {"kind": "host" if host else "solve", "material": material, "n": n,
            "nonlocal": bool(soc or rng.random() < 0.7), "soc": soc, "mixed": mixed, "nb": rng.randint(2, min(dim, 24)),
            "nk": min(nk, most), "out": out}


# ---------------------------------------------------------------- inputs

def _is_local(case):
    return not case.get("nonlocal", False)


def _material(case):
    return load(case["material"], os.path.join(_PARAMS, _FILES["local" if _is_local(case) else "nonlocal"]))


def _kpoints(case, seed):
    """Uniform points of the first Brillouin zone; for a host path, points on segments between some of them."""
    rs = np.random.RandomState(seed % (1 << 31))
    nk = case["nk"]
    want = nk if case["kind"] != "host" or nk < 8 else 7
    got = np.zeros((0, 3))
    while len(got) < want:
        x = rs.uniform(-1.0, 1.0, size=(2 * want + 16, 3))
        got = np.concatenate([got, x[np.abs(x).sum(axis=1) <= 1.5]])
    got = np.ascontiguousarray(got[:want])
    if want == nk:
        return got
    t = np.linspace(0.0, 6.0, nk)
    i = np.minimum(t.astype(np.int64), 5)
    f = (t - i)[:, None]
    return np.ascontiguousarray(got[i] * (1.0 - f) + got[i + 1] * f)


def _flags(case):
    f = 0
    f |= api.NONLOCAL if case["nonlocal"] else 0
    f |= api.SOC if case["soc"] else 0
    f |= api.MIXED if case["mixed"] else 0
    f |= api.VECTORS if case["out"] in "vg" else 0
    f |= api.GRADIENTS if case["out"] == "g" else 0
    return f


def _phase_vector(dim):
    """Fixed complex numbers of modulus one: a vector's phase is that of its product with them."""
    return np.exp(1j * 2.399963229728653 * np.arange(dim) ** 1.5)


def _fix_phase(vec, p):
    """Each vector times the phase that makes its product with p real and positive."""
    z = (vec * p).sum(axis=-1)
    return vec * (z.conj() / abs(z))[..., None]


def _weights(vec):
    """|c_G|^2 of each plane wave, in single precision."""
    return (vec.real * vec.real + vec.imag * vec.imag).to(torch.float32)


def _mesh(case, seed):
    """A cube of cells**3 cells, six tetrahedra each, with smooth bands and their gradients at its vertices."""
    m, nb = case["cells"], case["bands"]
    side = 1.1e10  # 1/m: about 2 pi / a
    g = np.linspace(-0.5 * side, 0.5 * side, m + 1)
    xyz = np.stack(np.meshgrid(g, g, g, indexing="ij"), axis=-1).reshape(-1, 3)
    i, j, k = (v.reshape(-1) for v in np.meshgrid(*(np.arange(m),) * 3, indexing="ij"))
    node = lambda a, b, c: ((i + a) * (m + 1) + (j + b)) * (m + 1) + (k + c)  # noqa: E731
    corner = {}
    for a in (0, 1):
        for b in (0, 1):
            for c in (0, 1):
                corner[a, b, c] = node(a, b, c)
    tets = []
    for order in ((0, 1, 2), (0, 2, 1), (1, 0, 2), (1, 2, 0), (2, 0, 1), (2, 1, 0)):
        at, path = [0, 0, 0], [corner[0, 0, 0]]
        for axis in order:
            at[axis] = 1
            path.append(corner[tuple(at)])
        tets.append(np.stack(path, axis=-1))
    tet = np.concatenate(tets).astype(np.int32)
    rs = np.random.RandomState(seed % (1 << 31))
    E = np.zeros((len(xyz), nb))
    G = np.zeros((len(xyz), nb, 3))
    for b in range(nb):
        for _ in range(5):
            q = rs.uniform(-2.0, 2.0, 3) * (2 * math.pi / side)
            amp, ph = rs.uniform(0.3, 1.5), rs.uniform(0.0, 2 * math.pi)
            arg = xyz @ q + ph
            E[:, b] += amp * np.cos(arg)
            G[:, b] -= amp * np.sin(arg)[:, None] * q
        E[:, b] += 2.0 * b
    return xyz, tet, E, G


def _dielectric_inputs(case, seed):
    rs = np.random.RandomState((seed + 77) % (1 << 31))
    k = _kpoints(case, seed)
    q = rs.uniform(0.05, 0.25, size=(case["nq"], 3))
    return k, q, np.linspace(0.0, 20.0, case["energies"]), 0.05


# ---------------------------------------------------------------- the pass

_ctx = None


def _context():
    global _ctx
    if _ctx is None:
        torch.zeros(1, device="cuda")
        _ctx = api.Context(0)
    return _ctx


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


def prepare(case, seed):
    ctx = _context()
    if case["kind"] == "dos":
        xyz, tet, E, G = _mesh(case, seed)
        mesh = MeshBZ.from_arrays(ctx, xyz, tet)
        mesh.set_bands(E, G)
        shape = (case["bands"], case["points"])
        return {"case": case, "mesh": mesh, "range": [(float(e.min()), float(e.max())) for e in E.T],
                "energies": torch.zeros(shape, dtype=torch.float64, device="cuda"),
                "dos": torch.zeros(shape, dtype=torch.float64, device="cuda")}
    mat = _material(case) if case["kind"] != "dielectric" else load(case["material"])
    G = api.basis_vectors(case["n"])
    if case["kind"] == "dielectric":
        k, q, en, eta = _dielectric_inputs(case, seed)
        return {"case": case, "plan": api.Plan(ctx, mat, G, api.NONLOCAL | api.VECTORS, case["nb"]), "k": k, "q": q,
                "en": en, "eta": eta}
    plan = api.Plan(ctx, mat, G, _flags(case), case["nb"])
    k, nk, nb = _kpoints(case, seed), case["nk"], case["nb"]
    plan.reserve(nk)
    if case["kind"] == "host":
        return {"case": case, "plan": plan, "k": k, "p": _phase_vector(plan.dim)}
    st = {"case": case, "plan": plan, "k": _dev(k), "p": _dev(_phase_vector(plan.dim)),
          "e": torch.zeros((nk, nb), dtype=torch.float64, device="cuda")}
    if case["out"] in "vg":
        st["v"] = torch.zeros((nk, nb, plan.dim), dtype=torch.complex128, device="cuda")
    if case["out"] == "g":
        st["g"] = torch.zeros((nk, nb, 3), dtype=torch.float64, device="cuda")
    return st


def run(st):
    case = st["case"]
    if case["kind"] == "dos":
        n = case["points"]
        for b, (lo, hi) in enumerate(st["range"]):
            st["mesh"].dos_device(b, n, lo, hi, 1.0, 2.0, False, st["energies"][b].data_ptr(), st["dos"][b].data_ptr())
        return {"energies": st["energies"], "dos": st["dos"]}
    if case["kind"] == "dielectric":
        return {"sums": api.dielectric(st["plan"], st["k"], st["q"], st["en"], st["eta"])}
    plan = st["plan"]
    if case["kind"] == "host":
        e, v, g = plan.solve(st["k"])
        if case["out"] == "e":
            return {"energies": e}
        vec = {"weights": _weights(torch.from_numpy(v))} if case["mixed"] else {"vectors": _fix_phase(v, st["p"])}
        return {"energies": e, **vec, **({"gradients": g} if case["out"] == "g" else {})}
    v, g = st.get("v"), st.get("g")
    plan.solve_device(st["k"].data_ptr(), case["nk"], st["e"].data_ptr(), v.data_ptr() if v is not None else 0,
                      g.data_ptr() if g is not None else 0)
    if v is None:
        return {"energies": st["e"]}
    vec = {"weights": _weights(v)} if case["mixed"] else {"vectors": _fix_phase(v, st["p"])}
    return {"energies": st["e"], **vec, **({"gradients": g} if g is not None else {})}


# ---------------------------------------------------------------- what a pass cannot do without

def _real_share(case):
    """Real operations of the eigen-problem over those of a complex Hermitian one of its dimension: an inversion centre
    (Si, Ge) makes H(k) real symmetric, and with spin-orbit a quaternion matrix of half the dimension."""
    if case["material"] not in ("Si", "Ge"):
        return 1.0
    return 0.5 if case.get("soc") else 0.25


def work(case):
    if case["kind"] == "dos":
        nv, nt = (case["cells"] + 1) ** 3, 6 * case["cells"] ** 3
        # vertices (position, energy, gradient), tetrahedra, the two curves; about a tenth of the tetrahedra are cut by
        # an energy, some 150 operations each
        return {"bytes": case["bands"] * (nv * 56.0 + 16.0 * case["points"]) + 16.0 * nt,
                "flops": case["bands"] * case["points"] * nt * 0.1 * 150.0}
    dim = _SIZE[case["n"]] * (2 if case.get("soc") else 1)
    nb, nk = case["nb"], case["nk"]
    one = _real_share(case) * ((16.0 / 3.0) * dim**3 + 8.0 * dim * dim * nb)
    if case["kind"] == "dielectric":
        pairs = nk * 4.0 * (nb - 4)
        return {"bytes": 24.0 * nk + 8.0 * case["energies"] * (1 + case["nq"]),
                "flops": (1 + case["nq"]) * nk * one + case["nq"] * pairs * (8.0 * dim + 12.0 * case["energies"])}
    out = 8.0 * nb + (16.0 * nb * dim if case["out"] in "vg" else 0.0) + (24.0 * nb if case["out"] == "g" else 0.0)
    return {"bytes": nk * (24.0 + out), "flops": nk * (one if case["out"] != "e" else
                                                       _real_share(case) * (16.0 / 3.0) * dim**3)}


# ---------------------------------------------------------------- the same in plain torch, 64 bits

def _basis(n):
    cut = _SHELL_G2[n]
    m = int(math.ceil(math.sqrt(cut)))
    got = []
    for i in range(-m, m + 1):
        for j in range(-m, m + 1):
            for k in range(-m, m + 1):
                v = (-i + j + k, i - j + k, i + j - k)
                if v[0] * v[0] + v[1] * v[1] + v[2] * v[2] <= cut:
                    got.append(v)
    return np.array(got, dtype=np.int64)


_H = 6.62607015e-34
_QE = 1.602176634e-19
_HBAR = _H / (2.0 * math.pi)
_KIN = _HBAR * _HBAR / (2.0 * 9.1093837015e-31 * _QE)
_BOHR = 5.29177210903e-11


def _sph(l, x):
    """Spherical Bessel function j_l, l = -1 .. 3: the series below x = max(1, l), closed forms above."""
    if l == -1:
        return torch.cos(x) / x
    s, c = torch.sin(x), torch.cos(x)
    if l == 0:
        big = s / x
    elif l == 1:
        big = s / x**2 - c / x
    elif l == 2:
        big = (3.0 / x**2 - 1.0) * s / x - 3.0 * c / x**2
    else:
        big = (15.0 / x**3 - 6.0 / x) * s / x - (15.0 / x**2 - 1.0) * c / x
    term = torch.ones_like(x)
    total = torch.ones_like(x)
    for k in range(1, 24):
        term = term * (-0.5 * x * x) / (k * (2 * l + 2 * k + 1))
        total = total + term
    small = x**l / float(np.prod([2 * i + 1 for i in range(1, l + 1)] or [1])) * total
    return torch.where(x < max(1, l), small, big)


def _radial(nK, R, l):
    """Integral of j_l(K1 r) j_l(K2 r) r^2 over [0, R] for every pair of norms."""
    x = nK * R
    jm, j0, jp = _sph(l - 1, x), _sph(l, x), _sph(l + 1, x)
    a, b = nK[:, :, None], nK[:, None, :]
    same = (a - b).abs() <= 1e-4
    den = torch.where(same, torch.ones_like(a * b), a * a - b * b)
    apart = R * R / den * (a * jp[:, :, None] * j0[:, None, :] - b * jp[:, None, :] * j0[:, :, None])
    equal = (0.5 * R**3 * (j0 * j0 - jm * jp))[:, :, None].expand_as(apart)
    return torch.where(same, equal, apart)


def _hamiltonian(mat, G, k, nonlocal_, soc):
    """H(k) (nk, dim, dim) of the k-points k (nk, 3), both torch, in 64 bits."""
    a = 1e-10 * mat.lattice_constant
    four = 2.0 * math.pi / a
    Gd = G.to(torch.float64)
    N = len(G)
    D = G[:, None, :] - G[None, :, :]
    D2 = (D * D).sum(-1)
    arg = (2.0 * math.pi / 8.0) * D.sum(-1).to(torch.float64)
    V = torch.zeros((N, N), dtype=torch.complex128, device=k.device)
    for g2, vs, va in zip((3, 4, 8, 11), mat.V_S, mat.V_A):
        V = torch.where(D2 == g2, torch.complex(vs * torch.cos(arg), va * torch.sin(arg)), V)
    kG = k[:, None, :] + Gd[None]
    H = V[None].repeat(len(k), 1, 1)
    H += torch.diag_embed(four * four * _KIN * (kG * kG).sum(-1)).to(torch.complex128)
    if nonlocal_:
        K = kG * four
        nK = K.norm(dim=-1)
        p = mat.non_local
        omega = a**3 / 8.0
        kF = (96.0 * math.pi**2) ** (1.0 / 3.0) / a
        nn = nK[:, :, None] * nK[:, None, :]
        cosang = (K @ K.transpose(1, 2)) / nn
        leg2 = 0.5 * (3.0 * cosang * cosang - 1.0)
        side = []
        for al, be, A2, R0, R2 in ((p.alpha_0_anion, p.beta_0_anion, p.A2_anion, p.R0_anion, p.R2_anion),
                                   (p.alpha_0_cation, p.beta_0_cation, p.A2_cation, p.R0_cation, p.R2_cation)):
            W = torch.zeros_like(nn)
            if R0 != 0.0 and (al != 0.0 or be != 0.0):
                W = W + 4.0 * math.pi / omega * (al + _KIN * be * (nn - kF * kF)) * _radial(nK, R0, 0)
            if A2 != 0.0 and p.well_type == "square":
                W = W + 4.0 * math.pi / omega * A2 * 5.0 * leg2 * _radial(nK, R2, 2)
            elif A2 != 0.0:
                x = 0.5 * R2 * R2 * nn
                i2 = ((x * x + 3.0) * torch.sinh(x) - 3.0 * x * torch.cosh(x)) / x**3
                gauss = torch.exp(-0.25 * R2 * R2 * (nK[:, :, None] ** 2 + nK[:, None, :] ** 2))
                W = W + 5.0 * math.pi**1.5 * R2**3 / omega * A2 * leg2 * i2 * gauss
            side.append(W)
        th = (2.0 * math.pi / 8.0) * D.sum(-1).to(torch.float64)[None]
        H += torch.complex(torch.cos(th) * (side[0] + side[1]) / 2.0, torch.sin(th) * (side[0] - side[1]) / 2.0)
    if soc:
        s = mat.spin_orbit
        nK = kG.norm(dim=-1) * four

        def shape(period, xi):
            x2 = (nK * _BOHR / xi) ** 2
            q = 1.0 + x2
            return 1.0 / q**3 if period == 2 else (5.0 - x2) / (5.0 * q**4) if period == 3 else \
                (5.0 - 3.0 * x2) / (5.0 * q**5)

        Bc, Ba = shape(s.period_cation, s.radial_extent_cation), shape(s.period_anion, s.radial_extent_anion)
        l1 = s.mu * Bc[:, :, None] * Bc[:, None, :]
        l2 = s.alpha * s.mu * Ba[:, :, None] * Ba[:, None, :]
        f = torch.complex((l1 - l2) / 2.0 * torch.sin(arg)[None], -(l1 + l2) / 2.0 * torch.cos(arg)[None])
        x, y, z = (kG[..., c] for c in range(3))
        cz = x[:, :, None] * y[:, None, :] - y[:, :, None] * x[:, None, :]
        cx = y[:, :, None] * z[:, None, :] - z[:, :, None] * y[:, None, :]
        cy = x[:, :, None] * z[:, None, :] - z[:, :, None] * x[:, None, :]
        up = torch.cat([H + cz * f, torch.complex(cx, cy) * f], dim=2)
        down = torch.cat([torch.complex(cx, -cy) * f, H - cz * f], dim=2)
        H = torch.cat([up, down], dim=1)
    return 0.5 * (H + H.transpose(1, 2).conj())


def _pairs(mat, n, k, nonlocal_, soc, nb, vectors):
    """The lowest nb eigenpairs (vectors as rows) of every k-point, as numpy arrays."""
    at = "cuda" if torch.cuda.is_available() else "cpu"
    G = torch.from_numpy(_basis(n)).to(at)
    dim = len(G) * (2 if soc else 1)
    step = max(1, int(6e7) // (dim * dim))
    E, X = [], []
    for c in range(0, len(k), step):
        for h in _hamiltonian(mat, G, torch.from_numpy(k[c:c + step]).to(at), nonlocal_, soc).cpu().numpy():
            if vectors:
                w, x = np.linalg.eigh(h)
                X.append(x[:, :nb].T)
            else:
                w = np.linalg.eigvalsh(h)
            E.append(w[:nb])
    return np.stack(E), np.stack(X) if vectors else None


def _exact_dos(case, seed):
    xyz, tet, E, G = _mesh(case, seed)
    at = "cuda" if torch.cuda.is_available() else "cpu"
    P = torch.from_numpy(xyz).to(at)[torch.from_numpy(tet).to(at).long()]
    en = np.zeros((case["bands"], case["points"]))
    dos = np.zeros_like(en)
    for b in range(case["bands"]):
        lo, hi = float(E[:, b].min()), float(E[:, b].max())
        step = (hi - lo) / (case["points"] - 1)
        e = torch.from_numpy(np.ascontiguousarray(E[:, b])).to(at)[torch.from_numpy(tet).to(at).long()]
        g = torch.from_numpy(np.ascontiguousarray(G[:, b])).to(at)[torch.from_numpy(tet).to(at).long()]
        e, order = torch.sort(e, dim=1, stable=True)
        pick = order[..., None].expand(-1, -1, 3)
        p, g = torch.gather(P, 1, pick), torch.gather(g, 1, pick)
        for i in range(case["points"]):
            x = lo + i * step
            en[b, i] = x
            total = 0.0
            # corners of the cut as (lower vertex, upper vertex), cyclic
            for edges, inside in ((((0, 1), (0, 2), (0, 3)), (x >= e[:, 0]) & (x < e[:, 1])),
                                  (((0, 2), (0, 3), (1, 3), (1, 2)), (x >= e[:, 1]) & (x < e[:, 2])),
                                  (((2, 3), (1, 3), (0, 3)), (x >= e[:, 2]) & (x <= e[:, 3]))):
                at_ = inside.nonzero()[:, 0]
                if not len(at_):
                    continue
                ee, pp, gg = e[at_], p[at_], g[at_]
                pts, inv = [], 0.0
                for u, v in edges:
                    t = ((x - ee[:, u]) / (ee[:, v] - ee[:, u]))[:, None]
                    pts.append(pp[:, u] + t * (pp[:, v] - pp[:, u]))
                    inv = inv + 1.0 / (gg[:, u] + t * (gg[:, v] - gg[:, u])).norm(dim=1).clamp_min(1e-12)
                if len(pts) == 3:
                    area = torch.linalg.cross(pts[1] - pts[0], pts[2] - pts[0])
                else:
                    area = torch.linalg.cross(pts[2] - pts[0], pts[3] - pts[1])
                one = 0.5 * area.norm(dim=1) * inv / len(pts)
                total += float(one[torch.isfinite(one)].sum())
            dos[b, i] = 2.0 * total / (8.0 * math.pi**3)
    return {"energies": en, "dos": dos}


def exact(case, seed):
    if case["kind"] == "dos":
        return _exact_dos(case, seed)
    if case["kind"] == "dielectric":
        k, q, en, eta = _dielectric_inputs(case, seed)
        mat = load(case["material"])
        E, X = _pairs(mat, case["n"], k, True, False, case["nb"], True)
        sums = np.zeros((case["nq"], case["energies"]))
        for i in range(case["nq"]):
            Eq, Xq = _pairs(mat, case["n"], k + q[i], True, False, case["nb"], True)
            w = np.abs(np.matmul(Xq[:, 4:], X[:, :4].transpose(0, 2, 1))) ** 2
            d = Eq[:, 4:, None] - E[:, None, :4]
            w, d = w.reshape(-1), d.reshape(-1)
            for j, x in enumerate(en):
                sums[i, j] = np.sum(w * ((d - x) / ((d - x) ** 2 + eta * eta) + (d + x) / ((d + x) ** 2 + eta * eta)))
        return {"sums": sums}
    dim = _SIZE[case["n"]] * (2 if case["soc"] else 1)
    vectors = case["out"] in "vg"
    if case["nk"] * dim**3 > 2e10:
        return None  # over twenty seconds
    mat = _material(case)
    k = _kpoints(case, seed)
    E, X = _pairs(mat, case["n"], k, case["nonlocal"], case["soc"], case["nb"], vectors)
    if not vectors:
        return {"energies": E}
    if case["mixed"]:
        got = {"energies": E, "weights": (X.real**2 + X.imag**2)}
    else:
        got = {"energies": E, "vectors": _fix_phase(X, _phase_vector(dim))}
    if case["out"] == "g":
        four = 2.0 * math.pi / (1e-10 * mat.lattice_constant)
        kG = k[:, None, :] + _basis(case["n"])[None]
        got["gradients"] = 2.0 * _KIN * four * np.einsum("kgc,kbg->kbc", kG, np.abs(X) ** 2)
    return got
