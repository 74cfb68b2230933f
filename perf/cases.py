"""Performance cases: calls a user of the framework makes, with their inputs,
their work, their tolerances and their values in 64 bits.

A case is one call of the k-mesh path through ``rustb_amd.Model``: a tight
binding model (seeded random hoppings that decay with |R|, as the framework's
own workloads have them) and the call's arguments.  ``kind`` names the call:

  onek   solve_onek: the eigenpairs of one k-point
  dos    dos: Gaussian density of states on a mesh (graphene)
  bands  solve_band_all: eigenvalues along a k-path
  berry  berry_curvature_on: Omega_n and E_n along a k-path
  hall   hall_conductivity, Direct integration on a mesh
  ecut   hall_conductivity, EnergyCut integration on a mesh
  dipole extrinsic_nonlinear_hall on a mesh

Model fields: dim, spin, norb, rmax (|R_i| <= rmax), layers (> 1: a slab of
that many layers of norb orbitals each), printed (the storage as read from a
file with six decimals: ham[-R] equals ham[R]^H only to the last digit).
"""
from __future__ import annotations

import math
import os
from concurrent.futures import ThreadPoolExecutor

import numpy as np

import rustb_amd as ra

KB = 8.617333262145e-5  # eV/K
DOS_RANGE, DOS_SIGMA = (-4.0, 4.0), 0.02  # the graphene workload's window and smearing
SQ3 = math.sqrt(3.0)


def _case(name, kind, **kw):
    c = dict(kind=kind, dim=2, spin=False, norb=1, rmax=1, layers=1, printed=False, nk=0, n1=1, n2=1, n3=1, n_mu=1,
             T=0.0, eta=1e-3, precision="fp64", spin_dir="", n_e=0)
    c.update(kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call: one k-point's eigenpairs of a small model (an
        # interactive look, or an optimiser's inner step)
        _case("onek_n8", "onek", spin=True, norb=4, rmax=1, nk=1),
        # the textbook call: graphene's density of states on 101 x 101
        _case("dos_graphene", "dos", norb=2, n1=101, n2=101, n_e=801),
        # a band structure plot of a mid-size 3D spinful model
        _case("bands_n36", "bands", dim=3, spin=True, norb=18, rmax=2, nk=301),
        # Berry curvature along a k-path of a model read from a file
        _case("berry_n72", "berry", dim=3, spin=True, norb=36, rmax=3, printed=True, nk=401),
        # two-band anomalous Hall conductivity (Haldane-sized models), a few
        # chemical potentials
        _case("hall_n2", "hall", norb=2, rmax=1, n1=101, n2=99, n_mu=5),
        # the random3d-n32 workload's model and mesh: sigma(mu) at room
        # temperature
        _case("hall_n32_mixed", "hall", dim=3, spin=True, norb=16, rmax=2, n1=64, n2=64, n3=64, n_mu=41, T=300.0,
              precision="mixed"),
        # a model read from a file, plain FP64, ragged mesh, sizes off the tiles
        _case("hall_n50_fp64", "hall", dim=3, spin=True, norb=25, rmax=3, printed=True, n1=17, n2=13, n3=11, n_mu=3),
        # the headline workload: wannier3d-n128 on 48^3
        _case("hall_n128_mixed", "hall", dim=3, spin=True, norb=64, rmax=5, n1=48, n2=48, n3=48, eta=1e-4,
              precision="mixed"),
        # a thin film: 32 layers x 8 orbitals (the slab workload's model)
        _case("slab_n256_mixed", "hall", norb=8, layers=32, rmax=3, n1=48, n2=50, eta=1e-4, precision="mixed"),
        # EnergyCut in 2D: the benchmark's random2d-n32 sizes
        _case("ecut2d_n32", "ecut", norb=32, rmax=3, n1=128, n2=128, n_mu=41),
        # EnergyCut in 3D at a finite temperature, a spin Hall current
        _case("ecut3d_n12", "ecut", dim=3, spin=True, norb=6, rmax=1, n1=20, n2=18, n3=16, n_mu=11, T=100.0,
              spin_dir="Z"),
        # Berry curvature dipole response at room temperature
        _case("dipole_n44_mixed", "dipole", dim=3, spin=True, norb=22, rmax=2, n1=15, n2=14, n3=13, n_mu=9, T=300.0,
              precision="mixed"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _mesh(rng, dim, nk):
    """A mesh of about nk points, its axes a little uneven."""
    side = max(2.0, nk ** (1.0 / dim))
    n = [max(2, int(round(side * rng.uniform(0.8, 1.2)))) for _ in range(dim)]
    return dict(n1=n[0], n2=n[1], n3=n[2] if dim == 3 else 1)


def draw(rng):
    kind = rng.choice(["onek", "dos", "bands", "berry", "hall", "hall", "hall", "hall", "slab", "ecut", "ecut", "dipole"])
    if kind == "dos":
        return _case("", "dos", norb=2, n1=_log_int(rng, 40, 200), n2=_log_int(rng, 40, 200), n_e=_log_int(rng, 200, 1600))
    if kind == "slab":
        layers = rng.randint(17, 32)
        return _case("", "hall", norb=8, layers=layers, rmax=3, n1=rng.randint(16, 40), n2=rng.randint(16, 40), eta=1e-4,
                     precision=rng.choice(["mixed", "mixed", "fp64"]))
    dim = rng.choice([2, 3])
    spin = rng.random() < 0.5
    if kind == "ecut":
        norb = _log_int(rng, 2, 40 if dim == 2 else 20)
        n = 2 * norb if spin else norb
        nk = _log_int(rng, 600, max(700, min(16384, int(16384 * (32.0 / n) ** 2)) if dim == 2 else min(8000, 10 ** 6 // n ** 2 * 4)))
        return _case("", "ecut", dim=dim, spin=spin, norb=norb, rmax=rng.randint(1, 3 if dim == 2 else 1),
                     n_mu=_log_int(rng, 1, 41), T=rng.choice([0.0, 0.0, 150.0]),
                     spin_dir=rng.choice(["", "X", "Z"]) if spin else "", **_mesh(rng, dim, nk))
    norb = _log_int(rng, 2, 64)
    n = 2 * norb if spin else norb
    rmax = rng.randint(1, 4 if dim == 2 else 3)
    printed = rng.random() < 0.3
    prec = rng.choice(["fp64", "mixed"])
    if kind == "onek":
        return _case("", "onek", dim=dim, spin=spin, norb=norb, rmax=min(rmax, 2), nk=1, precision=prec)
    if kind in ("bands", "berry"):
        return _case("", kind, dim=dim, spin=spin, norb=norb, rmax=rmax, printed=printed, nk=_log_int(rng, 50, 800),
                     precision=prec if kind == "berry" else "fp64")
    if kind == "dipole":
        norb = min(norb, 48)
        n = 2 * norb if spin else norb
        nk = _log_int(rng, 200, max(300, min(20000, int(4000 * (64.0 / n) ** 2))))
        return _case("", "dipole", dim=dim, spin=spin, norb=norb, rmax=min(rmax, 2), n_mu=_log_int(rng, 1, 21), T=300.0,
                     precision=prec, **_mesh(rng, dim, nk))
    nk = _log_int(rng, 400, max(600, min(200000, int((20000 if prec == "mixed" else 4000) * (64.0 / n) ** 2))))
    return _case("", "hall", dim=dim, spin=spin, norb=norb, rmax=rmax, printed=printed, n_mu=_log_int(rng, 1, 41),
                 T=rng.choice([0.0, 300.0]), eta=rng.choice([1e-3, 1e-3, 1e-2]), precision=prec,
                 spin_dir=rng.choice(["", "", "X", "Y", "Z"]) if spin else "", **_mesh(rng, dim, nk))


# ------------------------------------------------------------ inputs
def _n(case):
    return case["norb"] * case["layers"] * (2 if case["spin"] else 1)


def _n_R(case):
    return 5 if case["kind"] == "dos" else (2 * case["rmax"] + 1) ** case["dim"]


def _kmesh(case):
    return tuple(case[a] for a in ("n1", "n2", "n3")[:case["dim"]])


def _nk(case):
    return case["nk"] or int(np.prod(_kmesh(case)))


def _storage(case, seed):
    """lat, orb, hamR, ham of the case's model: R = 0 first, then R and -R in
    turn, ham[-R] = ham[R]^H."""
    g = np.random.default_rng([seed, 11])
    dim, n, rmax = case["dim"], _n(case), case["rmax"]
    if case["kind"] == "dos":  # graphene: two sites, three nearest-neighbour hoppings, a small site splitting
        t = -2.85 * (1.0 + 0.1 * g.uniform(-1.0, 1.0, 3))
        gap = 0.2 * g.uniform(0.2, 1.0)
        hamR = np.array([[0, 0], [1, 0], [-1, 0], [0, 1], [0, -1]], np.int64)
        ham = np.zeros((5, 2, 2), np.complex128)
        ham[0] = [[gap, t[0]], [t[0], -gap]]
        for r, a in ((2, t[1]), (4, t[2])):  # add_hop(t, 0, 1, -R) and its conjugate at +R
            ham[r, 0, 1] = a
            ham[r - 1, 1, 0] = a
        return np.array([[SQ3, -1.0], [SQ3, 1.0]]), np.array([[0.0, 0.0], [1.0 / 3.0, 1.0 / 3.0]]), hamR, ham
    grids = np.meshgrid(*[np.arange(-rmax, rmax + 1)] * dim, indexing="ij")
    allR = np.stack([x.reshape(-1) for x in grids], axis=1)
    half = allR[len(allR) // 2 + 1:]  # lexicographic order: the second half is minus the first
    hamR = np.zeros((2 * len(half) + 1, dim), np.int64)
    hamR[1::2], hamR[2::2] = half, -half
    norb = case["norb"] * case["layers"]
    scale, decay = (0.5, 1.0) if case["layers"] == 1 and n <= 64 else (1.0, 1.5 if dim == 3 else 1.0)
    amp = scale * np.exp(-np.linalg.norm(half, axis=1) / decay) * math.sqrt(0.5)
    up = g.standard_normal((len(half), n, 2 * n)).view(np.complex128) * amp[:, None, None]
    on = g.standard_normal((n, 2 * n)).view(np.complex128) * (scale * math.sqrt(0.5))
    if case["layers"] > 1:  # in-plane hoppings stay in a layer; layers couple at R = 0, halving per layer
        layer = np.repeat(np.arange(case["layers"]), case["norb"])
        dl = np.abs(layer[:, None] - layer[None, :])
        up *= dl == 0
        on *= np.where(dl == 0, 0.1, 0.3 * 0.5 ** np.maximum(dl - 1, 0))
    on = np.triu(on, 1)
    ham = np.zeros((2 * len(half) + 1, n, n), np.complex128)
    ham[0] = on + on.conj().T + np.diag(g.uniform(-1.0, 1.0, n))
    ham[1::2], ham[2::2] = up, up.conj().transpose(0, 2, 1)
    if case["printed"]:  # each entry printed by itself from values that differ in the last digits
        x = ham.view(np.float64)
        x += g.uniform(-1e-7, 1e-7, x.shape)
        np.round(x, 6, out=x)
    lat = np.eye(dim) * g.uniform(2.0, 4.0, dim) + g.uniform(-0.3, 0.3, (dim, dim))
    return lat, g.uniform(0.0, 1.0, (norb, dim)), hamR, ham


def _call(case, seed):
    """k-points, chemical potentials and directions of the call."""
    g = np.random.default_rng([seed, 12])
    dim = case["dim"]
    nodes = g.uniform(-0.5, 0.5, (4, dim))
    f = np.linspace(0.0, 3.0, max(case["nk"], 1))
    i = np.minimum(f.astype(int), 2)
    ks = nodes[i] + (f - i)[:, None] * (nodes[i + 1] - nodes[i])
    half = 0.35 * math.sqrt(_n(case)) if case["layers"] == 1 else 1.0
    mu = np.sort(g.uniform(-half, half, case["n_mu"]))
    dirs = np.eye(3)[:3, :dim] + g.uniform(-0.1, 0.1, (3, dim))
    if dim == 2:
        dirs[2] = dirs[0] + dirs[1]
    return ks, mu, dirs


def prepare(case, seed):
    lat, orb, hamR, ham = _storage(case, seed)
    ks, mu, dirs = _call(case, seed)
    if case["kind"] == "dos":
        m = ra.Model.tb_model(lat, orb, False)
        m.set_onsite([ham[0, 0, 0].real, ham[0, 1, 1].real])
        for r in (0, 2, 4):
            m.add_hop(ham[r, 0, 1].real, 0, 1, hamR[r])
    else:
        m = ra.Model.from_arrays(lat, orb, case["spin"], hamR, ham)
    m.gen_ham(np.zeros(case["dim"]))  # the model is on the GPU from its first use on
    rows = dirs if case["kind"] == "dipole" else dirs[:2]
    p = ra.Parameters(kmesh=_kmesh(case), direction=rows, mu=mu, T=np.array([case["T"]]), eta=case["eta"],
                      spin=case["spin_dir"] or None, integration="EnergyCut" if case["kind"] == "ecut" else "Direct",
                      precision=case["precision"])
    return dict(case=case, model=m, params=p, ks=ks)


def run(state):
    case, m, p = state["case"], state["model"], state["params"]
    kind = case["kind"]
    if kind == "onek":
        E, V = m.solve_onek(state["ks"][0], case["precision"])
        # a program that compares or interpolates eigenvectors fixes their
        # phases: the sum of each one's components real and positive
        s = V.sum(axis=1)
        return E, V * (np.conj(s) / np.abs(s))[:, None]
    if kind == "dos":
        return m.dos(_kmesh(case), *DOS_RANGE, case["n_e"], DOS_SIGMA, case["precision"])
    if kind == "bands":
        return m.solve_band_all(state["ks"], case["precision"])
    if kind == "berry":
        return m.berry_curvature_on(state["ks"], p)
    if kind == "dipole":
        return m.extrinsic_nonlinear_hall(p).conductivity
    return m.hall_conductivity(p).conductivity


# ------------------------------------------------------------ work and tolerance
def work(case):
    n, nk, kind, dim = float(_n(case)), float(_nk(case)), case["kind"], case["dim"]
    model = _n_R(case) * n * n * 16.0
    # H and d velocities: 8 flop per element, operator and term; on a mesh the
    # sum separates by axis, and the last axis is what every k-point pays
    nv = {"onek": 0, "dos": 0, "bands": 0, "dipole": 3}.get(kind, 2)
    terms = _n_R(case) if case["nk"] else 2.0 * case["rmax"] + 1.0
    per_k = 8.0 * terms * n * n * (1 + nv) + 16.0 / 3.0 * n ** 3
    out = n * 8.0 * nk
    if kind == "onek":
        per_k += 8.0 * n ** 3
        out += n * n * 16.0
    elif kind == "dos":
        per_k += 10.0 * n * case["n_e"]
        out = 16.0 * case["n_e"]
    elif kind != "bands":
        # eigenvectors, then U^H v U per operator
        per_k += 8.0 * n ** 3 + 16.0 * n ** 3 * nv
        if kind == "berry":
            out *= 2.0
        else:
            out = 8.0 * case["n_mu"]
        if kind == "ecut":  # overlaps with the next neighbour of each axis
            per_k += 8.0 * n ** 3 * dim
    return {"bytes": model + out + 24.0 * nk * (case["nk"] > 0), "flops": per_k * nk}


def tolerance(case):
    """About four times the largest difference seen over seeds and draws: from
    exact(), for the largest mixed calls from the FP64 form, for EnergyCut
    from a call on hoppings moved in their last bit."""
    kind, mixed = case["kind"], case["precision"] == "mixed"
    if kind in ("dos", "bands"):
        return {"rel": 3e-14, "max": 1e-13}
    if kind == "onek":  # eigenvectors: rounding over the gaps of one k-point
        return {"rel": 4e-10, "max": 5e-9} if mixed else {"rel": 2e-13, "max": 2e-12}
    if kind == "ecut":
        return {"rel": 1e-11, "max": 1e-10}
    # band sums hold 1 / (E_n - E_m)^2: an energy's rounding counts by the
    # narrowest gap the k-points meet, a slab's cancel the most
    if not mixed:
        return {"rel": 1e-11, "max": 2e-11}
    return {"rel": 8e-8, "max": 8e-8} if _n(case) > 128 else {"rel": 2.5e-9, "max": 2.6e-8}


# ------------------------------------------------------------ values in 64 bits
def _bloch(case, store, ks, dirs):
    """H(k) and the projected velocities (Atom gauge), from the literal sum."""
    lat, orb, hamR, ham = store
    n = _n(case)
    U = np.exp(2j * np.pi * (ks @ hamR.T))
    wR = dirs @ (hamR @ lat).T
    tau = np.concatenate([orb] * (2 if case["spin"] else 1))
    wt = dirs @ (tau @ lat).T
    ph = np.exp(2j * np.pi * (ks @ tau.T))
    gauge = np.conj(ph)[:, :, None] * ph[:, None, :]
    flat = ham.reshape(len(hamR), -1)
    Hl = (U @ flat).reshape(-1, n, n)
    vs = []
    for p in range(len(dirs)):
        d = ((U * wR[p]) @ flat).reshape(-1, n, n)
        vs.append(1j * (d + (wt[p][None, None, :] - wt[p][None, :, None]) * Hl) * gauge)
    return Hl * gauge, vs


def _hermitian(H, upper):
    """The matrix of H's upper (lower) triangle and Re of its diagonal."""
    t = np.triu(H, 1) if upper else np.tril(H, -1)
    t = t + np.conj(t.transpose(0, 2, 1))
    i = np.arange(H.shape[1])
    t[:, i, i] = H[:, i, i].real
    return t


def _spin_current(case, v):
    s = {"X": [[0, 1], [1, 0]], "Y": [[0, -1j], [1j, 0]], "Z": [[1, 0], [0, -1]]}[case["spin_dir"]]
    S = np.kron(0.5 * np.array(s, np.complex128), np.eye(case["norb"]))
    return 0.5 * (S @ v + v @ S)


def _omega(A, B, E, eta):
    d = E[:, :, None] - E[:, None, :]
    w = 1.0 / (d * d + eta * eta)
    i = np.arange(E.shape[1])
    w[:, i, i] = 0.0
    return -2.0 * ((A * B.transpose(0, 2, 1)).imag * w).sum(axis=2)


def _fermi(E, mu, T):
    if T == 0.0:
        return np.where(E < mu, 1.0, np.where(E > mu, 0.0, 0.5))
    return 1.0 / (1.0 + np.exp(np.clip((E - mu) / (T * KB), -700.0, 700.0)))


def _part(case, store, ks, mu, dirs):
    """The part of the result a few k-points give."""
    kind = case["kind"]
    H, vs = _bloch(case, store, ks, dirs[:0] if kind in ("onek", "dos", "bands") else dirs)
    if kind in ("dos", "bands"):
        return np.linalg.eigvalsh(_hermitian(H, False))
    E, U = np.linalg.eigh(_hermitian(H, True))
    if kind == "onek":
        V = U.transpose(0, 2, 1)[0]  # eigenvectors as rows
        s = V.sum(axis=1)
        return E[0], V * (np.conj(s) / np.abs(s))[:, None]
    Uh = np.conj(U.transpose(0, 2, 1))
    ops = [Uh @ v @ U for v in ([_spin_current(case, vs[0])] + vs[1:] if case["spin_dir"] else vs)]
    om = _omega(ops[0], ops[1], E, case["eta"])
    if kind == "berry":
        return om, E
    if kind == "dipole":
        om2 = _omega(ops[0], ops[2], E, case["eta"])
        i = np.arange(E.shape[1])
        kern = 0.5 * (om * ops[2][:, i, i].real + om2 * ops[1][:, i, i].real)
        out = []
        for m in mu:
            f = _fermi(E, m, case["T"])
            out.append((kern * f * (1.0 - f) / (case["T"] * KB)).sum())
        return np.array(out)
    return np.array([(om * _fermi(E, m, case["T"])).sum() for m in mu])


def exact(case, seed):
    n, nk, kind = _n(case), _nk(case), case["kind"]
    # EnergyCut: the tracking walk and the per-simplex cut in plain Python
    # take minutes; the rest in proportion to its dense sums and products
    if kind == "ecut" or nk * (60.0 * n ** 3 + 8.0 * _n_R(case) * n * n + 5e5) > 6e11:
        return None
    store = _storage(case, seed)
    ks, mu, dirs = _call(case, seed)
    dirs = dirs if kind == "dipole" else dirs[:2]
    if not case["nk"]:
        km = _kmesh(case)
        ks = np.stack([x.reshape(-1) for x in np.meshgrid(*[np.arange(m) / m for m in km], indexing="ij")], axis=1)
    per = max(1, min(512, int(2e6 / (n * n))))
    with ThreadPoolExecutor(min(8, os.cpu_count() or 1)) as pool:
        parts = list(pool.map(lambda i: _part(case, store, ks[i:i + per], mu, dirs), range(0, nk, per)))
    if kind == "onek":
        return parts[0]
    if kind == "bands":
        return np.concatenate(parts)
    if kind == "berry":
        return tuple(np.concatenate(x) for x in zip(*parts))
    if kind == "dos":
        E, sigma = np.linspace(*DOS_RANGE, case["n_e"]), DOS_SIGMA
        ev = np.concatenate(parts).reshape(-1)
        rho = sum(np.exp(-0.5 * ((E[:, None] - e[None, :]) / sigma) ** 2).sum(axis=1) for e in np.array_split(ev, 64))
        return E, rho / (sigma * math.sqrt(2.0 * math.pi)) / nk
    return np.sum(parts, axis=0) / nk / np.linalg.det(store[0])
