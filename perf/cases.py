"""The work that a user of the grid solver has it do, as cases that can be timed.

Kinds of cases:

* ``response``: the material law on trial deformation fields that live on the
  GPU (``dmk_constitutive_device``), as an outer program's iteration calls it;
* ``increment``: one load increment of an RVE through the solver plug-in
  (``forward``, ``solution``) and its results in host arrays
  (``dmk_mech_get_field``), for the three schemes;
* ``divergence``: the equilibrium norm of a device field without allocation
  (``dmk_divergence_rms_noalloc``);
* ``gradient``: the reverse sweep over recorded increments
  (``adjoint_backward``).

A case is a dict of plain values; ``x``, ``y``, ``z`` are the cells per axis.
"""
import copy
import ctypes
import math

import numpy as np
import torch

from damask_amd import _lib, config, workloads
from damask_amd.geom import Grid
from damask_amd.grid import FIELDS, GridMechSpectralBasic, grid_mechanical

DT = 0.5            # s per increment: 5e-4 strain at 1e-3/s, as in the 64^3 tension to 5 % in 100 increments
PATH_STEPS = 6      # increments of the strain path before a response case's trial fields (into plastic flow)
LOAD_STEPS = 4      # increments of the load case before an increment case's own one (into plastic flow)
TRIALS = 3          # trial fields of one response pass


def listed():
    return [
        # a single small RVE per call, as in parameter studies: launches and synchronisations count
        {"name": "response 8 fcc", "kind": "response", "phase": "fcc", "x": 8, "y": 8, "z": 8, "grains": 12},
        # the material law at the size of the headline RVE
        {"name": "response 64 fcc", "kind": "response", "phase": "fcc", "x": 64, "y": 64, "z": 64, "grains": 200},
        # a free stress exponent (fitted parameters), 24 slip systems, an odd grid
        {"name": "response 31x45x27 bcc", "kind": "response", "phase": "bcc", "n": 17.3, "x": 31, "y": 45, "z": 27,
         "grains": 50},
        # two phases in one grid (ferrite and a cF phase), non-Schmid terms in the cI one
        {"name": "response 48 dual", "kind": "response", "phase": "dual", "x": 48, "y": 48, "z": 48, "grains": 100},
        # the smoke-sized RVE of a parameter study: one increment
        {"name": "increment 16 fcc", "kind": "increment", "scheme": "spectral_basic", "phase": "fcc", "x": 16, "y": 16,
         "z": 16, "grains": 20},
        # the headline workload's increment
        {"name": "increment 64 fcc", "kind": "increment", "scheme": "spectral_basic", "phase": "fcc", "x": 64, "y": 64,
         "z": 64, "grains": 200},
        # a measured microstructure's odd grid, 24 slip systems
        {"name": "increment 45x50x54 bcc", "kind": "increment", "scheme": "spectral_basic", "phase": "bcc", "x": 45,
         "y": 50, "z": 54, "grains": 100},
        # a large RVE
        {"name": "increment 128 fcc", "kind": "increment", "scheme": "spectral_basic", "phase": "fcc", "x": 128,
         "y": 128, "z": 128, "grains": 500},
        # the reference's two other schemes at an ordinary size
        {"name": "increment 32 polarization", "kind": "increment", "scheme": "spectral_polarization", "phase": "fcc",
         "x": 32, "y": 32, "z": 32, "grains": 50},
        {"name": "increment 36x40x30 Galerkin", "kind": "increment", "scheme": "spectral_Galerkin", "phase": "fcc",
         "x": 36, "y": 40, "z": 30, "grains": 50},
        # an outer loop's equilibrium check between its own steps
        {"name": "divergence 64x60x63", "kind": "divergence", "x": 64, "y": 60, "z": 63},
        # the differentiation workload: gradient of a stress-strain curve with respect to the parameters
        {"name": "gradient 32 fcc", "kind": "gradient", "phase": "fcc", "x": 32, "y": 32, "z": 32, "grains": 50,
         "increments": 3},
    ]


def draw(rng):
    def edge(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["response", "response", "increment", "increment", "increment", "divergence", "gradient"])
    top = {"response": 72, "increment": 80, "divergence": 64, "gradient": 28}[kind]
    x = edge(6, top)
    # cubes and boxes: the other edges within a factor of about 1.5
    y, z = (x, x) if rng.random() < 0.4 else (min(top, edge(max(5, x / 1.5), x * 1.5)) for _ in range(2))
    case = {"kind": kind, "x": x, "y": y, "z": z}
    if kind == "divergence":
        return case
    case["grains"] = rng.randint(5, 200)
    case["phase"] = "fcc"
    if kind == "response":
        case["phase"] = rng.choice(["fcc", "bcc", "dual"])
    elif kind == "increment":
        case["scheme"] = rng.choice(["spectral_basic"] * 4 + ["spectral_polarization", "spectral_Galerkin"])
        if case["scheme"] == "spectral_basic":
            case["phase"] = rng.choice(["fcc", "fcc", "bcc"])
        else:
            case["x"], case["y"], case["z"] = (min(40, v) for v in (x, y, z))
    else:
        case["increments"] = rng.randint(2, 4)
    if case["phase"] != "dual" and rng.random() < 0.5:
        case["n"] = round(rng.uniform(10.0, 25.0), 1)
    return case


# ---------------------------------------------------------------------------- inputs
def _cells(case):
    return [case["x"], case["y"], case["z"]]


def _n(case):
    return case["x"] * case["y"] * case["z"]


def _phases(case):
    """Phase name -> material.yaml entry; in every matrix of slip interactions only the first types differ from 1.4."""
    out = {}
    for name in {"fcc": ["fcc"], "bcc": ["bcc"], "dual": ["fcc", "bcc_ns"]}[case["phase"]]:
        p = copy.deepcopy({"fcc": workloads.FCC_PHASE, "bcc": workloads.BCC_PHASE,
                           "bcc_ns": workloads.BCC_NS_STRONG_PHASE}[name])
        pl = p["mechanical"]["plastic"]
        if name != "fcc":
            pl["h_sl-sl"] = [1.0] + [1.4] * 23
        if "n" in case:
            pl["n_sl"] = [case["n"]] * len(pl["n_sl"])
        out[name] = p
    return out


def _microstructure(case, seed):
    """Periodic Voronoi map (grain of every cell, x fastest) on the GPU and one random orientation per grain."""
    rng = np.random.default_rng(seed)
    seeds = torch.tensor(rng.random((case["grains"], 3)), device="cuda")
    q = rng.standard_normal((case["grains"], 4))
    q /= np.linalg.norm(q, axis=1, keepdims=True) * np.where(q[:, :1] < 0.0, -1.0, 1.0)
    ax = [(torch.arange(c, device="cuda", dtype=torch.float64) + 0.5) / c for c in _cells(case)]
    best = torch.full((case["z"], case["y"], case["x"]), 1.0e9, device="cuda", dtype=torch.float64)
    grain = torch.zeros_like(best, dtype=torch.int64)
    for g in range(case["grains"]):
        dx, dy, dz = ((a - seeds[g, k]) - torch.round(a - seeds[g, k]) for k, a in enumerate(ax))
        d = (dz * dz)[:, None, None] + (dy * dy)[None, :, None] + (dx * dx)[None, None, :]
        closer = d < best
        best = torch.where(closer, d, best)
        grain[closer] = g
    return grain.reshape(-1), q


def _solver(case, seed, scheme="spectral_basic"):
    grain, q = _microstructure(case, seed)
    phases = _phases(case)
    names = list(phases)
    mat = workloads.material_dict(q, phases[names[0]], names[0])
    mat["phase"] = phases
    for g, m in enumerate(mat["material"]):
        m["constituents"][0]["phase"] = names[g % len(names)]
    cells = np.asarray(_cells(case))
    grid = Grid(cells, cells / cells.max(), np.zeros(3), grain.cpu().numpy())
    return grid_mechanical(scheme)(grid, config.parse_material(mat), config.Numerics()), grain, q


# ---------------------------------------------------------------------------- response
def _path(case, seed, grain):
    """F of every step of the strain path and of the trial fields, (N, 3, 3) with [e, j, i] = F_ij (the entry
    point's layout): a mean stretch and shear at 1e-3/s, 20 % fluctuation from grain to grain and 2 % within."""
    g = torch.Generator(device="cuda").manual_seed(seed + 1)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float64)

    mean = torch.diag(torch.tensor([1.0e-3, -0.45e-3, -0.45e-3], device="cuda", dtype=torch.float64))
    rate = mean + 0.1e-3 * normal(3, 3) + 0.2e-3 * normal(case["grains"], 3, 3)[grain] + 0.02e-3 * normal(len(grain), 3, 3)
    one = torch.eye(3, device="cuda", dtype=torch.float64)
    steps = [one + (k + 1) * DT * rate for k in range(PATH_STEPS)]
    trials = [one + (PATH_STEPS + 1) * DT * rate + DT * c * 1.0e-3 * normal(len(grain), 3, 3) for c in (0.1, 0.05, 0.02)]
    return steps, trials[:TRIALS]


def _prepare_response(case, seed):
    s, grain, _ = _solver(case, seed)
    steps, trials = _path(case, seed, grain)
    st = ctypes.c_int32()
    torch.cuda.synchronize()
    for F in steps:
        _lib.check(s.lib.dmk_constitutive_device(s.h, DT, F.data_ptr(), None, ctypes.byref(st)), "response")
        if st.value:
            raise RuntimeError("a material point of the strain path did not converge")
        s.materialpoint_forward()
    P = [torch.empty_like(F) for F in trials]
    torch.cuda.synchronize()
    return {"kind": "response", "s": s, "F": trials, "P": P}


def _run_response(state):
    s, st, status = state["s"], ctypes.c_int32(), []
    for F, P in zip(state["F"], state["P"]):
        _lib.check(s.lib.dmk_constitutive_device(s.h, DT, F.data_ptr(), P.data_ptr(), ctypes.byref(st)), "response")
        status.append(st.value)
    return {"P": state["P"], "status": status, "C_volAvg": s.scalar("C_volAvg")}


# ---------------------------------------------------------------------------- increment
def _load(case, steps):
    t = DT * (steps + 1)
    return config.parse_load(workloads.tension_x(t, steps + 1))[1][0]


def _prepare_increment(case, seed):
    s, _, _ = _solver(case, seed, case["scheme"])
    lc = _load(case, LOAD_STEPS)
    first = copy.copy(lc)
    first.t, first.N = lc.t - DT, LOAD_STEPS
    r = s.run_loadcase(first)
    if r["rc"]:
        raise RuntimeError(f"the load case ends with {r['rc']}")
    s.forward(False, True, DT, DT, DT, lc)
    s.materialpoint_forward()
    names = ["F", "P", "xi_sl"]
    width = {"xi_sl": s.nsl}
    bufs = {k: torch.empty((s.N, width.get(k, 9)), dtype=torch.float64, pin_memory=True) for k in names}
    ptrs = {k: ctypes.cast(b.data_ptr(), ctypes.POINTER(ctypes.c_double)) for k, b in bufs.items()}
    _lib.check(s.lib.dmk_device_synchronize(), "dmk_device_synchronize")
    return {"kind": "increment", "s": s, "lc": lc, "bufs": bufs, "ptrs": ptrs}


def _run_increment(state):
    """The increment's attempt from its stored start (as the driver repeats it after a cutback), and its results."""
    s = state["s"]
    s.forward(True, True, DT, DT, DT, state["lc"])
    sol = s.solution()
    for k, p in state["ptrs"].items():
        _lib.check(s.lib.dmk_mech_get_field(s.h, FIELDS[k], p), "dmk_mech_get_field")
    return {"converged": sol.converged, "P_av": s.scalar("P_av"), "F_aim": s.scalar("F_aim"),
            "C_volAvg": s.scalar("C_volAvg"), **state["bufs"]}


# ---------------------------------------------------------------------------- divergence
def _field(case, seed):
    """A stress-like field (MPa scale), (N, 9): a mean, smooth waves and noise."""
    g = torch.Generator(device="cuda").manual_seed(seed + 2)
    f = 1.0e6 * torch.randn(_n(case), 9, generator=g, device="cuda", dtype=torch.float64)
    k = torch.arange(_n(case), device="cuda", dtype=torch.float64)
    return f + 5.0e7 + 1.0e7 * torch.sin(2.0 * math.pi * k / case["x"])[:, None]


def _prepare_divergence(case, seed):
    return {"kind": "divergence", "lib": _lib.load(), "cells": np.asarray(_cells(case), np.int32),
            "size": np.asarray([1.0, 1.0, 1.0]), "field": _field(case, seed),
            "rms": torch.zeros(1, dtype=torch.float64, device="cuda")}


def _run_divergence(state):
    _lib.check(state["lib"].dmk_divergence_rms_noalloc(
        _lib.iptr(state["cells"]), _lib.dptr(state["size"]), 2, state["field"].data_ptr(), state["rms"].data_ptr(),
        torch.cuda.current_stream().cuda_stream), "dmk_divergence_rms_noalloc")
    return state["rms"]


# ---------------------------------------------------------------------------- gradient
def _prepare_gradient(case, seed):
    s, _, _ = _solver(case, seed)
    k = case["increments"]
    lc = config.parse_load(workloads.tension_x(DT * (LOAD_STEPS + k), LOAD_STEPS + k))[1][0]
    first = copy.copy(lc)
    first.t, first.N = DT * LOAD_STEPS, LOAD_STEPS
    last = copy.copy(lc)
    last.t, last.N = DT * k, k
    for part in (first, last):
        if part is last:
            s.adjoint_tape(2 * k + 16)      # the curve's last increments, in plastic flow
        r = s.run_loadcase(part)
        if r["rc"]:
            raise RuntimeError(f"the load case ends with {r['rc']}")
    P = s.adjoint_info()["P_av"]
    target = P * (1.0 + 0.02 * np.random.default_rng(seed).standard_normal(P.shape))
    Pb = np.zeros_like(P)
    Pb[:, 0] = 2.0 * (P[:, 0] - target[:, 0]) / len(P)
    return {"kind": "gradient", "s": s, "Pb": Pb}


def _run_gradient(state):
    return state["s"].adjoint_backward(state["Pb"], 1.0e-6)[0]


# ---------------------------------------------------------------------------- the interface
def prepare(case, seed):
    return {"response": _prepare_response, "increment": _prepare_increment, "divergence": _prepare_divergence,
            "gradient": _prepare_gradient}[case["kind"]](case, seed)


def run(state):
    return {"response": _run_response, "increment": _run_increment, "divergence": _run_divergence,
            "gradient": _run_gradient}[state["kind"]](state)


def _systems(case):
    return {"fcc": 12, "bcc": 24, "dual": 18}[case["phase"]]


def work(case):
    n = _n(case)
    spectrum = 9.0 * 16 * (case["x"] // 2 + 1) * case["y"] * case["z"]
    transform = 9 * 5.0 * n * math.log2(n) / 2 * 2          # 9 real fields, 2.5 N log2 N each, forward and back
    if case["kind"] == "divergence":
        return {"bytes": 72.0 * n + 8, "flops": transform / 2 + 9 * 6.0 * n}
    m = _systems(case)
    # the material law: F, F_0, F_p0, S_0, L_p, xi_0, gamma_0 in; P, F_p, F_e, S, L_p, xi, gamma out;
    # 5 Newton steps of 40 operations a system and 600 besides, 2 state steps
    point_bytes = 8.0 * (5 * 9 + 2 * m + 5 * 9 + 2 * m)
    point_flops = 5 * 2.0 * (40 * m + 600) + 2 * 2.0 * (m * m + 20 * m)
    tangent_bytes = 8.0 * (81 + 4 + 5 * 9 + m)
    tangent_flops = 2.0 * (40 * m + 9 * 150)
    if case["kind"] == "response":
        return {"bytes": TRIALS * n * (point_bytes + tangent_bytes + 2 * 72), "flops": TRIALS * n * (point_flops + tangent_flops)}
    if case["kind"] == "increment":
        # about 7 residual evaluations; each takes the material law and both transforms of nine fields (the
        # other schemes: three transforms a residual and the tangent at each)
        plain = case["scheme"] == "spectral_basic"
        res = 7
        nb = res * (n * (point_bytes + 9 * 8.0 * 2) + (2 if plain else 6) * spectrum) + n * tangent_bytes * (1 if plain else res)
        fl = res * (n * point_flops + (1 if plain else 3) * transform) + n * tangent_flops * (1 if plain else res)
        return {"bytes": nb + 8.0 * n * (18 + m), "flops": fl}
    # gradient: per increment the factorised local systems and about 18 applications of the adjoint operator
    # (a tangent a cell, both transforms, a basis vector written and the basis read)
    k = case["increments"]
    per = 8.0 * n * (9 + m) * (9 + m) + 18 * (n * 8.0 * (81 + 9 + 9) + 2 * spectrum)
    return {"bytes": k * per, "flops": k * n * (2.0 / 3.0 * (9 + m) ** 3 + 18 * 200.0) + k * 18 * transform}


def tolerance(case):
    # The Newton iterations stop at 1e-6 of L_p and the state iterations at 1e-6 of the state, so results depend on
    # the L_p they start from: measured between a first and a third pass, P of a response differs by up to 4e-8, P
    # of an increment by up to 8e-10 (a cell that takes one state iteration more is allowed for).  The gradient's
    # linear solves stop at 1e-6, which is within 2e-7 of a solve to 1e-12.
    return {"response": {"rel": 2.0e-7}, "increment": {"rel": 1.0e-7}, "divergence": {"rel": 1.0e-13},
            "gradient": {"rel": 1.0e-6}}[case["kind"]]


# ---------------------------------------------------------------------------- 64-bit references
def _exact_divergence(case, seed):
    x, y, z = _cells(case)
    f = torch.fft.rfftn(_field(case, seed).reshape(z, y, x, 9), dim=(0, 1, 2))     # component i + 3 j of P_ij
    k = []
    for n, axis in ((z, 0), (y, 1), (x, 2)):
        freq = torch.fft.rfftfreq if axis == 2 else torch.fft.fftfreq
        v = 2.0 * math.pi * freq(n, 1.0 / n, dtype=torch.float64, device="cuda")
        if n % 2 == 0:
            v = torch.where(torch.arange(len(v), device="cuda") == n // 2, 0.0, v)
        k.append(v.reshape([-1 if a == axis else 1 for a in range(3)]))
    div = [f[..., i] * k[2] + f[..., i + 3] * k[1] + f[..., i + 6] * k[0] for i in range(3)]
    s = sum(d.real**2 + d.imag**2 for d in div)
    w = torch.full((x // 2 + 1,), 2.0, device="cuda", dtype=torch.float64)
    w[0] = w[-1] = 1.0          # the reference counts the last plane once for odd x too
    return ((s * w).sum().sqrt() / _n(case)).reshape(1)


def _slip(lattice):
    """Slip directions and normals, self-interaction and (cF) coplanar pairs marked with 1, all others 1.4."""
    def family(d, n):
        import itertools
        signs = list(itertools.product((1, -1), repeat=3))
        dirs = {tuple(s * c for s, c in zip(sg, p)) for p in itertools.permutations(d) for sg in signs}
        norm = {tuple(s * c for s, c in zip(sg, p)) for p in itertools.permutations(n) for sg in signs}
        half = [{max(v, tuple(-c for c in v)) for v in u} for u in (dirs, norm)]
        return [(a, b) for b in sorted(half[1]) for a in sorted(half[0]) if sum(p * q for p, q in zip(a, b)) == 0]

    pairs = family((0, 1, 1), (1, 1, 1)) if lattice == "cF" else family((1, 1, 1), (0, 1, 1)) + family((1, 1, 1), (1, 1, 2))
    d = np.asarray([p[0] for p in pairs], float)
    n = np.asarray([p[1] for p in pairs], float)
    same = np.asarray([[p == q or (lattice == "cF" and p[1] == q[1]) for q in pairs] for p in pairs])
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    n /= np.linalg.norm(n, axis=1, keepdims=True)
    to = {"device": "cuda", "dtype": torch.float64}
    return torch.tensor(d[:, :, None] * n[:, None, :], **to), torch.tensor(np.where(same, 1.0, 1.4), **to)


def _exact_response(case, seed):
    """The strain path and the trial fields through the material law, one phase without non-Schmid terms: the
    damped fixed point of the state as the reference iterates it, the stress of each state to rounding."""
    if case["phase"] == "dual":
        return None
    grain, q = _microstructure(case, seed)
    ph = _phases(case)[case["phase"]]["mechanical"]
    el, pl = ph["elastic"], ph["plastic"]
    M, H = _slip({"fcc": "cF", "bcc": "cI"}[case["phase"]])
    C11, C12, C44 = el["C_11"], el["C_12"], el["C_44"]
    g0, n, a = pl["dot_gamma_0_sl"][0], pl["n_sl"][0], pl["a_sl"][0]
    h0, xi_inf = pl["h_0_sl-sl"][0], pl["xi_inf_sl"][0]
    one = torch.eye(3, device="cuda", dtype=torch.float64)
    w, v = torch.tensor(q[:, 0], device="cuda"), torch.tensor(q[:, 1:], device="cuda")
    # passive rotation matrix, with the sign of the quaternion's vector part that the reference takes (P = -1)
    cross = torch.zeros(len(q), 3, 3, device="cuda", dtype=torch.float64)
    for i, j, k, s in ((0, 1, 2, -1), (0, 2, 1, 1), (1, 0, 2, 1), (1, 2, 0, -1), (2, 0, 1, -1), (2, 1, 0, 1)):
        cross[:, i, j] = s * v[:, k]
    om = (w * w - (v * v).sum(1))[:, None, None] * one + 2.0 * v[:, :, None] * v[:, None, :] - 2.0 * w[:, None, None] * cross
    Fp0 = om[grain]
    N = len(grain)
    xi0 = torch.full((N, len(M)), pl["xi_0_sl"][0], device="cuda", dtype=torch.float64)
    S0 = torch.zeros(N, 3, 3, device="cuda", dtype=torch.float64)
    Lp = torch.zeros_like(S0)

    def hooke(E):
        tr = E.diagonal(dim1=1, dim2=2).sum(1)
        d = torch.diag_embed((C11 - C12) * E.diagonal(dim1=1, dim2=2) + C12 * tr[:, None])
        return d + 2.0 * C44 * (E - torch.diag_embed(E.diagonal(dim1=1, dim2=2)))

    def rates(S, xi):
        tau = torch.einsum("nij,aij->na", S, M)
        gd = torch.sign(tau) * g0 * (tau.abs() / xi) ** n
        return tau, gd

    def xi_rate(gd, xi):
        x = 1.0 - xi / xi_inf
        return h0 * torch.sign(x) * x.abs() ** a * (gd.abs() @ H.T)

    def stress(F, Fp0, xi, Lp):
        """L_p = sum rate P to rounding (Newton with halving), its S and rates."""
        A = F @ torch.linalg.inv(Fp0)

        def residual(L):
            Fe = A @ (one - DT * L)
            S = hooke(0.5 * (Fe.mT @ Fe - one))
            tau, gd = rates(S, xi)
            return Fe, S, tau, gd, L - torch.einsum("na,aij->nij", gd, M)

        Fe, S, tau, gd, r = residual(Lp)
        rn = r.flatten(1).norm(dim=1)
        for _ in range(60):
            todo = rn > 1.0e-13 * Lp.flatten(1).norm(dim=1) + 1.0e-22
            if not bool(todo.any()):
                break
            dg = torch.where(tau == 0.0, 0.0, n * gd / torch.where(tau == 0.0, 1.0, tau))
            G = Fe.mT @ A
            Y = torch.stack([G.mT @ hooke(m[None])[0] for m in 0.5 * (M + M.mT)], 1)
            J = torch.eye(9, device="cuda", dtype=torch.float64) + DT * torch.einsum(
                "na,ap,naq->npq", dg, M.flatten(1), Y.flatten(2))
            d = torch.linalg.solve(J, r.flatten(1)).reshape(-1, 3, 3)
            step = todo.double()
            for _ in range(40):
                new = Lp - step[:, None, None] * d
                got = residual(new)
                gn = got[4].flatten(1).norm(dim=1)
                worse = todo & ~(gn < rn) & (step > 1.0e-3)
                if not bool(worse.any()):
                    break
                step = torch.where(worse, 0.5 * step, step)
            better = todo & (gn < rn)
            if not bool(better.any()):
                break
            Lp = torch.where(better[:, None, None], new, Lp)
            Fe, S, tau, gd, r = residual(Lp)
            rn = r.flatten(1).norm(dim=1)
        return Lp, S, gd

    def response(F, Lp):
        _, gd = rates(S0, xi0)
        xd, gdot = xi_rate(gd, xi0), gd.abs()
        xi, gam = xi0 + DT * xd, DT * gdot
        last, last2 = torch.cat([xd, gdot], 1), torch.zeros(N, 2 * len(M), device="cuda", dtype=torch.float64)
        open_ = torch.ones(N, dtype=torch.bool, device="cuda")
        S = S0
        for it in range(20):
            L_new, S_new, gd = stress(F, Fp0, xi, Lp)
            Lp = torch.where(open_[:, None, None], L_new, Lp)
            S = torch.where(open_[:, None, None], S_new, S)
            now = torch.cat([xi_rate(gd, xi), gd.abs()], 1)
            d1, d2 = now - last, last - last2
            d12, d22, d01 = (d1 * d2).sum(1), (d2 * d2).sum(1), (now * last).sum(1)
            damp = (torch.minimum(d01, d12) < 0.0) & (d22 > 0.0)
            zeta = torch.where(damp, 0.75 + 0.25 * torch.tanh(2.0 + 4.0 * d12 / torch.where(d22 > 0.0, d22, 1.0)), 1.0)[:, None]
            now = now * zeta + last * (1.0 - zeta)
            last2, last = last, now
            state = torch.cat([xi, gam], 1)
            res = state - torch.cat([xi0, torch.zeros_like(gam)], 1) - DT * now
            state = state - res
            m = len(M)
            ok = ((res[:, :m].abs() <= torch.clamp(1.0e-6 * state[:, :m].abs(), min=pl["atol_xi"])).all(1)
                  & (res[:, m:].abs() <= torch.clamp(1.0e-6 * state[:, m:].abs(), min=1.0e-6)).all(1))
            xi = torch.where(open_[:, None], state[:, :m], xi)
            gam = torch.where(open_[:, None], state[:, m:], gam)
            open_ = open_ & ~ok
            if not bool(open_.any()):
                break
        inv = torch.linalg.inv(Fp0) @ (one - DT * Lp)
        Fp = torch.linalg.inv(inv)
        P = F @ inv @ S @ inv.mT
        return P, Fp / torch.linalg.det(Fp)[:, None, None] ** (1.0 / 3.0), xi, S, Lp

    steps, trials = _path(case, seed, grain)
    for F in steps:
        P, Fp0, xi0, S0, Lp = response(F.mT, Lp)
    return {"P": [response(F.mT, Lp)[0].mT.contiguous() for F in trials], "status": [None] * len(trials), "C_volAvg": None}


def exact(case, seed):
    if case["kind"] == "divergence":
        return _exact_divergence(case, seed)
    if case["kind"] == "response":
        return _exact_response(case, seed)
    # an increment's and a gradient's results are those of iterations that stop at a tolerance: they have no
    # such value
    return None
