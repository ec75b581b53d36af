"""The work that users of this framework have it do, as cases to time and compare.

A pass of a stepping case is one batch of the reference's time loop through the framework's own
entry point: the state lies in the program's host arrays (the reference's layout), the host
modules' globals point at them, cuda_timeIntCommence takes the state to the device, runs NtBatch
RK3 steps and brings the state and the surface fields back.  The other passes set up an ensemble
and step it, evaluate and differentiate the SGS network, and reduce a stored state to the
statistics a post-processing program reads.

The library holds one model at a time, so the model of a case is set up once and its states take
turns on it.  Each state is made from its seed alone: the base state of the case (restated here)
with smooth velocity, temperature, SGS energy and moisture perturbations and small-scale noise.
exact() restates the model step, the network and the statistics in 64 bits with plain torch.
"""
import ctypes
import json
import math
import os
import sys
import tempfile

import numpy as np
import torch

_REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_REPO, "fasteddy-model_amd"))
import fe_py  # noqa: E402

_DEV = "cuda" if torch.cuda.is_available() else "cpu"
_NH = 3

# ----------------------------------------------------------------------------------------------
# the cases


def listed():
    return [
        # the repository's smallest configuration, its 200-step batch: 8 tiles of columns, one
        # launch takes some 20 us, so launches and latency count
        {"name": "cbl_64x64x48", "kind": "steps", "physics": "cbl", "nx": 64, "ny": 64, "nz": 48, "dx": 20.0, "steps": 200},
        # the dry convective boundary layer at production size (the headline configuration)
        {"name": "cbl_512x512x128", "kind": "steps", "physics": "cbl", "nx": 512, "ny": 512, "nz": 128, "dx": 10.0, "steps": 100},
        # the stable boundary layer example at its full size: ragged in y, skin-temperature
        # surface layer, SGS stresses written with every batch
        {"name": "sbl_128x126x122", "kind": "steps", "physics": "sbl", "nx": 128, "ny": 126, "nz": 122, "dx": 3.125, "steps": 200},
        # moist shallow cumulus at production size: q_v and q_l (WENO5), saturation adjustment
        {"name": "cumulus_256x256x160", "kind": "steps", "physics": "cumulus", "nx": 256, "ny": 256, "nz": 160, "dx": 25.0, "steps": 100},
        # the BOMEX example at its full size: ragged in x and y, HYB34 q_v, vertical filter,
        # large-scale forcing with subsidence, SGS stresses and moisture fluxes written
        {"name": "bomex_152x146x122", "kind": "steps", "physics": "bomex", "nx": 152, "ny": 146, "nz": 122, "dx": 100.0, "steps": 100},
        # the Smagorinsky closure on a mid-size grid, ragged in every direction, stretched
        {"name": "smagorinsky_200x186x75", "kind": "steps", "physics": "smagorinsky", "nx": 200, "ny": 186, "nz": 75, "dx": 20.0, "steps": 100},
        # a terrain-following grid: the dry boundary layer over a hill
        {"name": "hill_256x256x128", "kind": "steps", "physics": "hill", "nx": 256, "ny": 256, "nz": 128, "dx": 10.0, "steps": 100},
        # one GPU's block of the production case on 8 GPUs: halos from a buffer filled every stage
        {"name": "block_128x256x128", "kind": "steps", "physics": "block", "nx": 128, "ny": 256, "nz": 128, "dx": 10.0, "steps": 100},
        # the learned SGS closure with the committed network on its evaluation grid
        {"name": "learned_128x128x48", "kind": "steps", "physics": "learned", "nx": 128, "ny": 128, "nz": 48, "dx": 20.0, "steps": 50},
        # a batched ensemble of small members, each with its own surface heat flux and wind
        {"name": "ensemble_16x64x64x48", "kind": "ensemble", "physics": "cbl", "nx": 64, "ny": 64, "nz": 48, "dx": 20.0, "members": 16, "steps": 200},
        # the network's forward and backward over one training batch of rows
        {"name": "network_8192", "kind": "network", "rows": 8192},
        # statistics of a stored state: profiles and the per-field summary, as a post-processing
        # program asks for them
        {"name": "statistics_256x256x96", "kind": "statistics", "physics": "cumulus", "nx": 256, "ny": 256, "nz": 96, "dx": 25.0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the same ranges: grids from the smallest to the production size, odd extents among
    them, batches of tens to hundreds of steps, every kind of physics."""
    physics = rng.choice(["cbl", "cbl", "sbl", "cumulus", "bomex", "smagorinsky", "hill", "block", "learned", "ensemble",
                          "network", "statistics"])
    if physics == "network":
        return {"kind": "network", "rows": _log(rng, 900, 60000)}
    dx = {"sbl": 3.125, "cumulus": 25.0, "bomex": 100.0, "learned": 20.0}.get(physics, rng.choice([10.0, 20.0]))
    if physics == "ensemble":
        return {"kind": "ensemble", "physics": "cbl", "nx": 64, "ny": 8 * rng.randint(5, 12), "nz": 2 * rng.randint(16, 32),
                "dx": 20.0, "members": rng.randint(4, 16), "steps": 10 * rng.randint(8, 20)}
    nx, ny, nz = _log(rng, 64, 400), _log(rng, 64, 400), _log(rng, 40, 150)
    if physics == "block":                               # a block holds whole 64 x 8 tiles
        nx, ny = 64 * max(1, nx // 64), 8 * (ny // 8)
    if physics == "statistics":
        return {"kind": "statistics", "physics": rng.choice(["cbl", "cumulus"]), "nx": nx, "ny": ny, "nz": nz, "dx": 25.0}
    if physics == "learned":
        nx, ny, nz = min(nx, 192), min(ny, 192), min(nz, 64)
    steps = max(20, min(200, int(6e8 / (nx * ny * nz))))
    return {"kind": "steps", "physics": physics, "nx": nx, "ny": ny, "nz": nz, "dx": dx, "steps": steps}


def _fields(case):
    p = case["physics"]
    return 5 + (p != "smagorinsky") + 2 * (p in ("cumulus", "bomex"))


def work(case):
    """What a pass cannot do without: a step reads the stage input and the RK base and writes the
    output once per stage (32 B per field and cell), and the batch takes the state in and out."""
    if case["kind"] == "network":
        layers = 256 * 64 + 64 * 64 + 64 * 64 + 64 * 16
        return {"bytes": 4.0 * case["rows"] * (256 + 16) + 8.0 * layers, "flops": 6.0 * case["rows"] * layers}
    cells = case["nx"] * case["ny"] * case["nz"] * case.get("members", 1)
    nf = _fields(case)
    if case["kind"] == "statistics":
        return {"bytes": 4.0 * nf * cells * 2, "flops": 30.0 * cells}
    per = 32.0 * nf
    flops = 1100.0 * cells * case["steps"] * nf / 6
    if case["physics"] == "learned":
        flops += 2.0 * cells * case["steps"] * (256 * 64 + 64 * 64 + 64 * 64 + 64 * 16)
    return {"bytes": per * cells * case["steps"] + 8.0 * nf * cells, "flops": flops}


# ----------------------------------------------------------------------------------------------
# parameter sets (the repository's configurations and the reference's examples)

_SBL = dict(coriolisLatitude=73.0, dampingLayerDepth=100.0, surflayerSelector=2, surflayer_z0=0.1, surflayer_z0t=0.1,
            surflayer_wth=0.0, surflayer_tr=-0.25, stabilityScheme=2, temp_grnd=265.0, zStableBottom=100.0, stableGradient=0.01,
            thetaHeight=75.0, U_g=8.0, hydroSubGridWrite=1)
_BOMEX = dict(moistureAdvSelectorQv=2, coriolisLatitude=14.94, filterSelector=1, dampingLayerDepth=500.0, surflayer_z0=0.0002,
              surflayer_z0t=0.0002, temp_grnd=299.9728, pres_grnd=101500.0, stableGradient=0.003854, zStableBottom2=1480.0,
              stableGradient2=0.011154, zStableBottom3=2000.0, stableGradient3=0.00365, z_Ug=0.0, Ug_grad=0.0018,
              hydroSubGridWrite=1, lsfSelector=1, lsf_horMnSubTerms=1, lsf_freq=1.0, lsf_w_surf=0.0, lsf_w_lev1=-23.4,
              lsf_w_lev2=0.0, lsf_w_zlev1=1500.0, lsf_w_zlev2=2100.0, lsf_th_surf=-0.0833333, lsf_th_lev1=-0.0833333,
              lsf_th_lev2=0.0, lsf_th_zlev1=1500.0, lsf_th_zlev2=3000.0, lsf_qv_surf=-0.0432, lsf_qv_lev1=-0.0432,
              lsf_qv_lev2=0.0, lsf_qv_zlev1=300.0, lsf_qv_zlev2=500.0)


def _params(case):
    ph, dx = case["physics"], case["dx"]
    dz = {"bomex": 40.0}.get(ph, dx)
    p = dict(fe_py.CFG2 if ph in ("cumulus", "bomex") else fe_py.CFG0)
    p.update(Nx=case["nx"], Ny=case["ny"], Nz=case["nz"], d_xi=dx, d_eta=dx, d_zeta=dz,
             dt={"sbl": 0.005, "bomex": 0.075}.get(ph, 0.002 * dx), NtBatch=case.get("steps", 1), Nt=10 ** 7)
    if ph == "sbl":
        p.update(_SBL)
    elif ph == "bomex":
        p.update(_BOMEX)
    elif ph == "smagorinsky":
        p.update(TKESelector=0, verticalDeformSwitch=1)
    elif ph == "block":
        p.update(amd_haloBuffer=1)
    return p


def _hill(case):
    """Height and radius of the hill: flat within four cells of every edge."""
    return 4.0 * case["dx"], 0.5 * (min(case["nx"], case["ny"]) - 10) * case["dx"]


def _topography(case):
    """Surface elevation [nx][ny] in float32: a cos^2 hill in the middle, or flat."""
    nx, ny, dx = case["nx"], case["ny"], case["dx"]
    if case["physics"] != "hill":
        return np.zeros((nx, ny), np.float32)
    h, rad = _hill(case)
    r = np.hypot(((np.arange(nx) + 0.5) * dx - nx * dx / 2)[:, None], ((np.arange(ny) + 0.5) * dx - ny * dx / 2)[None, :])
    return np.where(r < rad, h * np.cos(np.pi * r / (2 * rad)) ** 2, 0.0).astype(np.float32)


# ----------------------------------------------------------------------------------------------
# grid and base state, restated; float32 where they are the model's inputs


class _Grid:
    """Coordinates, metrics (J33, D) and the hydrostatic base state on levels -3 .. nz+2 of every
    column (one column when flat), float64 tensors of float32 values."""

    def __init__(self, case, p):
        f = np.float32
        nx, ny, nz, dz = case["nx"], case["ny"], case["nz"], f(p["d_zeta"])
        self.case, self.p, self.nx, self.ny, self.nz = case, p, nx, ny, nz
        h = _topography(case) if case["physics"] == "hill" else np.zeros((1, 1), f)
        ztop = f(f(nz) * dz - 0.5 * float(dz))
        z = (np.arange(nz).astype(f) * dz + f(0.5 * float(dz))).astype(f)
        if p["verticalDeformSwitch"]:
            c1, fc, zc = float(f(p["verticalDeformFactor"])), float(f(p["verticalDeformQuadCoeff"])), float(ztop)
            c2 = fc * (1.0 - c1) / zc
            c3 = float(f((1.0 - c2 * zc - c1) / zc ** 2))
            z = (c3 * z.astype(np.float64) ** 3 + float(f(c2)) * z.astype(np.float64) ** 2 + c1 * z).astype(f)
        z = (z[None, None, :] * ((ztop - h) / ztop).astype(f)[:, :, None] + h[:, :, None]).astype(f)
        lo = [z[..., :1] - f(n) * (z[..., 1:2] - z[..., :1]) for n in (3, 2, 1)]
        hi = [z[..., -1:] + f(n) * (z[..., -1:] - z[..., -2:-1]) for n in (1, 2, 3)]
        z = np.concatenate(lo + [z] + hi, axis=2).astype(f)
        t22 = ((z[..., 4:4 + nz] - z[..., 2:2 + nz]) * f(1.0 / (2.0 * float(dz)))).astype(f)
        # the lateral coordinates do not vary along a column: D = T00 T11 T22, J33 = T00 T11 / D
        t = f(f(2) * f(p["d_xi"]) * f(1.0 / (2.0 * p["d_xi"])))
        det = (t * t22 * t).astype(f)
        j33 = (t * t * (f(1) / det)).astype(f)
        pad = lambda a: np.concatenate([a[..., :1]] * 3 + [a] + [a[..., -1:]] * 3, axis=2)
        g = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(_DEV).double()
        self.z, self.D, self.J33 = g(z), g(pad(det)), g(pad(j33))
        self._base(g, z.astype(np.float64), p)

    def _base(self, g, z, p):
        R, cv = float(np.float32(287.04)), 718.0
        cp = float(np.float32(np.float32(287.04) + np.float32(718.0)))
        G = float(np.float32(9.81))
        self.R, self.cp, self.g, self.gam, self.rcp, self.pref = R, cp, G, cp / cv, R / cp, 1.0e5
        self.c1 = R / self.pref ** self.rcp
        tg = p["temp_grnd"] * (p["pres_grnd"] / self.pref) ** -self.rcp
        z1, g1, z2, g2 = p["zStableBottom"], p["stableGradient"], p["zStableBottom2"], p["stableGradient2"]
        z3, g3 = p["zStableBottom3"], p["stableGradient3"]
        pg = (p["pres_grnd"] / self.pref) ** self.rcp
        if p["stabilityScheme"] == 1:
            z2 = z3 = 1e9
        thA = tg + g1 * (np.minimum(z, z2) - z1)
        th2, th3 = tg + g1 * (z2 - z1), tg + g1 * (z2 - z1) + g2 * (z3 - z2)
        thB = th2 + g2 * (np.minimum(z, z3) - z2)
        thC = th3 + g3 * (z - z3)
        th = np.where(z <= z1, tg, np.where(z <= z2, thA, np.where(z <= z3, thB, thC)))
        safe = lambda a: np.log(np.maximum(a, 1e-30))
        integral = np.where(z <= z1, z / tg, z1 / tg + safe(1 + g1 * (np.clip(z, z1, z2) - z1) / tg) / g1
                            + np.where(z > z2, safe(1 + g2 * (np.clip(z, z2, z3) - z2) / th2) / g2, 0)
                            + np.where(z > z3, safe(1 + g3 * (z - z3) / th3) / g3, 0))
        pb = self.pref * ((-G / cp) * integral + pg) ** (cp / R)
        rho = pb / (th * (pb / self.pref) ** self.rcp * R)
        self.rho = g(rho.astype(np.float32))
        self.rth = g((th * rho).astype(np.float32))
        ug = np.where(z < p["z_Ug"], p["U_g"], p["U_g"] + p["Ug_grad"] * (z - p["z_Ug"]))
        self.ug = g(ug)
        self.theta = g(th)


_grids = {}


def _grid(case, **over):
    key = json.dumps([{k: v for k, v in case.items() if k not in ("name", "steps", "members")}, over], sort_keys=True)
    if key not in _grids:
        _grids.clear()
        _grids[key] = _Grid(case, dict(_params(case), **over))
    return _grids[key]


def _initial(case, seed, grid=None):
    """Initial state of a seed: float32 [field][x][y][z], fields rho, rho u, rho v, rho w, rho theta,
    then rho e (prognostic closure) and rho q_v, rho q_l in g/kg (moist)."""
    g = grid or _grid(case)
    nx, ny, nz = g.nx, g.ny, g.nz
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device=_DEV).manual_seed(int(rng.integers(2 ** 31)))
    X, Y, Z = (torch.arange(n, device=_DEV, dtype=torch.float64) for n in (nx, ny, nz))

    def wave(amp):
        out = torch.zeros((nx, ny, nz), device=_DEV, dtype=torch.float64)
        for _ in range(3):
            kx, ky = rng.integers(1, 4, size=2)
            kz, (a, b, c) = rng.uniform(0.5, 2.5), rng.uniform(0, 2 * np.pi, size=3)
            out += (torch.sin(2 * np.pi * kx * X / nx + a)[:, None, None] * torch.sin(2 * np.pi * ky * Y / ny + b)[None, :, None]
                    * torch.sin(np.pi * kz * (Z + 0.5) / nz + c)[None, None, :])
        return amp * out / 2

    def noise(amp):
        return amp * (2 * torch.rand((nx, ny, nz), generator=gen, device=_DEV, dtype=torch.float32).double() - 1)

    inner = lambda a: a[..., _NH:_NH + nz].expand(nx, ny, nz)
    z = inner(g.z)
    rho = inner(g.rho) * (1 + wave(1e-5))
    moist = case["physics"] in ("cumulus", "bomex")
    out = torch.empty((_fields(case), nx, ny, nz), dtype=torch.float32, device=_DEV)
    out[0] = rho
    out[1] = rho * (inner(g.ug) + wave(0.8) + noise(0.05))
    out[2] = rho * (wave(0.8) + noise(0.05))
    out[3] = rho * (wave(0.4) + noise(0.02))
    depth = float(g.p["thetaHeight"])
    out[4] = inner(g.rth) * (1 + wave(2e-4)) + rho * torch.where(z < depth, noise(0.25 if not moist else 0.1), torch.zeros_like(z))
    if case["physics"] != "smagorinsky":
        out[5] = rho * (0.02 + 0.3 * torch.exp(-z / max(depth, 50.0)) * (1 + wave(0.4) + noise(0.2)).clamp_min(0.1))
    if moist:
        pts = np.array([0.0, 1500.0, 3000.0, 1e6]), np.array([17.0, 13.0, 4.0, 4.0])
        qv = torch.from_numpy(np.interp(z[:1, :1].cpu().numpy(), *pts)).to(_DEV)
        cloud = (wave(1.0) - 0.4).clamp_min(0.0) * ((z > 500) & (z < 1800))
        out[6] = rho * (qv + wave(0.4) + noise(0.1)).clamp_min(0.1)
        out[7] = rho * 0.4 * cloud
    return out


# ----------------------------------------------------------------------------------------------
# the one live model, and a program's own host arrays in its place

_live = {"key": None, "model": None, "sgs": None}
_work = tempfile.mkdtemp(prefix="fe_cases_")
_SURFACE = ("fricVel", "htFlux", "tskin", "qFlux", "qskin")


def _close():
    if _live["sgs"] is not None:
        if _live["model"].device:
            _live["sgs"].enable(False)
        _live["sgs"].clear()
    if _live["model"] is not None:
        _live["model"].close()
    _live.update(key=None, model=None, sgs=None)


def _network():
    s = fe_py.LearnedSGS()
    s.load(os.path.join(_REPO, "fasteddy-model_amd", "sgs_cbl20m.npz"))
    return s


def _model(case):
    """The model of a case, set up once; a model of another case makes way for it."""
    key = json.dumps({k: v for k, v in case.items() if k != "name"}, sort_keys=True)
    if _live["key"] == key:
        return _live["model"]
    _close()
    if case["kind"] == "network":
        p = dict(fe_py.CFG0, Nx=64, Ny=8, Nz=16)
    else:
        p = _params(case)
        if case["physics"] == "hill":
            p["topoFile"] = fe_py.hill_topo(os.path.join(_work, "hill.bin"), case["nx"], case["ny"], case["dx"], *_hill(case))
    m = fe_py.Model(p, _work, device=case["kind"] != "ensemble")
    _live.update(key=key, model=m)
    if case["kind"] == "network" or case.get("physics") == "learned":
        _live["sgs"] = _network()
    if case.get("physics") == "learned":
        _live["sgs"].enable(True)
    return m


class _Bound:
    """The host modules' globals point at a program's own arrays while its state is the model's."""

    def __init__(self, lib, arrays):
        self.cells = {n: ctypes.c_void_p.in_dll(lib, n) for n in arrays}
        self.arrays = arrays

    def __enter__(self):
        self.before = {n: c.value for n, c in self.cells.items()}
        for n, c in self.cells.items():
            c.value = self.arrays[n].ctypes.data

    def __exit__(self, *_):
        for n, c in self.cells.items():
            c.value = self.before[n]


def _host_arrays(m, case, init):
    """A program's host arrays (halo-inclusive, z fastest) holding the initial state."""
    init = init.cpu().numpy()
    arrays = {}
    put = (slice(None),) + (slice(_NH, -_NH),) * 3
    at = 0
    for name, n in (("hydroFlds", 5), ("sgstkeScalars", int(case["physics"] != "smagorinsky")),
                    ("moistScalars", 2 * int(case["physics"] in ("cumulus", "bomex")))):
        if n:
            a = np.zeros((n,) + m.shape3, np.float32)
            a[put] = init[at:at + n]
            arrays[name] = a
            at += n
    for name in _SURFACE:
        if m.array(name) is not None:
            arrays[name] = m.array(name).copy()
    return arrays


def _rows(case, seed):
    """Normalised features and targets, some rows far out as in a developed flow."""
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((case["rows"], 256), np.float32)
    x *= np.where(rng.random((case["rows"], 1)) < 0.05, 3.0, 1.0).astype(np.float32)
    x[:, 250:] = 0
    t = rng.standard_normal((case["rows"], 16), np.float32)
    t[:, 9:] = 0
    return x, t


def prepare(case, seed):
    if case["kind"] == "network":
        _model(case)
        x, t = _rows(case, seed)
        return {"case": case, "x": x, "t": t}
    m = _model(case)
    if case["kind"] == "ensemble":
        members = []
        for k in range(case["members"]):
            over = _member(case, seed, k)
            members.append((over, _host_arrays(m, case, _initial(case, seed * 1000 + k, _grid(case, U_g=over["U_g"])))))
        return {"case": case, "members": members}
    return {"case": case, "arrays": _host_arrays(m, case, _initial(case, seed))}


def _member(case, seed, k):
    rng = np.random.default_rng([seed, k])
    return {"U_g": float(np.float32(rng.uniform(5.0, 15.0))), "surflayer_wth": float(np.float32(rng.uniform(0.1, 0.5)))}


# ----------------------------------------------------------------------------------------------
# a pass


def run(state):
    case = state["case"]
    m = _model(case)
    if case["kind"] == "network":
        s = _live["sgs"]
        y = s.forward(state["x"])
        loss, grad = s.gradient(state["x"], state["t"])
        return {"y": y, "loss": np.float32(loss), "grad": grad}
    if case["kind"] == "ensemble":
        return _run_ensemble(m, state)
    if case["kind"] == "statistics":
        with _Bound(m.L, state["arrays"]):
            m.upload()
            s = m.state_summary()
            return {"profiles": m.profiles(), "summary": np.array([list(r.values()) for r in s.values()])}
    # a batch from the state in the host arrays, at the start of a run
    m.seti("simTime_it", 0)
    m.seti("simTime_itRestart", 0)
    m.setf("simTime", 0.0)
    with _Bound(m.L, state["arrays"]):
        m.commence()
    # the prognostic state and the surface fields; p' is a diagnostic of rho theta
    cut = (slice(None),) + (slice(_NH, -_NH),) * 3
    out = {n: state["arrays"][n][cut] for n in ("hydroFlds", "sgstkeScalars", "moistScalars") if n in state["arrays"]}
    out.update({n: state["arrays"][n][_NH:-_NH, _NH:-_NH] for n in ("fricVel", "htFlux", "tskin")})
    if m.geti("hydroSubGridWrite") == 1:
        out["hydroTauFlds"] = m.array("hydroTauFlds")[cut].copy()
    return out


def _run_ensemble(m, state):
    """An ensemble from its members' host states: device set-up member by member, the steps, the
    members' states back."""
    L, case = m.L, state["case"]
    ens = fe_py.Ensemble()

    def ok(rc):
        if rc != 0:
            raise RuntimeError(f"member set-up failed with {rc}")

    base = {k: m.getf(k) for k in ("U_g", "surflayer_wth")}
    out = []
    try:
        for over, arrays in state["members"]:
            for k, v in over.items():
                m.setf(k, v)
            arrays["htFlux"][:] = over["surflayer_wth"]
            m.seti("simTime_it", 0)
            m.setf("simTime", 0.0)
            with _Bound(L, arrays):
                for f in ("fecuda_Init", "cuda_gridInit", "cuda_hydroCoreInit", "cuda_timeIntInit"):
                    ok(getattr(L, f)())
                ens.add(m)
                for f in ("cuda_timeIntCleanup", "cuda_hydroCoreCleanup", "cuda_gridCleanup", "fecuda_Cleanup"):
                    ok(getattr(L, f)())
        ens.steps(case["steps"])
        out = [ens.state(k) for k in range(len(state["members"]))]
    finally:
        ens.clear()
        for k, v in base.items():
            m.setf(k, v)
    return out


# ----------------------------------------------------------------------------------------------
# the same in 64 bits with plain torch


def exact(case, seed):
    if case["kind"] == "network":
        return _exact_network(case, seed)
    if case["kind"] == "statistics":
        return {"profiles": _exact_profiles(case, _initial(case, seed).double()).cpu().numpy(), "summary": None}
    if case["physics"] == "learned":
        return None      # its masks are decisions on 16-bit network outputs
    if case["nx"] * case["ny"] * case["nz"] * case.get("members", 1) * case["steps"] > 1.5e9:
        return None      # takes over 20 seconds
    if case["kind"] == "ensemble":
        out = []
        for k in range(case["members"]):
            over = _member(case, seed, k)
            g = _grid(case, **over)
            s = _LES(g)
            init = _initial(case, seed * 1000 + k, _grid(case, U_g=over["U_g"]))
            out.append(s.steps(init.double(), case["steps"])["state"].cpu().numpy())
        return out
    r = _LES(_grid(case)).steps(_initial(case, seed).double(), case["steps"])
    st = r["state"].cpu().numpy()
    out = {"hydroFlds": st[:5]}
    if case["physics"] != "smagorinsky":
        out["sgstkeScalars"] = st[5:6]
    if case["physics"] in ("cumulus", "bomex"):
        out["moistScalars"] = st[6:8]
    for k, n in (("fricVel", "ust"), ("htFlux", "hf"), ("tskin", "tsk")):
        out[k] = r[n].cpu().numpy()
    if _params(case)["hydroSubGridWrite"] == 1:
        out["hydroTauFlds"] = r["tau"].cpu().numpy()
    return out


def _exact_network(case, seed):
    x, t = _rows(case, seed)
    w = torch.from_numpy(np.load(os.path.join(_REPO, "fasteddy-model_amd", "sgs_cbl20m.npz"))["params"]).to(_DEV).double()
    w.requires_grad_(True)
    # the closure's activation: z (1/2 + zc Q(zc^2)), zc = z within [-4, 4]
    c = [3.988074278e-01, -6.606890165e-02, 9.584851178e-03, -1.022127353e-03, 7.636147270e-05, -3.724001524e-06,
         1.050534689e-07, -1.288297990e-09]

    def gelu(z):
        zc = z.clamp(-4, 4)
        q = torch.zeros_like(z)
        for a in reversed(c):
            q = q * zc * zc + a
        return z * (0.5 + zc * q)

    a, at = torch.from_numpy(x).to(_DEV).double(), 0
    for nin, nout in ((256, 64), (64, 64), (64, 64), (64, 16)):
        W, b = w[at:at + nin * nout].view(nin, nout), w[at + nin * nout:at + nin * nout + nout]
        at += nin * nout + nout
        a = a @ W + b
        if nout == 64:
            a = gelu(a)
    loss = (a[:, :9] - torch.from_numpy(t).to(_DEV).double()[:, :9]).square().mean()
    loss.backward()
    return {"y": a.detach().cpu().numpy(), "loss": loss.detach().cpu().numpy()[()], "grad": w.grad.cpu().numpy()}


def _exact_profiles(case, S):
    rho = S[0]
    u, v, w, th = (S[k] / rho for k in (1, 2, 3, 4))
    mean = lambda a: a.mean(dim=(0, 1))
    cov = lambda a, b: mean(a * b) - mean(a) * mean(b)
    uu, vv, ww = cov(u, u), cov(v, v), cov(w, w)
    zero = torch.zeros_like(uu)
    moist = S.shape[0] == 8
    cols = [mean(u), mean(v), mean(w), mean(th), uu, cov(u, w), vv, cov(v, w), ww, 0.5 * (uu + vv + ww), cov(th, w),
            mean(S[5] / rho), mean(S[6] / rho) if moist else zero, mean(S[7] / rho) if moist else zero, zero, zero, zero]
    return torch.stack(cols, dim=1)


class _LES:
    """The RK3 step of the model: flux-form advection, pressure gradient, buoyancy, Coriolis, Rayleigh
    damping and filter on every stage, SGS turbulence, surface layer and condensation on the last.
    Arrays are [x][y][z]; 'extended' ones hold levels -3 .. nz+2."""

    def __init__(self, g):
        self.g, self.p = g, g.p
        p, f = g.p, lambda v: float(np.float32(v))
        self.case, self.nz = g.case, g.nz
        self.dt = f(p["dt"])
        self.dxi = self.dyi = 1 / f(p["d_xi"])
        self.dzi = 1 / f(p["d_zeta"])
        self.ck, self.cs = f(p["c_k"]), f(p["c_s"])
        self.tke = p["TKESelector"] > 0
        self.moist = p["moistureSelector"] > 0
        self.fh = 1.45842e-4 * math.sin(math.radians(f(p["coriolisLatitude"])))
        self.rv_r = f(461.60) / g.R
        self.delta = (f(p["d_xi"]) ** 2 * f(p["d_zeta"]) * g.D) ** (1 / 3)
        self.lv = 2.5e6
        N = _NH + g.nz
        zt = g.z[..., N - 1:N]
        s = torch.sin(0.5 * math.pi * (1 - (zt - g.z) / f(p["dampingLayerDepth"])))
        self.damp = torch.where(g.z >= zt - f(p["dampingLayerDepth"]), 0.2 * s * s, torch.zeros_like(s))[..., _NH:N]
        self.sl = slice(_NH, N)

    # -- small operators --
    @staticmethod
    def rx(a, n=1):
        return torch.roll(a, n, 0)

    @staticmethod
    def ry(a, n=1):
        return torch.roll(a, n, 1)

    def ext(self, a, kind):
        nx, ny, nz = a.shape
        g, N = self.g, _NH + self.nz
        if kind in ("rho", "rth"):
            b = (g.rho if kind == "rho" else g.rth).expand(nx, ny, nz + 6)
            return torch.cat([b[..., :_NH], a, b[..., N:]], 2)
        lo = a[..., :1].expand(nx, ny, 3)
        if kind == "u":
            hi = (g.ug * g.rho)[..., N - 1:N].expand(nx, ny, 3)
        elif kind in ("v", "w", "e"):
            hi = torch.zeros_like(lo)
        else:
            hi = a[..., -1:].expand(nx, ny, 3)
        return torch.cat([lo, a, hi], 2)

    @staticmethod
    def weno(a, b, c, d, e):
        t = 1e-6
        f1, f2, f3 = a / 3 - 7 / 6 * b + 11 / 6 * c, -b / 6 + 5 / 6 * c + d / 3, c / 3 + 5 / 6 * d - e / 6
        b1 = 13 / 12 * (a - 2 * b + c) ** 2 + 0.25 * (a - 4 * b + 3 * c) ** 2
        b2 = 13 / 12 * (b - 2 * c + d) ** 2 + 0.25 * (b - d) ** 2
        b3 = 13 / 12 * (c - 2 * d + e) ** 2 + 0.25 * (3 * c - 4 * d + e) ** 2
        w1, w2, w3 = 0.1 / (t + b1) ** 2, 0.6 / (t + b2) ** 2, 0.3 / (t + b3) ** 2
        return (w1 * f1 + w2 * f2 + w3 * f3) / (w1 + w2 + w3)

    def flux(self, scheme, U, m3, m2, m1, c0, p1, p2):
        sg = torch.where(torch.signbit(U), -1.0, 1.0).double()
        if scheme == "hyb56":
            return U / 60 * (37 * (c0 + m1) - 8 * (p1 + m2) + (p2 + m3) - sg * ((p2 - m3) - 5 * (p1 - m2) + 10 * (c0 - m1)))
        if scheme == "hyb34":
            return U / 12 * (7 * (c0 + m1) - (p1 + m2) + sg * ((p1 - m2) - 3 * (c0 - m1)))
        return U * torch.where(sg > 0, self.weno(m3, m2, m1, c0, p1), self.weno(p2, p1, c0, m1, m2))

    def divergence(self, scheme, E, U, V, W):
        a = E[..., self.sl]
        out = 0
        for roll, vel in ((self.rx, U), (self.ry, V)):
            fl = self.flux(scheme, vel, roll(a, 3), roll(a, 2), roll(a, 1), a, roll(a, -1), roll(a, -2))
            out = out + roll(fl, -1) - fl
        n = self.nz + 1
        fl = self.flux(scheme, W, *(E[..., j:j + n] for j in range(6)))
        return out + fl[..., 1:] - fl[..., :-1]

    # -- one stage's tendency --
    def tendency(self, S, physics, it):
        g, sl, nz, p = self.g, self.sl, self.nz, self.p
        rx, ry, dxi, dyi, dzi = self.rx, self.ry, self.dxi, self.dyi, self.dzi
        kinds = ["rho", "u", "v", "w", "rth"] + (["e"] if self.tke else []) + (["q", "q"] if self.moist else [])
        E = [self.ext(S[k], kind) for k, kind in enumerate(kinds)]
        rho, u, v, w, rth = S[0], S[1], S[2], S[3], S[4]
        D, J = g.D[..., sl], g.J33[..., sl]
        Dr = D / rho
        U = 0.5 * dxi * (Dr * u + rx(Dr * u))
        V = 0.5 * dyi * (Dr * v + ry(Dr * v))
        wz = g.D * g.J33 * E[3] / E[0]
        W = 0.5 * dzi * (wz[..., 3:4 + nz] + wz[..., 2:3 + nz])
        W[..., 0] = 0
        W[..., -1] = 0
        schemes = ["hyb56"] * (6 if self.tke else 5)
        if self.moist:
            schemes += ["hyb34" if p["moistureAdvSelectorQv"] == 2 else "hyb56", "weno5"]
        F = torch.stack([-self.divergence(s, e, U, V, W) / D for s, e in zip(schemes, E)])
        # pressure gradient
        mf = 1 + self.rv_r * S[6] / rho * 1e-3 if self.moist else 1.0
        pp = (rth * mf * g.c1) ** g.gam - (g.rth[..., sl] * g.c1) ** g.gam
        pe = torch.cat([pp[..., :1], pp, pp[..., -1:]], 2)
        fac = 1 / (1 + (S[6] + S[7]) / rho * 1e-3) if self.moist else 1.0
        F[1] -= fac * 0.5 * dxi * (rx(pp, -1) - rx(pp))
        F[2] -= fac * 0.5 * dyi * (ry(pp, -1) - ry(pp))
        F[3] -= fac * 0.5 * dzi * J * (pe[..., 2:] - pe[..., :-2])
        # damping, buoyancy, Coriolis
        F[3] -= self.damp * w
        tot = rho + (S[6] + S[7]) * 1e-3 if self.moist else rho
        F[3] -= rho / tot * g.g * (tot - g.rho[..., sl])
        F[1] += self.fh * v / rho
        F[2] -= self.fh * (u / rho - g.ug[..., sl])
        if physics:
            self.physics(F, S, E, it)
        if p["filterSelector"]:
            a = [E[3][..., j:j + nz] for j in range(7)]
            gm, gp = a[3] - a[2], a[4] - a[3]
            fm = 10 * gm - 5 * (a[4] - a[1]) + (a[5] - a[0])
            fp = 10 * gp - 5 * (a[5] - a[2]) + (a[6] - a[1])
            fm, fp = torch.where(torch.signbit(gm * fm), 0.0, fm), torch.where(torch.signbit(gp * fp), 0.0, fp)
            F[3] += 0.015625 * p["filter_6th_coeff"] / self.dt * (fp - fm)
        return F

    def physics(self, F, S, E, it):
        g, nz, p = self.g, self.nz, self.p
        rx, ry, dxi, dyi, dzi = self.rx, self.ry, self.dxi, self.dyi, self.dzi
        ri = 1 / E[0]
        vel = [E[k] * ri for k in (1, 2, 3, 4)]
        lev = lambda a, lo, n: a[..., _NH + lo:_NH + lo + n]      # n levels of an extended array from level lo
        J = lev(g.J33, 0, nz + 1)                                 # faces 0 .. nz
        (u, v, w, th), (um, vm, wm, thm) = ([lev(a, k, nz + 1) for a in vel] for k in (0, -1))
        dx, dy = (lambda a: dxi * (a - rx(a))), (lambda a: dyi * (a - ry(a)))
        dzf = lambda a, am: J * dzi * (a - am)
        s11, s22, s33 = dx(u), dy(v), dzf(w, wm)
        s21 = 0.25 * (dx(v) + ry(dx(v)) + dy(u) + rx(dy(u)))
        s31 = 0.25 * (dx(w) + dx(wm) + dzf(u, um) + rx(dzf(u, um)))
        s32 = 0.25 * (dy(w) + dy(wm) + dzf(v, vm) + ry(dzf(v, vm)))
        dl = lev(self.delta, 0, nz + 1)
        rho = lev(E[0], 0, nz + 1)
        if self.tke:
            n2 = g.g / lev(vel[3], -1, nz + 2) * 0.5 * lev(g.J33, -1, nz + 2) * dzi * (lev(vel[3], 0, nz + 2) - lev(vel[3], -2, nz + 2))
            e = lev(E[5] * ri, -1, nz + 2)
            d = lev(self.delta, -1, nz + 2).expand_as(e)
            l = torch.where(n2 > 0, torch.maximum(torch.minimum(0.76 * e.sqrt() * n2.clamp_min(1e-300) ** -0.5, d),
                                                  torch.full_like(d, 1e-2)), d)
            q = l * e.sqrt()
            K = self.ck * 0.5 * (q[..., 1:] + q[..., :-1])
            l = l[..., 1:]
            pr = 1 + 2 * l / dl
            iso = 2 / 3 * (rho * K * (s11 + s22 + s33) + lev(E[5], 0, nz + 1))
        else:
            t1 = 0.5 * (s11 ** 2 + s22 ** 2 + s33 ** 2) + s21 ** 2 + s31 ** 2 + s32 ** 2
            t2 = (3 * g.g / th * dzf(th, thm)).clamp_min(0)
            K = (self.cs * dl) ** 2 * (t1 - t2).clamp_min(0).sqrt()
            pr, iso = 3.0, 0.0
        A = rho * K
        T = [-2 * A * s11 + iso, -2 * A * s21, -2 * A * s31, -2 * A * s32, -2 * A * s22 + iso, -2 * A * s33 + iso,
             -A * pr * dx(th), -A * pr * dy(th), -A * pr * dzf(th, thm)]
        M = []
        if self.moist:
            for k in (6, 7):
                c = E[k] * ri
                c0, cm = lev(c, 0, nz + 1), lev(c, -1, nz + 1)
                M.append([-A * pr * dx(c0), -A * pr * dy(c0), -A * pr * dzf(c0, cm)])
        self.surface(S, T, M, it)
        self.tau = T
        z0 = g.J33[..., self.sl] * dzi
        hx, hy = (lambda a: dxi * (rx(a, -1) - a)[..., :-1]), (lambda a: dyi * (ry(a, -1) - a)[..., :-1])
        vz = lambda a: z0 * (a[..., 1:] - a[..., :-1])
        F[1] -= hx(T[0]) + hy(T[1]) + vz(T[2])
        F[2] -= hx(T[1]) + hy(T[4]) + vz(T[3])
        F[3] -= hx(T[2]) + hy(T[3]) + vz(T[5])
        F[4] -= hx(T[6]) + hy(T[7]) + vz(T[8])
        for k, m in enumerate(M):
            F[6 + k] -= hx(m[0]) + hy(m[1]) + vz(m[2])
        c = lambda a: a[..., :-1]
        if self.tke:
            cx = lambda a: 0.5 * dxi * (rx(a, -1) - rx(a))
            cy = lambda a: 0.5 * dyi * (ry(a, -1) - ry(a))
            cz = lambda k: 0.5 * z0 * (lev(vel[k], 1, nz) - lev(vel[k], -1, nz))
            ec, lc = lev(E[5] * ri, 0, nz), c(l)
            src = g.g / c(th) * c(T[8])
            src -= (1.9 * self.ck + (0.93 - 1.9 * self.ck) * lc / c(dl)) * S[5] * ec.sqrt() / lc
            src -= (c(T[0]) * cx(c(u)) + c(T[1]) * cy(c(u)) + c(T[2]) * cz(0) + c(T[1]) * cx(c(v)) + c(T[4]) * cy(c(v))
                    + c(T[3]) * cz(1) + c(T[2]) * cx(c(w)) + c(T[3]) * cy(c(w)) + c(T[5]) * cz(2))
            ee = E[5] * ri
            Ac = c(A)
            fx, fy = cx(ec) * Ac, cy(ec) * Ac
            dez = 0.5 * lev(g.J33, -1, nz + 2) * dzi * (lev(ee, 0, nz + 2) - lev(ee, -2, nz + 2))
            fz = dez * torch.cat([torch.zeros_like(A[..., :1]), A], 2)
            src += dxi * (rx(fx, -1) - rx(fx)) + dyi * (ry(fy, -1) - ry(fy)) + z0 * (fz[..., 2:] - fz[..., :-2])
            F[5] += src
        if self.moist and it % int(round(max(p["moistureMPcallTscale"], p["dt"]) / p["dt"])) == 0:
            self.condense(F, S)

    def surface(self, S, T, M, it):
        g, p = self.g, self.p
        f = lambda v: float(np.float32(v))
        k2 = f(0.4) ** 2
        rho, ru, rv = S[0][..., 0], S[1][..., 0], S[2][..., 0]
        u, v, th1 = ru / rho, rv / rho, S[4][..., 0] / rho
        z1 = (0.5 / (self.dzi * g.J33[..., _NH])).expand_as(u)
        lz, lzt = torch.log((z1 + f(p["surflayer_z0"])) / f(p["surflayer_z0"])), torch.log((z1 + f(p["surflayer_z0t"])) / f(p["surflayer_z0t"]))
        sp = torch.sqrt(u * u + v * v)
        sel = p["surflayerSelector"]
        if it == 0:
            self.cd, self.ch = k2 / lz ** 2, k2 / lzt ** 2
            self.hf = torch.full_like(u, f(p["surflayer_wth"]) if sel == 1 else 0.0)
            self.tsk = torch.full_like(u, f(p["temp_grnd"]))
        ex = (g.pref / f(p["pres_grnd"])) ** g.rcp
        if sel == 2:
            tf = int(round(10.0 / p["dt"]))
            if it % tf == 0:
                self.tsk = self.tsk + f(p["surflayer_tr"]) * self.dt * tf / 3600.0
            self.hf = self.ch * sp * (self.tsk * ex - th1)
        cd = self.cd
        for _ in range(6):
            us = (cd * sp * sp).sqrt()
            iol = (-(f(0.4) * g.g * self.hf) / (us ** 3 * th1)).clamp(-1, 1)
            zol = iol * (z1 + f(p["surflayer_z0"]))
            xi = (1 - 16 * zol.clamp_max(0)) ** 0.25
            pm = torch.where(zol < 0, torch.log(0.5 * (1 + xi * xi) * (0.5 * (1 + xi)) ** 2) - 2 * torch.atan(xi) + 0.5 * math.pi, -5 * zol)
            ph = torch.where(zol < 0, 2 * torch.log(0.5 * (1 + xi * xi)), -5 * zol)
            cd, ch = k2 / (lz - pm) ** 2, k2 / ((lzt - pm) * (lzt - ph))
            if sel > 1:
                self.hf = ch * sp * (self.tsk * ex - th1)
        self.cd, self.ch = cd, ch
        tx, ty = -cd * sp * ru, -cd * sp * rv
        self.ust = (tx * tx + ty * ty) ** 0.25
        T[2][..., 0], T[3][..., 0], T[8][..., 0] = tx, ty, self.hf * rho
        if M:
            M[0][2][..., 0] = f(p["surflayer_wq"]) * rho

    def condense(self, F, S):
        g, p = self.g, self.p
        rho, rth, qv, ql = S[0], S[4], S[6], S[7]
        th = rth / rho
        rvap = float(np.float32(461.60))
        pr = (g.rth[..., self.sl] * g.c1) ** g.gam
        T = th * (pr / g.pref) ** g.rcp
        tc = (T - 273.16).clamp_min(-80.0)
        warm = [6.11239921, 0.443987641, 0.142986287e-1, 0.264847430e-3, 0.302950461e-5, 0.206739458e-7, 0.640689451e-10,
                -0.952447341e-13, -0.976195544e-15]
        cold = [6.11147274, 0.503160820, 0.188439774e-1, 0.420895665e-3, 0.615021634e-5, 0.602588177e-7, 0.385852041e-9,
                0.146898966e-11, 0.252751365e-14]
        poly = lambda c: sum(a * tc ** n for n, a in enumerate(c)) * 100
        es = torch.minimum(0.99 * pr, torch.where(T >= 273.15, poly(warm), poly(cold)))
        rvs = es / (pr - es) / self.rv_r * rho
        ff = (qv * 1e-3 - rvs) / (1 + self.lv ** 2 * rvs / rho / (g.cp * rvap * T * T))
        fc = (ff.clamp_min(0) - torch.minimum(ql * 1e-3, -ff).clamp_min(0)) / p["moistureCondTscale"]
        F[6] -= fc * 1e3
        F[7] += fc * 1e3
        tl = th * (((rth * g.c1) ** g.gam) / g.pref) ** g.rcp
        F[4] += th * self.lv / (tl * g.cp) * fc

    def forcing(self, S, it):
        """Large-scale advection and subsidence of the slab means, due every lsf_freq seconds."""
        p, g, nz = self.p, self.g, self.nz
        itn = int(round(p["lsf_freq"] / p["dt"])) if p["lsfSelector"] else 0
        if not itn or it < itn or it % itn:
            return None
        nx, ny = S[0].shape[:2]
        wx, wy = (torch.ones(n, dtype=torch.float64, device=_DEV) for n in (nx, ny))
        for a in (wx, wy):                       # the mean spans the halo-inclusive plane
            a[:_NH] += 1
            a[-_NH:] += 1
        mean = lambda a: torch.einsum("xyz,x,y->z", a, wx, wy) / ((nx + 6) * (ny + 6))
        M = [mean(self.ext(S[k], kind)[..., 2:nz + 4]) for k, kind in ((0, "rho"), (1, "u"), (2, "v"), (4, "rth"), (6, "q"))]
        z, rho = g.z[0, 0, self.sl], g.rho[0, 0, self.sl]

        def piece(n):
            a, b, c, z1, z2 = (p[f"lsf_{n}_{k}"] for k in ("surf", "lev1", "lev2", "zlev1", "zlev2"))
            r = torch.where(z <= z1, a + (b - a) / z1 * z, torch.where(z <= z2, b + (c - b) / (z2 - z1) * (z - z1), c + 0 * z))
            return r * rho * itn / 3600.0

        fw, dz = piece("w"), g.z[0, 0, 4:4 + nz] - g.z[0, 0, 2:2 + nz]
        sub = [fw * rho * (m[2:] / M[0][2:] - m[:-2] / M[0][:-2]) / dz for m in M[1:]]
        out = torch.zeros((8, 1, 1, nz), dtype=torch.float64, device=_DEV)
        out[1, 0, 0], out[2, 0, 0] = -sub[0], -sub[1]
        out[4, 0, 0], out[6, 0, 0] = piece("th") - sub[2], piece("qv") - sub[3]
        return out

    def steps(self, S, n):
        for it in range(n):
            base, cur = S, S
            lsf = self.forcing(S, it)
            for stage, c in enumerate((1 / 3, 0.5, 1.0)):
                F = self.tendency(cur, stage == 2, it)
                if lsf is not None and stage == 2:
                    F += lsf
                cur = base + c * self.dt * F
                if self.tke:
                    cur[5].clamp_min_(1e-10)
                if self.moist:
                    cur[6:8].clamp_min_(0.0)
            S = cur
        return {"state": S, "ust": self.ust, "hf": self.hf, "tsk": self.tsk,
                "tau": torch.stack([t[..., :-1] for t in self.tau])}
