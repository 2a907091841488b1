"""The work that users of this solver have it do, as measurable cases.

A case is a dict of plain values.  `prepare` builds what a program holds before it calls
(mesh, solver, state), `run` makes one pass through the public API, `exact` restates the
pass in plain float64 torch, `work` counts the bytes and operations that the pass cannot do
without.  The meshes, schemes and states are those of the repository's benchmark and tests:
the wall-modelled channel (uniform x and z, tanh-clustered y, constant mass flux), the
smooth ramp (curvilinear, synthetic inflow, sponge), ensembles of uneven channels, and a
skewed periodic box.  States are a mean profile plus seeded Gaussian velocity and density noise.
"""
import math

import numpy as np
import torch

import wmles_jax_amd as wmx

NG = 3
GAMMA, R_GAS, PR, PR_T = 1.4, 287.05, 0.72, 0.9
CP = GAMMA * R_GAS / (GAMMA - 1.0)


# ------------------------------------------------------------------------------- cases
def _channel(name, n, prec, scheme="hybrid", sgs="vreman", blocks=1, call="step", wm="newton",
             n_match=1, Re_b=2.0e4):
    return {"name": name, "kind": "channel", "nx": n[0], "ny": n[1], "nz": n[2], "prec": prec,
            "scheme": scheme, "sgs": sgs, "blocks": blocks, "call": call, "wm": wm,
            "n_match": n_match, "Re_b": Re_b}


def listed():
    return [
        # the smallest call: a unit-test sized channel in the plain FP64 form (launch latency)
        _channel("channel_24_fp64", (24, 16, 12), "fp64", "kep4"),
        # a coarse ragged channel, the size of a quick look: still latency
        _channel("channel_45_fp32", (45, 39, 35), "fp32"),
        # two blocks, odd sizes, KEP2 + WALE, by the reference driver's two calls
        _channel("channel_odd_2blk_fp32", (133, 75, 61), "fp32", "kep2", "wale", blocks=2, call="advance"),
        # the repository's headline benchmark, both arithmetic forms
        _channel("channel_256_fp32", (256, 128, 128), "fp32"),
        _channel("channel_256_fp64", (256, 128, 128), "fp64"),
        # the learned wall model sampling off the wall
        _channel("channel_learned_fp32", (128, 96, 96), "fp32", wm="learned", n_match=10, Re_b=1.0e5),
        # the largest: the wall-resolving grid at Re_b 1e5
        _channel("channel_512_fp32", (512, 256, 256), "fp32", n_match=10, Re_b=1.0e5),
        # curvilinear block with synthetic inflow and sponge, both forms
        {"name": "ramp_512_fp32", "kind": "ramp", "nx": 512, "ny": 128, "nz": 64, "prec": "fp32"},
        {"name": "ramp_190_fp64", "kind": "ramp", "nx": 190, "ny": 63, "nz": 33, "prec": "fp64"},
        # sixteen uneven multiblock channels in one plan
        {"name": "ensemble_16_fp32", "kind": "ensemble", "cases": 16, "prec": "fp32", "scheme": "kep2",
         "sgs": "wale"},
        # right-hand side of a skewed two-block mesh (verification, user time integrators)
        {"name": "skewed_rhs_fp64", "kind": "skewed", "nx": 128, "ny": 72, "nz": 56, "scheme": "muscl",
         "sgs": "smagorinsky"},
        # what a run writes every so many steps: dt, wall stresses, plane averages
        _channel("channel_diagnostics", (192, 96, 96), "fp64", call="diagnostics"),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["channel"] * 5 + ["ramp", "ramp", "ensemble", "skewed"])
    prec = rng.choice(["fp32", "fp64"])
    if kind == "channel":
        case = _channel("", (size(16, 300), size(12, 150), size(12, 150)), prec,
                        rng.choice(["hybrid", "hybrid", "kep2", "kep4", "keep4", "muscl"]),
                        rng.choice(["vreman", "wale", "smagorinsky", "none"]), rng.choice([1, 1, 2, 3]),
                        rng.choice(["step", "step", "advance", "diagnostics"]), "newton",
                        rng.choice([1, 1, 3]), math.exp(rng.uniform(math.log(5e3), math.log(1e5))))
        if case["nx"] < 8 * case["blocks"]:
            case["blocks"] = 1
    elif kind == "ramp":
        case = {"kind": kind, "nx": size(64, 512), "ny": size(24, 128), "nz": size(12, 64), "prec": prec}
    elif kind == "ensemble":
        case = {"kind": kind, "cases": rng.randint(2, 16), "prec": prec,
                "scheme": rng.choice(["kep2", "hybrid"]), "sgs": rng.choice(["wale", "vreman"])}
    else:
        case = {"kind": kind, "nx": size(16, 192), "ny": size(10, 96), "nz": size(8, 96),
                "scheme": rng.choice(["muscl", "hybrid", "kep4"]),
                "sgs": rng.choice(["smagorinsky", "vreman"])}
    case.pop("name", None)
    return case


# ------------------------------------------------------------------- meshes and states
def _scheme(name):
    return {"kep2": lambda: wmx.KEP(2), "kep4": lambda: wmx.KEP(4), "keep4": lambda: wmx.KEEP(4),
            "muscl": lambda: wmx.MUSCLHLLC("albada"),
            "hybrid": lambda: wmx.Hybrid(wmx.KEP(4), wmx.MUSCLHLLC("albada"))}[name]()


def _mu(T):
    return 1.716e-5 * (T / 273.15) ** 1.5 * (273.15 + 110.4) / (T + 110.4)


def _channel_scales(Re_b, Ma_b=0.3, T0=300.0, rho0=1.2):
    Ub = Ma_b * math.sqrt(GAMMA * R_GAS * T0)
    return {"rho0": rho0, "p0": rho0 * R_GAS * T0, "Ub": Ub, "d": Re_b * (_mu(T0) / rho0) / Ub}


def _channel_axes(case):
    d = _channel_scales(case["Re_b"])["d"]
    eta = np.linspace(0.0, 1.0, case["ny"] + 1)
    return (np.linspace(0.0, 2.0 * np.pi * d, case["nx"] + 1),
            d * (1.0 + np.tanh(2.0 * (2.0 * eta - 1.0)) / np.tanh(2.0)),
            np.linspace(0.0, np.pi * d, case["nz"] + 1))


def _cuts(case):
    """Block boundaries along i; several blocks are uneven."""
    nb, nx = case.get("blocks", 1), case["nx"]
    if "cuts" in case:
        return list(case["cuts"])
    return [0] + [nx * (3 * b) // (3 * nb + 1) for b in range(1, nb)] + [nx]


def _box(x, y, z):
    return np.stack(np.meshgrid(x, y, z, indexing="ij"))


def _ramp_props():
    return wmx.flow_properties(0.2, 667000.0)


def _ramp_wall(xl):
    s = np.clip(xl, 0.0, 1.0)
    return 0.22 * (1.0 - (10 * s ** 3 - 15 * s ** 4 + 6 * s ** 5))


def _ramp_profile():
    yt = 0.22 + 0.52 * np.linspace(0.0, 1.0, 64) ** 2
    U = np.minimum(((yt - 0.22) / 0.028) ** (1.0 / 7.0), 1.0)
    a = 0.08 ** 2 + 0.0 * yt
    return np.stack([yt, U, 0.0 * yt, a, a, a, 0.0 * yt], axis=1)


def _ramp_nodes(case, L):
    x = np.linspace(-0.76, 4.0, case["nx"] + 1)
    eta = np.linspace(0.0, 1.0, case["ny"] + 1)
    s = 1.0 + np.tanh(2.5 * (eta - 1.0)) / np.tanh(2.5)
    wall = _ramp_wall(x)
    y = wall[:, None] + (0.74 - wall[:, None]) * s[None, :]
    z = np.linspace(0.0, 0.288, case["nz"] + 1)
    shp = (len(x), len(eta), len(z))
    return L * np.stack([np.broadcast_to(x[:, None, None], shp), np.broadcast_to(y[:, :, None], shp),
                         np.broadcast_to(z[None, None, :], shp)])


BOX = (1.0, 0.6, 0.5)                     # the skewed box


def _skewed_nodes(case):
    X, Y, Z = _box(*[BOX[a] * np.arange(case[k] + 1) / case[k] for a, k in enumerate(("nx", "ny", "nz"))])
    sx, sy, sz = (2 * np.pi * c / l for c, l in zip((X, Y, Z), BOX))
    return np.stack([X + 0.04 * np.sin(sy) * np.sin(sz), Y + 0.02 * np.sin(sx),
                     Z + 0.02 * np.sin(sx) * np.cos(sy)])


def _nodes(case):
    """Nodes of the whole domain (blocks are runs of i cells of it) and its extents (x, z)."""
    if case["kind"] == "channel":
        x, y, z = _channel_axes(case)
        return _box(x, y, z), (x[-1], z[-1])
    if case["kind"] == "ramp":
        L = _ramp_props()["L"]
        return _ramp_nodes(case, L), (None, 0.288 * L)
    return _skewed_nodes(case), (BOX[0], BOX[2])


def _prim(case, xc, gen):
    """Primitive state at the cell centres xc (3, ...): mean profile, velocity noise and 1% of
    density (temperature) noise."""
    noise = torch.randn((4,) + tuple(xc.shape[1:]), generator=gen, device=xc.device, dtype=torch.float64)
    one, noise = 1.0 + 0.01 * noise[3], noise[:3]
    if case["kind"] == "channel":
        s = _channel_scales(case["Re_b"])
        eta = xc[1] / s["d"] - 1.0
        u = s["Ub"] * (0.75 * (1.0 - eta * eta)
                       + (4.0 / 7.0) * torch.clamp(1.0 - eta.abs(), min=1e-3) ** (1.0 / 7.0))
        vel, rho, p = 0.05 * s["Ub"] * noise, s["rho0"] * one, torch.full_like(u, s["p0"])
        vel[0] += u
    elif case["kind"] == "ramp":
        pr = _ramp_props()
        xl = torch.clamp(xc[0] / pr["L"], 0.0, 1.0)
        wall = 0.22 * (1.0 - (10 * xl ** 3 - 15 * xl ** 4 + 6 * xl ** 5))
        yd = torch.clamp(xc[1] / pr["L"] - wall, min=0.0)
        vel, rho, p = 0.02 * pr["U_inf"] * noise, pr["rho_inf"] * one, torch.full_like(xl, pr["p_inf"])
        vel[0] += pr["U_inf"] * torch.clamp((yd / 0.028) ** (1.0 / 7.0), max=1.0)
    else:
        x, y, z = (2 * math.pi * xc[a] / BOX[a] for a in range(3))
        rho = 1.2 * one * (1 + 0.05 * torch.sin(x) * torch.cos(z))
        p = 1e5 * (1 + 0.03 * torch.cos(x) * torch.sin(y))
        vel = 2.0 * noise
        vel[0] += 60 * torch.sin(y) + 20 * torch.cos(z)
        vel[1] += 15 * torch.sin(x) * torch.sin(z)
        vel[2] += 10 * torch.cos(x) + 5 * torch.sin(y)
    return torch.cat([rho[None], vel, p[None]])


def _members(case):
    """The channel cases of an ensemble: uneven sizes and splits, fixed by the member number."""
    out = []
    for c in range(case["cases"]):
        r = np.random.default_rng(c)
        nx, ny, nz = (16 * int(r.integers(lo, hi)) for lo, hi in ((4, 13), (3, 7), (2, 5)))
        nb = int(r.integers(2, 5))
        w = np.cumsum(r.uniform(0.5, 1.5, nb))
        cuts = [0] + [int(round(v)) for v in nx * w[:-1] / w[-1]] + [nx]
        m = _channel("", (nx, ny, nz), case["prec"], case["scheme"], case["sgs"], nb,
                     Re_b=float(np.exp(r.uniform(np.log(5e3), np.log(4e4)))))
        out.append(dict(m, cuts=cuts))
    return out


def _learned_model():
    model = wmx.LearnedWallModel()
    model.train(n_samples=65536, batch=4096, steps=1500, seed=0)
    return model


def _build(case, model=None):
    """(mesh, solver) of one channel, ramp or skewed case."""
    nodes, (Lx, Lz) = _nodes(case)
    cuts = _cuts(case) if case["kind"] != "skewed" else [0, case["nx"] // 2, case["nx"]]
    blocks = [wmx.Block(f"B{b}", nodes[:, lo:hi + 1]) for b, (lo, hi) in enumerate(zip(cuts, cuts[1:]))]
    mesh = wmx.Mesh(blocks)
    kw = {"sgs": case.get("sgs", "vreman"), "precision": case.get("prec", "fp64")}
    if case["kind"] != "ramp":
        for b, blk in enumerate(blocks):
            nxt = blocks[(b + 1) % len(blocks)]
            mesh.connect(blk, "imax", nxt, "imin", shift=(Lx if nxt is blocks[0] else 0.0, 0.0, 0.0))
    for blk in blocks:
        mesh.connect(blk, "kmin", blk, "kmax", shift=(0.0, 0.0, -Lz))
        if case["kind"] == "channel":
            for face in ("jmin", "jmax"):
                blk.set_bc(face, wmx.WallModel(model or wmx.EquilibriumWallModel(), T_wall=300.0,
                                               n_match=case["n_match"]))
        elif case["kind"] == "skewed":
            for face in ("jmin", "jmax"):
                blk.set_bc(face, wmx.SlipWall())
    if case["kind"] == "channel":
        s = _channel_scales(case["Re_b"])
        kw["constraints"] = [wmx.ConstantMassFlux(0, s["rho0"] * s["Ub"])]
    elif case["kind"] == "ramp":
        pr = _ramp_props()
        inf = np.array([pr["rho_inf"], pr["U_inf"], 0.0, 0.0, pr["p_inf"]])
        blocks[0].set_bc("imin", wmx.SmoothRampInflow(pr, _ramp_profile(), seed=0, n_modes=64,
                                                      span_cells=case["nz"]))
        blocks[0].set_bc("imax", wmx.CharacteristicFarfield(inf))
        blocks[0].set_bc("jmin", wmx.WallModel(wmx.EquilibriumWallModel(), T_wall=None))
        blocks[0].set_bc("jmax", wmx.SlipWall())
        kw.update(sources=[wmx.SmoothRampSponge(pr, 3.0, 4.0, 1.0)], cfl=0.5)
    mesh.finalize()
    return mesh, wmx.Solver(mesh, wmx.Gas(), _scheme(case.get("scheme", "hybrid")), **kw)


def _state(case, solver, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    return tuple(solver.gas.prim_to_cons(_prim(case, g.xc, gen)).contiguous() for g in solver.geoms)


RAMP_TIME = 1.0e-3                        # the inflow's fluctuations move with time


def prepare(case, seed):
    if case["kind"] == "ensemble":
        built = [(m, _build(m)[1]) for m in _members(case)]
        return {"case": case, "solver": wmx.EnsembleSolver([s for _, s in built]),
                "Q": [_state(m, s, seed * 64 + c) for c, (m, s) in enumerate(built)]}
    mesh, solver = _build(case, _learned_model() if case.get("wm") == "learned" else None)
    return {"case": case, "mesh": mesh, "solver": solver, "Q": _state(case, solver, seed)}


def run(state):
    case, s, Q = state["case"], state["solver"], state["Q"]
    if case["kind"] == "skewed":
        return s.rhs(Q)
    if case["kind"] == "ramp":
        return s.step(Q, time=RAMP_TIME)
    if case["kind"] == "channel" and case["call"] == "advance":
        dt = s.max_dt(Q)
        return s.advance(Q, dt), dt
    if case["kind"] == "channel" and case["call"] == "diagnostics":
        dt = s.max_dt(Q)
        stats = wmx.PlaneStats(state["mesh"], s)
        stats.accumulate(Q)
        y, avg = stats.result()
        return {"dt": dt, "wall": s.wall_stats(Q), "y": y, "profiles": avg, "tau": stats.mean_tau_w}
    return s.step(Q)


# ------------------------------------------------------------------------ counted work
def _cells(case):
    if case["kind"] == "ensemble":
        return sum(_cells(m) for m in _members(case))
    return case["nx"] * case["ny"] * case["nz"]


def work(case):
    """State in and out once (five doubles a cell each way) and the grid's nodes (three
    doubles a cell where they are not products of lines); the operations of three
    right-hand sides (one for `rhs`): per cell three faces and the cell's gradients, closure
    and update."""
    n = _cells(case)
    curved = 24.0 if case["kind"] in ("ramp", "skewed") else 0.0
    if case.get("call") == "diagnostics":
        return {"bytes": 40.0 * n, "flops": 90.0 * n}
    face = {"kep2": 35, "kep4": 95, "keep4": 120, "muscl": 230, "hybrid": 160}[case.get("scheme", "hybrid")]
    per_stage = 3 * (face + 60) + 110 + 60
    return {"bytes": (80.0 + curved) * n, "flops": float(per_stage) * n * (1 if case["kind"] == "skewed" else 3)}


# ------------------------------------------- the pass in plain float64 torch (one block)
def _sl(d, s, nd):
    """Index of slice s along spatial axis d of an nd-dimensional array."""
    at = [slice(None)] * nd
    at[nd - 3 + d] = s
    return tuple(at)


def _dot(a, b):
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]


def _cross(a, b):
    return torch.stack([a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]])


class _Grid:
    """Ghosted metrics of the whole domain: periodic directions continue the nodes by a shift,
    the others reflect them through the boundary plane."""

    def __init__(self, nodes, periods):
        X = torch.as_tensor(np.ascontiguousarray(nodes), device="cuda")
        self.n = tuple(k - 1 for k in X.shape[1:])
        self.periodic = tuple(p is not None for p in periods)
        for d in range(3):
            n = X.shape[1 + d] - 1
            lo = X[_sl(d, slice(n - NG, n), 4)] if periods[d] else X[_sl(d, slice(1, NG + 1), 4)].flip(1 + d)
            hi = X[_sl(d, slice(1, NG + 1), 4)] if periods[d] else X[_sl(d, slice(n - NG, n), 4)].flip(1 + d)
            if periods[d]:
                sh = torch.zeros(3, 1, 1, 1, dtype=X.dtype, device=X.device)
                sh[d] = periods[d]
                X = torch.cat([lo - sh, X, hi + sh], 1 + d)
            else:
                X = torch.cat([2 * X[_sl(d, slice(0, 1), 4)] - lo, X, 2 * X[_sl(d, slice(n, n + 1), 4)] - hi], 1 + d)
        self.S, self.xf, vol = [], [], 0.0
        for d in range(3):
            a, b = (d + 1) % 3, (d + 2) % 3

            def corner(ia, ib):
                return X[_sl(a, slice(ia, X.shape[1 + a] - 1 + ia), 4)][_sl(b, slice(ib, X.shape[1 + b] - 1 + ib), 4)]
            c00, c10, c01, c11 = corner(0, 0), corner(1, 0), corner(0, 1), corner(1, 1)
            S, f = 0.5 * _cross(c11 - c00, c01 - c10), 0.25 * (c00 + c10 + c01 + c11)
            vol = vol + torch.diff(_dot(f, S), dim=d) / 3.0
            self.S.append(S)
            self.xf.append(f)
        self.vol = vol
        self.xc = sum(X[:, i:X.shape[1] - 1 + i, j:X.shape[2] - 1 + j, k:X.shape[3] - 1 + k]
                      for i in (0, 1) for j in (0, 1) for k in (0, 1)) / 8.0

    def inner(self, a):
        return a[..., NG:NG + self.n[0], NG:NG + self.n[1], NG:NG + self.n[2]]

    def slab(self, a, d, lo, hi):
        """Cells (or faces) ng + lo .. ng + n_d + hi along d, interior along the others."""
        at = [slice(None)] * (a.ndim - 3) + [slice(NG, NG + k) for k in self.n]
        at[a.ndim - 3 + d] = slice(NG + lo, NG + self.n[d] + hi)
        return a[tuple(at)]


def _cons_prim(q):
    vel = q[1:4] / q[0]
    p = (GAMMA - 1.0) * (q[4] - 0.5 * q[0] * _dot(vel, vel))
    return torch.cat([q[:1], vel, p[None]]), p / (q[0] * R_GAS)


def _prim_cons(w):
    return torch.cat([w[:1], w[0] * w[1:4], (w[4] / (GAMMA - 1.0) + 0.5 * w[0] * _dot(w[1:4], w[1:4]))[None]])


def _inflow(case, g, time):
    """Ghost layers at i-min: profile mean and Fourier-mode fluctuations."""
    pr, tab, layers = _ramp_props(), _ramp_profile(), []
    modes = wmx.SmoothRampInflow(pr, tab, seed=0, n_modes=64, span_cells=case["nz"]).modes
    U = pr["U_inf"]
    inner = slice(NG, NG + case["nz"])
    for gi in range(NG):
        y, z = (g.xc[a, gi].cpu().numpy() / pr["L"] for a in (1, 2))
        f = []
        for c in range(3):
            kx, ky, kz, ph = (m[:, None, None] for m in modes[c])
            v = np.cos(kx * (U * time / pr["L"]) + ky * y + kz * z + ph).sum(0)
            v = v - v[:, inner].mean(1, keepdims=True)
            if c == 1:
                v = v - (v[:, inner] * f[0][:, inner]).mean(1, keepdims=True) * f[0]
            f.append(v / np.sqrt(np.maximum((v[:, inner] ** 2).mean(1, keepdims=True), 1e-20)))
        col = [np.interp(y, tab[:, 0], tab[:, k]) for k in range(7)]
        a, b, c, uv = (np.maximum(col[k], 0.0) * U * U for k in (3, 4, 5, 6))
        l10 = uv / np.maximum(np.sqrt(a), 1e-14)
        one = np.ones_like(y)
        w = [pr["rho_inf"] * one, U * col[1] + np.sqrt(a) * f[0],
             U * col[2] + l10 * f[0] + np.sqrt(np.maximum(b - l10 ** 2, 0.0)) * f[1], np.sqrt(c) * f[2],
             pr["p_inf"] * one]
        layers.append(torch.as_tensor(np.stack(w), device="cuda"))
    return _prim_cons(torch.stack(layers, 1))


def _farfield(case, q, nrm):
    pr = _ramp_props()
    w, T = _cons_prim(q)
    r0, p0, u0 = pr["rho_inf"], pr["p_inf"], torch.zeros_like(w[1:4])
    u0[0] = pr["U_inf"]
    c0 = math.sqrt(GAMMA * p0 / r0)
    un, c, dun, dp = _dot(w[1:4], nrm), torch.sqrt(GAMMA * R_GAS * T), _dot(w[1:4] - u0, nrm), w[4] - p0
    zero = torch.zeros_like(un)
    ap = torch.where(un + c > 0, dp + r0 * c0 * dun, zero)
    am = torch.where(un - c > 0, dp - r0 * c0 * dun, zero)
    out = un > 0
    rho = r0 + 0.5 * (ap + am) / c0 ** 2 + torch.where(out, w[0] - r0 - dp / c0 ** 2, zero)
    ut = torch.where(out[None], w[1:4] - u0 - dun * nrm, torch.zeros_like(u0))
    return _prim_cons(torch.cat([rho[None], u0 + (ap - am) / (2 * r0 * c0) * nrm + ut,
                                 (p0 + 0.5 * (ap + am))[None]]))


def _fill(case, g, q, time):
    for _ in range(2):
        for d in range(3):
            n = g.n[d]
            if g.periodic[d]:
                q[_sl(d, slice(0, NG), 4)] = q[_sl(d, slice(n, n + NG), 4)]
                q[_sl(d, slice(NG + n, None), 4)] = q[_sl(d, slice(NG, 2 * NG), 4)]
                continue
            for side in (0, 1):
                fb = NG if side == 0 else NG + n
                S = g.S[d][_sl(d, slice(fb, fb + 1), 4)]
                nrm = S / torch.sqrt(_dot(S, S))
                src = q[_sl(d, slice(NG, 2 * NG) if side == 0 else slice(n, NG + n), 4)].flip(1 + d)
                if d == 0 and side == 0:
                    new = _inflow(case, g, time)
                elif d == 0:
                    new = _farfield(case, src, nrm)
                else:                                    # slip: the momentum's normal part turns
                    m = src[1:4] - 2.0 * _dot(src[1:4], nrm) * nrm
                    new = torch.cat([src[:1], m, src[4:]])
                q[_sl(d, slice(0, NG) if side == 0 else slice(NG + n, None), 4)] = new
    return q


def _gradients(g, phi):
    acc = 0.0
    for d in range(3):
        N = phi.shape[1 + d]
        pf = 0.5 * (phi[_sl(d, slice(0, N - 1), 4)] + phi[_sl(d, slice(1, N), 4)])
        fl = pf[:, None] * g.S[d][_sl(d, slice(1, N), 4)][None]
        at = [slice(None)] * 2 + [slice(1, -1)] * 3
        at[2 + d] = slice(None)
        acc = acc + torch.diff(fl[tuple(at)], dim=2 + d)
    out = torch.zeros((4, 3) + tuple(phi.shape[1:]), dtype=phi.dtype, device=phi.device)
    out[..., 1:-1, 1:-1, 1:-1] = acc / g.vol[1:-1, 1:-1, 1:-1]
    return out


def _eddy(name, gu, delta):
    S = 0.5 * (gu + gu.transpose(0, 1))
    if name == "smagorinsky":
        return (0.16 * delta) ** 2 * torch.sqrt(2.0 * (S * S).sum((0, 1)))
    if name == "wale":
        g2 = torch.stack([torch.stack([_dot(gu[i], gu[:, j]) for j in range(3)]) for i in range(3)])
        Sd = 0.5 * (g2 + g2.transpose(0, 1))
        tr = (g2[0, 0] + g2[1, 1] + g2[2, 2]) / 3.0
        for i in range(3):
            Sd[i, i] -= tr
        ss, dd = (S * S).sum((0, 1)), (Sd * Sd).sum((0, 1))
        return (0.325 * delta) ** 2 * dd ** 1.5 / (ss ** 2.5 + dd ** 1.25 + 1e-30)
    if name == "vreman":
        b = delta ** 2 * torch.stack([torch.stack([_dot(gu[i], gu[j]) for j in range(3)]) for i in range(3)])
        B = (b[0, 0] * b[1, 1] - b[0, 1] ** 2 + b[0, 0] * b[2, 2] - b[0, 2] ** 2 + b[1, 1] * b[2, 2]
             - b[1, 2] ** 2)
        return 2.5 * 0.17 ** 2 * torch.sqrt(torch.clamp(B, min=0.0) / ((gu * gu).sum((0, 1)) + 1e-30))
    return torch.zeros_like(delta)


def _kep(a, b, S):
    rho, vel, p = 0.5 * (a[0] + b[0]), 0.5 * (a[1:4] + b[1:4]), 0.5 * (a[4] + b[4])
    e = 0.5 * sum(w[4] / ((GAMMA - 1.0) * w[0]) + 0.5 * _dot(w[1:4], w[1:4]) for w in (a, b))
    un = _dot(vel, S)
    return torch.cat([(rho * un)[None], rho * un * vel + p * S, (rho * un * e + p * un)[None]])


def _keep(a, b, S):
    rho, vel, p = 0.5 * (a[0] + b[0]), 0.5 * (a[1:4] + b[1:4]), 0.5 * (a[4] + b[4])
    m = rho * _dot(vel, S)
    e = 0.5 * (a[4] / a[0] + b[4] / b[0]) / (GAMMA - 1.0)
    E = m * (0.5 * _dot(a[1:4], b[1:4]) + e) + 0.5 * (_dot(b[1:4], S) * a[4] + _dot(a[1:4], S) * b[4])
    return torch.cat([m[None], m * vel + p * S, E[None]])


def _central(two, order, st, S):
    if order == 2:
        return two(st[1], st[2], S)
    return (4.0 / 3.0) * two(st[1], st[2], S) - (two(st[1], st[3], S) + two(st[0], st[2], S)) / 6.0


def _albada(a, b, eps=1e-12):
    return (a * (b * b + eps) + b * (a * a + eps)) / (a * a + b * b + 2.0 * eps)


def _upwind(st, S):
    l = st[1] + 0.5 * _albada(st[1] - st[0], st[2] - st[1])
    r = st[2] - 0.5 * _albada(st[2] - st[1], st[3] - st[2])
    bad = (l[0] <= 0) | (l[4] <= 0) | (r[0] <= 0) | (r[4] <= 0)
    l, r = torch.where(bad, st[1], l), torch.where(bad, st[2], r)
    area = torch.sqrt(_dot(S, S))
    nrm = S / area
    ul, ur = _dot(l[1:4], nrm), _dot(r[1:4], nrm)
    cl, cr = torch.sqrt(GAMMA * l[4] / l[0]), torch.sqrt(GAMMA * r[4] / r[0])
    sl, sr = torch.minimum(ul - cl, ur - cr), torch.maximum(ul + cl, ur + cr)
    ss = ((r[4] - l[4] + l[0] * ul * (sl - ul) - r[0] * ur * (sr - ur))
          / (l[0] * (sl - ul) - r[0] * (sr - ur)))

    def side(w, un, s):
        U = _prim_cons(w)
        F = U * un
        F[1:4] += w[4] * nrm
        F[4] += w[4] * un
        f = w[0] * (s - un) / (s - ss)
        e = U[4] / w[0] + (ss - un) * (ss + w[4] / (w[0] * (s - un)))
        return F, F + s * (torch.cat([f[None], f * (w[1:4] + (ss - un) * nrm), (f * e)[None]]) - U)

    (Fl, Fsl), (Fr, Fsr) = side(l, ul, sl), side(r, ur, sr)
    return area * torch.where(sl >= 0, Fl, torch.where(ss >= 0, Fsl, torch.where(sr > 0, Fsr, Fr)))


def _viscous(g, d, phi, gr, mu, k, S):
    def L(a):
        return g.slab(a, d, -1, 0)

    def Rr(a):
        return g.slab(a, d, 0, 1)
    dx = Rr(g.xc) - L(g.xc)
    dist = torch.sqrt(_dot(dx, dx))
    e = dx / dist
    gf = 0.5 * (L(gr) + Rr(gr))
    corr = (Rr(phi) - L(phi)) / dist - (gf[:, 0] * e[0] + gf[:, 1] * e[1] + gf[:, 2] * e[2])
    gf = gf + corr[:, None] * e[None]
    uf, muf, kf = 0.5 * (L(phi[:3]) + Rr(phi[:3])), 0.5 * (L(mu) + Rr(mu)), 0.5 * (L(k) + Rr(k))
    div = gf[0, 0] + gf[1, 1] + gf[2, 2]
    t = torch.stack([muf * (_dot(gf[i] + gf[:3, i], S) - (2.0 / 3.0) * div * S[i]) for i in range(3)])
    return torch.cat([torch.zeros_like(div)[None], -t, (-_dot(uf, t) - kf * _dot(gf[3], S))[None]])


def _wall_law(h, U, T_h, p_h, T_wall):
    """Spalding's u_tau and Kader's heat flux."""
    kappa, ekb = 0.41, math.exp(-0.41 * 5.2)
    U = torch.clamp(U, min=1e-8)
    T_w = T_h + PR ** (1.0 / 3.0) * U ** 2 / (2.0 * CP) if T_wall is None else T_wall + 0.0 * T_h
    rho, mu = p_h / (R_GAS * T_w), _mu(T_w)
    Re = h * U * rho / mu
    up = torch.clamp(torch.sqrt(Re), 1.0, 25.0)
    for _ in range(30):
        ku = kappa * up
        ex = torch.exp(ku)
        F = up + ekb * (ex - 1.0 - ku - 0.5 * ku ** 2 - ku ** 3 / 6.0) - Re / up
        dF = 1.0 + ekb * kappa * (ex - 1.0 - ku - 0.5 * ku ** 2) + Re / up ** 2
        up = torch.minimum(torch.maximum(up - F / dF, 0.5 * up), torch.full_like(up, 100.0))
    ut = U / up
    if T_wall is None:
        return rho * ut ** 2, torch.zeros_like(ut)
    yp = torch.clamp(h * ut * rho / mu, min=1e-6)
    G = torch.clamp(0.01 * (PR * yp) ** 4 / (1.0 + 5.0 * PR ** 3 * yp), min=1e-20)
    beta = (3.85 * PR ** (1.0 / 3.0) - 1.3) ** 2 + 2.12 * math.log(PR)
    Tp = PR * yp * torch.exp(-G) + (2.12 * torch.log(1.0 + yp) + beta) * torch.exp(-1.0 / G)
    return rho * ut ** 2, rho * CP * ut * (T_w - T_h) / Tp


def _wall(case, g, w, T, side):
    """(flux along +j, tau_w, q_w) of a wall-modelled j face."""
    n, nm = g.n[1], case.get("n_match", 1)
    fb, ci, mi = ((NG, NG, NG + nm - 1) if side == 0 else (NG + n, NG + n - 1, NG + n - nm))

    def at(a, j):
        return a[..., NG:NG + g.n[0], j, NG:NG + g.n[2]]
    S = at(g.S[1], fb)
    area = torch.sqrt(_dot(S, S))
    out = S / area if side == 1 else -S / area
    h = _dot(at(g.xc, mi) - at(g.xf[1], fb), -out)
    vel = at(w[1:4], mi)
    par = vel - _dot(vel, out) * out
    U = torch.sqrt(_dot(par, par) + 1e-20)
    tau, qw = _wall_law(h, U, at(T, mi), at(w[4], mi), 300.0 if case["kind"] == "channel" else None)
    F = torch.cat([torch.zeros_like(tau)[None], (at(w[4], ci) * out + tau * par / U) * area, (-qw * area)[None]])
    return (F if side == 1 else -F), tau, qw


def _rhs(case, g, q, time):
    w, T = _cons_prim(_fill(case, g, q.clone(), time))
    phi = torch.cat([w[1:4], T[None]])
    gr = _gradients(g, phi)
    gu = gr[:3]
    mu, mut = _mu(T), w[0] * _eddy(case.get("sgs", "vreman"), gu, g.vol ** (1.0 / 3.0))
    k = CP * (mu / PR + mut / PR_T)
    mu = mu + mut
    scheme = case.get("scheme", "hybrid")
    if scheme == "hybrid":
        div2 = (gu[0, 0] + gu[1, 1] + gu[2, 2]) ** 2
        rot = (gu[2, 1] - gu[1, 2]) ** 2 + (gu[0, 2] - gu[2, 0]) ** 2 + (gu[1, 0] - gu[0, 1]) ** 2
        theta = div2 / (div2 + rot + 1e-30)
    r = 0.0
    for d in range(3):
        S = g.slab(g.S[d], d, 0, 1)
        st = [g.slab(w, d, o, o + 1) for o in (-2, -1, 0, 1)]
        if scheme == "hybrid":
            s = torch.clamp((torch.maximum(g.slab(theta, d, -1, 0), g.slab(theta, d, 0, 1)) - 0.6) / (0.9 - 0.6),
                            0.0, 1.0)
            F = (1.0 - s) * _central(_kep, 4, st, S) + s * _upwind(st, S)
        elif scheme == "muscl":
            F = _upwind(st, S)
        else:
            F = _central(_keep if scheme == "keep4" else _kep, int(scheme[-1]), st, S)
        F = F + _viscous(g, d, phi, gr, mu, k, S)
        if d == 1 and case["kind"] != "skewed":
            F[:, :, 0] = _wall(case, g, w, T, 0)[0]
            if case["kind"] == "channel":
                F[:, :, -1] = _wall(case, g, w, T, 1)[0]
        r = r - torch.diff(F, dim=1 + d)
    r = r / g.inner(g.vol)
    if case["kind"] == "ramp":
        pr = _ramp_props()
        qi, vol = g.inner(q), g.inner(g.vol)
        mean = (qi * vol).sum(3, keepdim=True) / vol.sum(2, keepdim=True)
        eta = torch.clamp(g.inner(g.xc[0]) / pr["L"] - 3.0, 0.0, 1.0)
        r = r - pr["U_inf"] / pr["L"] * eta ** 3 * (10.0 + eta * (-15.0 + 6.0 * eta)) * (qi - mean)
    return torch.nn.functional.pad(r, [NG] * 6)


def _max_dt(g, q, cfl):
    w, T = _cons_prim(g.inner(q))
    c, vol = torch.sqrt(GAMMA * R_GAS * T), g.inner(g.vol)
    nu = max(4.0 / 3.0, GAMMA / PR) * _mu(T) / w[0]
    lam = visc = 0.0
    for d in range(3):
        S = g.slab(g.S[d], d, 0, 1)
        S = 0.5 * (S[_sl(d, slice(0, -1), 4)] + S[_sl(d, slice(1, None), 4)])
        a2 = _dot(S, S)
        lam, visc = lam + _dot(w[1:4], S).abs() + c * torch.sqrt(a2), visc + nu * a2 / vol
    return (cfl / ((lam + 4.0 * visc) / vol)).min()


def _exact_case(case, Q):
    """One channel, ramp or skewed case from its blocks' states Q."""
    nodes, (Lx, Lz) = _nodes(case)
    g = _Grid(nodes, (Lx, None, Lz))
    cuts = _cuts(case) if case["kind"] != "skewed" else [0, case["nx"] // 2, case["nx"]]
    # the domain's state: the blocks' cells side by side (the ghosts are filled before use)
    q = torch.cat([b[:, NG:NG + hi - lo] for b, lo, hi in zip(Q, cuts, cuts[1:])], 1)
    q = torch.nn.functional.pad(q, [0, 0, 0, 0, NG, NG], value=1.0)

    def split(a, ghosts):
        out = []
        for b, lo, hi in zip(ghosts, cuts, cuts[1:]):
            b = b.clone()
            b[:, NG:NG + hi - lo, NG:-NG, NG:-NG] = a[:, NG + lo:NG + hi, NG:-NG, NG:-NG]
            out.append(b)
        return tuple(out)

    if case["kind"] == "skewed":
        return split(_rhs(case, g, q, 0.0), [torch.zeros_like(b) for b in Q])
    dt = _max_dt(g, q, 0.5 if case["kind"] == "ramp" else 0.8)
    if case.get("call") == "diagnostics":
        w, T = _cons_prim(q)
        wall = {(f"B{b}", face): tuple(a[lo:hi] for a in _wall(case, g, w, T, side)[1:])
                for b, (lo, hi) in enumerate(zip(cuts, cuts[1:])) for side, face in enumerate(("jmin", "jmax"))}
        w, T = w[:, NG:NG + cuts[1], NG:-NG, NG:-NG], T[NG:NG + cuts[1], NG:-NG, NG:-NG]
        avg = {k: a.mean((0, 2)) for k, a in zip(("rho", "u", "v", "w", "p", "T"), [*w, T])}
        for a, b in ("uu", "vv", "ww", "uv", "uw", "vw"):
            wa, wb = (w["_uvw".index(c)] - avg[c][:, None] for c in (a, b))
            avg[a + b] = (wa * wb).mean((0, 2))
        tau = sum(t[0].mean() for t in wall.values()) / len(wall)
        return {"dt": dt, "wall": wall, "y": g.inner(g.xc)[1, 0, :, 0], "profiles": avg, "tau": tau}
    t0 = RAMP_TIME if case["kind"] == "ramp" else 0.0
    q1 = q + dt * _rhs(case, g, q, t0)
    q2 = 0.75 * q + 0.25 * (q1 + dt * _rhs(case, g, q1, t0 + float(dt)))
    q3 = split((q + 2.0 * (q2 + dt * _rhs(case, g, q2, t0 + 0.5 * float(dt)))) / 3.0, Q)
    if case["kind"] == "channel":
        s = _channel_scales(case["Re_b"])
        vol = g.inner(g.vol)
        mean = sum((b[1, NG:-NG, NG:-NG, NG:-NG] * vol[lo:hi]).sum() for b, lo, hi in zip(q3, cuts, cuts[1:]))
        delta = s["rho0"] * s["Ub"] - mean / vol.sum()
        for b in q3:
            b[4] += (2.0 * b[1] * delta + delta ** 2) / (2.0 * b[0])
            b[1] += delta
    return q3, dt


def exact(case, seed):
    """What `run` returns, in float64 torch; None for the largest grids (its temporaries)."""
    if _cells(case) > 12_000_000:
        return None
    st = prepare(case, seed)
    if case["kind"] == "ensemble":
        got = [_exact_case(m, Q) for m, Q in zip(_members(case), st["Q"])]
        return [q for q, _ in got], torch.stack([dt for _, dt in got])
    return _exact_case(case, st["Q"])
