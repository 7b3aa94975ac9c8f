"""Timed cases of the peridynamic force path: what its users run, through the
public entry points (peridigm_amd.Context, .quasistatic, .learned,
.discretization and the C ABI behind them).

A case is a dict of plain values; "kind" says which call it stands for:

  explicit   an output interval of an explicit run: state in, nsteps
             velocity-Verlet steps (optionally with critical-stretch damage,
             prescribed displacements and short-range contact), output fields
             out. Meshes: a bar (no damage), a notched plate (damage, pulled
             ends), a randomly perturbed tube (damage, expanding).
  force      Material::computeForce as a host code calls it: positions in,
             dilatation and force density out.
  evaluate   one model evaluation of a host code: DamageModel::computeDamage,
             then Material::computeForce with the new bond damage (both bond
             fields on the host).
  tangent    K(u) w of the quasi-static tangent, host vectors in and out.
  solve      one linear solve K(u) x = b to a relative residual of 1e-8.
  tension    a quasi-static tension run: load steps, Newton, linear solves.
  network    forward and gradient of the learned preconditioner's network.
  search     the fixed-radius neighbourhood search with plane filters that
             builds a block's bond list.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

STEEL = dict(K=130.0e9, mu=78.0e9, rho=7800.0)
MODELS = ("Elastic", "Elastic Bond Based", "Linear LPS")


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the 10,000-node bar, its whole run of 1,000 steps: the smallest
        # explicit mesh in use, where every step is two short kernels
        dict(name="bar_10k_1000_steps", kind="explicit", mesh="bar", nx=100, ny=10, nz=10,
             nsteps=1000, dt=1.0e-8, influence=0, model=0, sc=0.0, pull=0.0, contact=0),
        # an irregular mesh with growing damage (a fragmenting tube; 69k nodes
        # with every neighbour count from 30 to 128), one output interval
        dict(name="tube_300_steps", kind="explicit", mesh="tube", r_in=20, r_out=25, length=97,
             nsteps=300, dt=5.0e-8, influence=0, model=0, sc=1.5e-3, pull=0.0, contact=0),
        # the notched plate of the headline workload, one output interval
        dict(name="plate_640k_500_steps", kind="explicit", mesh="plate", nx=400, ny=400, nz=4,
             nsteps=500, dt=2.5e-8, influence=0, model=0, sc=5.0e-4, pull=2.0, contact=0),
        # the plate with short-range contact on every node, searched every 50
        # steps, its notch closing
        dict(name="plate_contact_200_steps", kind="explicit", mesh="plate", nx=200, ny=200, nz=4,
             nsteps=200, dt=2.5e-8, influence=0, model=0, sc=5.0e-4, pull=2.0, contact=50),
        # drop-in force evaluation of an elastic block
        dict(name="force_160k", kind="force", mesh="plate", nx=200, ny=200, nz=4, influence=0,
             model=0),
        # drop-in model evaluation with damage (bond fields on the host)
        dict(name="evaluate_36k", kind="evaluate", mesh="plate", nx=95, ny=95, nz=4, influence=0,
             sc=5.0e-4),
        # one tangent application on the quasi-static bar: the smallest call
        # of the quasi-static path
        dict(name="tangent_24k", kind="tangent", mesh="bar", nx=60, ny=20, nz=20, influence=0),
        # a linear solve of the quasi-static bar with the default solver
        dict(name="solve_24k_block_jacobi", kind="solve", mesh="bar", nx=60, ny=20, nz=20,
             influence=0, precond="block_jacobi"),
        # the large quasi-static bar with the two-level preconditioner
        dict(name="solve_200k_two_level", kind="solve", mesh="bar", nx=125, ny=40, nz=40,
             influence=0, precond="two_level"),
        # a whole quasi-static run on a small bar: many short linear solves
        dict(name="tension_3k_block_jacobi", kind="tension", mesh="bar", nx=30, ny=10, nz=10,
             influence=0, precond="block_jacobi", load_steps=5),
        # one training step's network work on the quasi-static bar
        dict(name="network_24k", kind="network", mesh="bar", nx=60, ny=20, nz=20, gradient=True),
        # the bond list of a notched plate with perturbed points
        dict(name="search_160k", kind="search", mesh="plate", nx=200, ny=200, nz=4, jitter=0.05),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _log_bar(rng, lo, hi, aspect=(1.0, 10.0)):
    """nx >= ny ~ nz with about N nodes, N log-uniform in [lo, hi]."""
    n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    a = rng.uniform(*aspect)
    s = (n / a) ** (1.0 / 3.0)
    ny = max(5, int(round(s * rng.uniform(0.85, 1.15))))
    nz = max(4, int(round(s)))
    return max(8, int(round(n / (ny * nz)))), ny, nz


def _log_plate(rng, lo, hi):
    """nx x ny x nz of a thin plate with about N nodes, N log-uniform."""
    n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    nz = rng.choice((3, 4, 4, 5))
    a = rng.uniform(0.6, 1.7)
    ny = max(16, int(round(math.sqrt(n / nz / a))))
    return max(16, int(round(n / nz / ny))), ny, nz


def draw(rng):
    kind = rng.choice(("explicit", "explicit", "explicit", "force", "evaluate", "tangent", "solve",
                       "solve", "tension", "network", "search"))
    infl = rng.choice((0, 0, 0, 1, 2))
    if kind == "explicit":
        mesh = rng.choice(("bar", "plate", "plate", "tube"))
        nsteps = _log_int(rng, 100, 400)
        if mesh == "bar":
            nx, ny, nz = _log_bar(rng, 1000, 100000)
            return dict(kind=kind, mesh=mesh, nx=nx, ny=ny, nz=nz, nsteps=nsteps, dt=1.0e-8,
                        influence=infl, model=rng.choice((0, 0, 1)), sc=0.0, pull=0.0, contact=0)
        if mesh == "tube":
            r = _log_int(rng, 12, 30)
            return dict(kind=kind, mesh=mesh, r_in=r, r_out=r + rng.randint(4, 8),
                        length=_log_int(rng, 20, 120), nsteps=nsteps, dt=5.0e-8, influence=infl,
                        model=0, sc=1.5e-3, pull=0.0, contact=0)
        nx, ny, nz = _log_plate(rng, 3000, 300000)
        return dict(kind=kind, mesh=mesh, nx=nx, ny=ny, nz=nz, nsteps=nsteps, dt=2.5e-8,
                    influence=infl, model=rng.choice((0, 0, 0, 1)), sc=5.0e-4, pull=2.0,
                    contact=rng.choice((0, 0, 25, 100)))
    if kind == "force":
        if rng.random() < 0.5:
            nx, ny, nz = _log_plate(rng, 2000, 300000)
            return dict(kind=kind, mesh="plate", nx=nx, ny=ny, nz=nz, influence=infl,
                        model=rng.choice((0, 0, 1, 2)))
        nx, ny, nz = _log_bar(rng, 1000, 200000)
        return dict(kind=kind, mesh="bar", nx=nx, ny=ny, nz=nz, influence=infl,
                    model=rng.choice((0, 0, 1, 2)))
    if kind == "evaluate":
        nx, ny, nz = _log_plate(rng, 2000, 100000)
        return dict(kind=kind, mesh="plate", nx=nx, ny=ny, nz=nz, influence=infl, sc=5.0e-4)
    if kind == "tangent":
        nx, ny, nz = _log_bar(rng, 1000, 200000)
        return dict(kind=kind, mesh="bar", nx=nx, ny=ny, nz=nz, influence=infl)
    if kind == "solve":
        nx, ny, nz = _log_bar(rng, 1000, 150000, aspect=(2.0, 5.0))
        return dict(kind=kind, mesh="bar", nx=nx, ny=ny, nz=nz, influence=infl,
                    precond=rng.choice(("block_jacobi", "two_level", "none")))
    if kind == "tension":
        nx, ny, nz = _log_bar(rng, 1000, 24000, aspect=(2.0, 4.0))
        return dict(kind=kind, mesh="bar", nx=max(12, nx), ny=ny, nz=nz, influence=0,
                    precond=rng.choice(("block_jacobi", "two_level")),
                    load_steps=rng.randint(2, 5))
    if kind == "network":
        nx, ny, nz = _log_bar(rng, 1000, 100000)
        return dict(kind=kind, mesh="bar", nx=nx, ny=ny, nz=nz,
                    gradient=rng.choice((True, True, False)))
    nx, ny, nz = _log_plate(rng, 3000, 200000)
    return dict(kind="search", mesh="plate", nx=nx, ny=ny, nz=nz,
                jitter=rng.choice((0.0, 0.05, 0.2)))


# ---------------------------------------------------------------------------
# meshes and inputs (numpy only, from the seed)
# ---------------------------------------------------------------------------
def _spacing(case):
    return 5.0e-4 if case["mesh"] == "plate" else 1.0e-3


def _points(case, rng):
    """Points and volumes: a lattice, or a tube cut from one and perturbed."""
    h = _spacing(case)
    if case["mesh"] == "tube":
        m = case["r_out"] + 1
        i, j, k = np.meshgrid(np.arange(-m, m), np.arange(-m, m), np.arange(case["length"]),
                              indexing="ij")
        x = (np.stack([i.ravel(), j.ravel(), k.ravel()], axis=1) + 0.5) * h
        r = np.hypot(x[:, 0], x[:, 1])
        x = x[(r >= case["r_in"] * h) & (r <= case["r_out"] * h)]
        x = x + rng.uniform(-0.05 * h, 0.05 * h, size=x.shape)
    else:
        k, j, i = np.meshgrid(np.arange(case["nz"]), np.arange(case["ny"]), np.arange(case["nx"]),
                              indexing="ij")
        x = (np.stack([i.ravel(), j.ravel(), k.ravel()], axis=1) + 0.5) * h
        if case["kind"] == "search":  # one point cloud, numbered from a point of the seed's choice
            d = np.random.default_rng(7).uniform(-1.0, 1.0, size=x.shape) * (case["jitter"] * h)
            x = np.roll(x + d, int(rng.integers(1, len(x))), axis=0)
    return np.ascontiguousarray(x), np.full(len(x), h ** 3)


def _notch(case):
    """The plate's edge notch on its mid plane y = y0, from x = 0 to `tip`:
    FinitePlane parameters (normal, corner, bottom direction, two lengths)."""
    h = _spacing(case)
    y0, cells = 0.5 * case["ny"] * h + 0.01 * h, max(2, case["nx"] // 10)
    return np.array([[0.0, 1.0, 0.0, -h, y0, -h, 1.0, 0.0, 0.0, (cells + 1.03) * h,
                      (case["nz"] + 2) * h]])


def _waves(x, rng, strain):
    """A smooth random displacement with strains of about `strain`."""
    span = (x.max(axis=0) - x.min(axis=0)).max()
    u = np.zeros_like(x)
    for _ in range(3):
        k = 2.0 * np.pi * rng.integers(1, 4, size=3) / span
        d = rng.normal(size=3)
        u += np.sin(x @ k + rng.uniform(0.0, 6.28))[:, None] * d / (np.linalg.norm(d)
                                                                    * np.linalg.norm(k))
    return u * (strain / math.sqrt(3.0))


def _inputs(case, seed):
    rng = np.random.default_rng(seed)
    x, vol = _points(case, rng)
    h = _spacing(case)
    p = dict(x=x, vol=vol, h=h, horizon=3.015 * h,
             planes=_notch(case) if case["mesh"] == "plate" else None, bcs=[])
    kind = case["kind"]
    if kind == "explicit":
        if case["mesh"] == "bar":  # a velocity step at one end, and a gentle random field
            p["u0"] = _waves(x, rng, 2.0e-5)
            p["v0"] = np.zeros_like(x)
            p["v0"][x[:, 0] < 5 * h, 0] = 1.0 + 0.2 * rng.random()
        elif case["mesh"] == "tube":
            r = np.hypot(x[:, 0], x[:, 1])
            speed = 200.0 * (1.0 + rng.uniform(-0.01, 0.01, size=len(x)))
            p["u0"] = np.zeros_like(x)
            p["v0"] = np.stack([speed * x[:, 0] / r, speed * x[:, 1] / r, 0.0 * r], axis=1)
        else:
            p["u0"] = _waves(x, rng, 2.0e-4)
            p["v0"] = np.zeros_like(x)
            if case["contact"]:  # the halves close on the notch
                p["v0"][:, 1] = np.where(x[:, 1] > p["planes"][0][4], -10.0, 10.0)
            j = np.rint(x[:, 1] / h - 0.5).astype(int)
            p["bcs"] = [(np.nonzero(j >= case["ny"] - 3)[0], 1, 0.0, case["pull"]),
                        (np.nonzero(j <= 2)[0], 1, 0.0, -case["pull"])]
    elif kind == "force":
        p["y"] = x + _waves(x, rng, 1.0e-3)
    elif kind == "evaluate":  # the earlier state broke some bonds, the present one breaks more
        p["y_prev"] = x + _waves(x, rng, 5.0e-4)
        p["y"] = x + _waves(x, rng, 6.0e-4)
    elif kind in ("tangent", "solve", "tension"):
        i = np.rint(x[:, 0] / h - 0.5).astype(int)
        p["left"], p["right"] = np.nonzero(i <= 2)[0], np.nonzero(i >= case["nx"] - 3)[0]
        ends = np.concatenate([p["left"], p["right"]])
        p["fixed"] = (3 * ends[:, None] + np.arange(3)[None, :]).ravel()
        p["u"] = _waves(x, rng, 5.0e-4)
        if kind == "tangent":
            p["w"] = rng.normal(size=x.shape) * 1.0e-6
        if kind == "solve":  # a smooth body load with some noise, in force units
            b = _waves(x, rng, 1.0) / h + 0.05 * rng.normal(size=x.shape)
            b.reshape(-1)[p["fixed"]] = 0.0
            p["b"] = b
        if kind == "tension":
            p["strain"] = 1.0e-3 * (1.0 + 0.2 * rng.uniform(-1.0, 1.0))
    elif kind == "network":
        p["features"] = rng.normal(size=(len(x), 8)).astype(np.float32)
        p["gout"] = rng.normal(size=(len(x), 3)).astype(np.float32) if case["gradient"] else None
        par = []
        for di, do in ((8, 32), (32, 32), (32, 3)):
            par.append(rng.normal(0.0, math.sqrt(2.0 / (2 * di + do)), size=2 * di * do))
            par.append(rng.normal(0.0, 0.1, size=do))
        p["params"] = np.concatenate(par).astype(np.float32)
    return p


# ---------------------------------------------------------------------------
# the timed work
# ---------------------------------------------------------------------------
def prepare(case, seed):
    from peridigm_amd import Context, learned, quasistatic
    from peridigm_amd.discretization import radius_search

    p = _inputs(case, seed)
    state = dict(case=case, p=p)
    if case["kind"] == "search":
        return state
    nl = radius_search(p["x"], p["horizon"], p["planes"])
    ctx = Context(0)
    ctx.set_topology(nl, len(p["x"]))
    ctx.set_material_model(MODELS[case.get("model", 0)])
    ctx.set_constants(p["x"], p["vol"], STEEL["K"], STEEL["mu"], p["horizon"],
                      case.get("influence", 0), case.get("sc", 0.0))
    state["ctx"] = ctx
    kind = case["kind"]
    if kind == "explicit":
        ctx.set_density(STEEL["rho"])
        ctx.set_bcs(p["bcs"])
        if case["contact"]:
            ctx.set_contact(p["horizon"], case["contact"], 0.9 * p["h"], 15.0 * STEEL["K"])
    elif kind == "evaluate":
        state["damage"] = ctx.compute_damage(p["y_prev"])[0]
    elif kind in ("tangent", "solve"):
        quasistatic.set_fixed(ctx, p["fixed"])
    elif kind == "tension":
        state["problem"] = dict(left=p["left"], right=p["right"], strain=p["strain"],
                                load_steps=case["load_steps"],
                                length=[case["nx"] * p["h"], case["ny"] * p["h"],
                                        case["nz"] * p["h"]])
    elif kind == "network":
        learned.init(ctx, 1)
        learned.set_params(ctx, p["params"])
    return state


def _output_fields(ctx, damage):
    """The node fields of an output frame (the bond field stays on the
    device, as in a run that writes node output)."""
    n = ctx.N
    out = dict(u=np.zeros((n, 3)), v=np.zeros((n, 3)), force=np.zeros((n, 3)), theta=np.zeros(n))
    if damage:
        out["damage"] = np.zeros(n)
    at = {k: a.ctypes.data_as(C.c_void_p) for k, a in out.items()}
    ctx.check(ctx.lib.pdg_state_download(ctx.h, at["u"], at["v"], None, None, at.get("damage"),
                                         at["theta"], at["force"]))
    return out


def run(state):
    from peridigm_amd import learned, quasistatic
    from peridigm_amd.discretization import radius_search

    case, p = state["case"], state["p"]
    kind = case["kind"]
    if kind == "search":
        return radius_search(p["x"], p["horizon"], p["planes"])
    ctx = state["ctx"]
    if kind == "explicit":
        ctx.upload_state(u=p["u0"], v=p["v0"])
        ctx.verlet_run(case["nsteps"], case["dt"])
        out = _output_fields(ctx, case["sc"] > 0.0)
        if case["contact"]:
            out["contact_force"] = ctx.contact_force_density()
        return out
    if kind == "force":
        theta, f = ctx.compute_force(p["y"])
        return dict(theta=theta, force=f)
    if kind == "evaluate":
        bd, damage, near = ctx.compute_damage(p["y"], state["damage"])
        theta, f = ctx.compute_force(p["y"], bd)
        return dict(bond_damage=bd, damage=damage, near=near, theta=theta, force=f)
    if kind == "tangent":
        return quasistatic.tangent_apply(ctx, p["u"], p["w"])
    if kind == "solve":
        return quasistatic.solve(ctx, p["u"], p["b"], precond=case["precond"])[0]
    if kind == "tension":
        u, stats, _ = quasistatic.run_tension(ctx, state["problem"], precond=case["precond"])
        return dict(u=u, newton=[s["newton"] for s in stats])
    out, grad = learned.forward_backward(ctx, p["features"], p["gout"])
    return dict(out=out, grad=grad) if grad is not None else dict(out=out)


# ---------------------------------------------------------------------------
# work of one pass
# ---------------------------------------------------------------------------
def _counts(case):
    """Nodes and directed bonds, from the mesh sizes (122 neighbours inside,
    fewer at the surfaces)."""
    r2 = 3.015 ** 2
    off = [(i, j, k) for i in range(-3, 4) for j in range(-3, 4) for k in range(-3, 4)
           if 0 < i * i + j * j + k * k <= r2]
    if case["mesh"] == "tube":
        area = math.pi * (case["r_out"] ** 2 - case["r_in"] ** 2)
        n = int(area * case["length"])
        t = case["r_out"] - case["r_in"]
        share = [max(0.0, 1 - abs(i) / t) * max(0.0, 1 - abs(k) / case["length"])
                 for i, _, k in off]
        return n, int(n * sum(share))
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    b = sum(max(0, nx - abs(i)) * max(0, ny - abs(j)) * max(0, nz - abs(k)) for i, j, k in off)
    return nx * ny * nz, b


def work(case):
    """Per bond and pass a 4-byte neighbour index; per node the FP64 state.
    Floating-point operations: about 40 (dilatation) and 45 (force) a bond."""
    n, b = _counts(case)
    kind = case["kind"]
    if kind == "explicit":  # per step: bonds from both passes, u and v read and written
        s = case["nsteps"]
        return dict(bytes=s * (4.0 * b + b / 8.0 + 96.0 * n) + 200.0 * n, flops=85.0 * b * s)
    if kind == "force":
        return dict(bytes=4.0 * b + 56.0 * n, flops=85.0 * b)
    if kind == "evaluate":  # bond damage in, out and in again
        return dict(bytes=4.0 * b + 24.0 * b + 88.0 * n, flops=125.0 * b)
    if kind == "tangent":
        return dict(bytes=4.0 * b + 72.0 * n, flops=110.0 * b)
    if kind in ("solve", "tension"):  # iterations grow with the bar's length in horizons
        two = case["precond"] == "two_level"
        its = (25.0 if two else 8.0 + 1.2 * case["nx"]) * (1.5 if case["precond"] == "none" else 1)
        its *= 2.0 * case["load_steps"] if kind == "tension" else 1.0
        return dict(bytes=its * (4.0 * b + 240.0 * n), flops=its * (110.0 * b + 100.0 * n))
    if kind == "network":
        k = 3.0 if case["gradient"] else 1.0
        return dict(bytes=k * (4.0 * b + 300.0 * n), flops=k * (80.0 * b + 2.0 * 2800.0 * n))
    return dict(bytes=4.0 * b + 28.0 * n, flops=8.0 * 3.5 * b)


# ---------------------------------------------------------------------------
# the same results in 64 bits, with plain torch
# ---------------------------------------------------------------------------
class _Bonds:
    """All directed bonds (i, j) within the horizon, i ascending, j ascending
    in a row, without those the notch plane cuts; per-bond reference data."""

    def __init__(self, case, p, dev):
        self.dev = dev
        self.x = torch.tensor(p["x"], dtype=torch.float64, device=dev)
        self.vol = torch.tensor(p["vol"], dtype=torch.float64, device=dev)
        self.n = len(p["x"])
        self.i, self.j = _pairs(self.x, p["horizon"])
        if p["planes"] is not None:
            y0, length = p["planes"][0][4], p["planes"][0][3] + p["planes"][0][9]
            a, b = self.x[self.i], self.x[self.j]
            t = (y0 - a[:, 1]) / (b[:, 1] - a[:, 1])
            keep = ~((t >= 0) & (t <= 1) & (a[:, 0] + t * (b[:, 0] - a[:, 0]) <= length))
            self.i, self.j = self.i[keep], self.j[keep]
        self.xi = self.x[self.j] - self.x[self.i]
        self.zeta = self.xi.norm(dim=1)
        z = self.zeta / p["horizon"]
        infl = case.get("influence", 0)
        self.om = (torch.ones_like(z) if infl == 0 else
                   torch.where(z < 0.5, torch.ones_like(z), 4 * z - 4 * z * z) if infl == 1 else
                   torch.exp(-(z / 0.4) ** 2))
        self.vj = self.vol[self.j]
        self.m = self.sum(self.om * self.zeta ** 2 * self.vj)
        K, mu = STEEL["K"], STEEL["mu"]
        self.alpha = 15.0 * mu / self.m
        self.beta = 3.0 * K / self.m - self.alpha / 3.0
        self.model = case.get("model", 0)
        self.c = 18.0 * K / (math.pi * p["horizon"] ** 4)

    def sum(self, v):
        shape = (self.n,) + tuple(v.shape[1:])
        return torch.zeros(shape, dtype=v.dtype, device=self.dev).index_add_(0, self.i, v)

    def stretch(self, u):
        Y = self.xi + (u[self.j] - u[self.i])
        yl = Y.norm(dim=1)
        return Y, yl, yl - self.zeta

    def force(self, u, keep=None):
        """Dilatation and force density at displacement u."""
        Y, yl, e = self.stretch(u)
        k = self.om if keep is None else self.om * keep
        if self.model == 1:
            t = self.c * (e / self.zeta) * self.vj
            if keep is not None:
                t = t * keep
            return torch.zeros_like(self.m), self.sum((t / yl)[:, None] * Y)
        if self.model == 2:  # linear in u, the force along the reference bond
            pr = (self.xi * (u[self.j] - u[self.i])).sum(dim=1)
            th = 3.0 / self.m * self.sum(k * pr * self.vj)
            q = th * self.beta
            s = k * (q[self.i] + q[self.j]) + k * (self.alpha[self.i] + self.alpha[self.j]) \
                * pr / self.zeta ** 2
            return th, self.sum((s * self.vj)[:, None] * self.xi)
        th = 3.0 / self.m * self.sum(k * self.zeta * e * self.vj)
        q = th * self.beta
        t = k * ((q[self.i] + q[self.j]) * self.zeta
                 + (self.alpha[self.i] + self.alpha[self.j]) * e) * self.vj
        return th, self.sum((t / yl)[:, None] * Y)

    def tangent(self, u, fixed):
        """w -> K(u) w = -V (df/du) w on free DOFs, w on the others."""
        Y, yl, e = self.stretch(u)
        nrm = Y / yl[:, None]
        th, _ = self.force(u)
        q = th * self.beta
        a = self.om * (self.alpha[self.i] + self.alpha[self.j])
        T = self.om * (q[self.i] + q[self.j]) * self.zeta + a * e
        cz = self.om * self.zeta * self.vj
        oz = self.om * self.zeta

        def apply(w):
            d = w[self.j] - w[self.i]
            de = (nrm * d).sum(dim=1)
            dq = 3.0 / self.m * self.sum(cz * de) * self.beta
            dT = (dq[self.i] + dq[self.j]) * oz + a * de - T / yl * de
            f = (dT * self.vj)[:, None] * nrm + (T / yl * self.vj)[:, None] * d
            return torch.where(fixed, w, -self.sum(f) * self.vol[:, None])
        diag = self.sum((self.vj * a)[:, None] * nrm ** 2) * self.vol[:, None]
        return apply, torch.where(fixed, torch.ones_like(diag), diag)


def _pairs(x, r):
    """All ordered pairs of points within r of each other, sorted."""
    n, dev = len(x), x.device
    cell = torch.floor((x - x.min(dim=0).values) / (r * 1.0001)).long() + 1
    dims = cell.max(dim=0).values + 2
    key = (cell[:, 2] * dims[1] + cell[:, 1]) * dims[0] + cell[:, 0]
    skey, order = torch.sort(key)
    probe = torch.arange(int(dims.prod()) + 1, device=dev)
    start = torch.searchsorted(skey, probe)
    most = int((start[1:] - start[:-1]).max())
    steps = torch.tensor([(c * int(dims[1]) + b) * int(dims[0]) + a for c in (-1, 0, 1)
                          for b in (-1, 0, 1) for a in (-1, 0, 1)], device=dev)
    found = []
    rows = max(1, int(2.0e8 / (27 * most)))
    for lo in range(0, n, rows):
        me = torch.arange(lo, min(n, lo + rows), device=dev)
        near = key[me][:, None] + steps[None, :]
        at = start[near][:, :, None] + torch.arange(most, device=dev)
        ok = at < start[near + 1][:, :, None]
        j = order[at.clamp(max=n - 1)]
        d = x[j] - x[me][:, None, None, :]
        ok &= ((d * d).sum(dim=-1) <= r * r) & (j != me[:, None, None])
        i = me[:, None, None].expand_as(j)[ok]
        found.append(i * n + j[ok])
    found = torch.sort(torch.cat(found)).values
    return found // n, found % n


def _cg(apply, diag, b, tol=1.0e-13, most=5000):
    x = torch.zeros_like(b)
    r = b.clone()
    z = r / diag
    p, rz, stop = z.clone(), (r * z).sum(), tol * b.norm()
    for k in range(most):
        q = apply(p)
        al = rz / (p * q).sum()
        x += al * p
        r -= al * q
        if k % 10 == 9 and r.norm() <= stop:
            break
        z = r / diag
        rz, old = (r * z).sum(), rz
        p = z + rz / old * p
    return x


def _exact_explicit(case, p, dev):
    B = _Bonds(case, p, dev)
    T = lambda a: torch.tensor(a, dtype=torch.float64, device=dev)  # noqa: E731
    dt, rho, steps = case["dt"], STEEL["rho"], case["nsteps"]
    u, v = T(p["u0"]), T(p["v0"])
    keep = torch.ones_like(B.zeta) if case["sc"] > 0.0 else None
    bcs = [(torch.tensor(ids, device=dev), c, c0, c1) for ids, c, c0, c1 in p["bcs"]]
    hz, rc = p["horizon"], 0.9 * p["h"]
    cc = 9.0 * 15.0 * STEEL["K"] / (math.pi * hz ** 4)
    bond_key = B.i * B.n + B.j

    def search(y):
        i, j = _pairs(y, hz)
        key = i * B.n + j
        at = torch.searchsorted(bond_key, key).clamp(max=len(bond_key) - 1)
        free = bond_key[at] != key
        return i[free], j[free]

    def contact(pairs, y):
        i, j = pairs
        d = y[j] - y[i]
        r = d.norm(dim=1)
        f = torch.where(r < rc, -2.0 * cc * (rc - r) / hz * B.vol[j] / r, torch.zeros_like(r))
        return torch.zeros_like(y).index_add_(0, i, f[:, None] * d)

    pairs = search(B.x + u) if case["contact"] else None
    fc = torch.zeros_like(u)
    for k in range(steps + 1):
        if k > 0:
            if case["contact"] and k % case["contact"] == 0:
                pairs = search(B.x + u)
            v = v + 0.5 * dt * acc  # noqa: F821
            for ids, c, c0, c1 in bcs:
                v[ids, c] = ((c1 * (k * dt) + c0) - (c1 * ((k - 1) * dt) + c0)) / (k * dt
                                                                                 - (k - 1) * dt)
            u = u + dt * v
        if keep is not None:
            _, _, e = B.stretch(u)
            keep = torch.where(e > case["sc"] * B.zeta, torch.zeros_like(keep), keep)
        th, f = B.force(u, keep)
        if case["contact"]:
            fc = contact(pairs, B.x + u)
            f = f + fc
        acc = f / rho
        if k > 0:
            v = v + 0.5 * dt * acc
    out = dict(u=u, v=v, force=f, theta=th)
    if keep is not None:
        out["damage"] = B.sum(1.0 - keep) / B.sum(torch.ones_like(keep)).clamp(min=1.0)
    if case["contact"]:
        out["contact_force"] = fc
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "search":
        return None
    n, b = _counts(case)
    if kind == "explicit" and b * case["nsteps"] > 8.0e9:
        return None  # over about 20 seconds
    p = _inputs(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    T = lambda a: torch.tensor(a, dtype=torch.float64, device=dev)  # noqa: E731
    if kind == "explicit":
        return _exact_explicit(case, p, dev)
    B = _Bonds(case, p, dev)
    if kind == "force":
        th, f = B.force(T(p["y"]) - B.x)
        return dict(theta=th, force=f)
    if kind == "evaluate":
        old = B.stretch(T(p["y_prev"]) - B.x)[2] > case["sc"] * B.zeta
        new = B.stretch(T(p["y"]) - B.x)[2] > case["sc"] * B.zeta
        broken = (old | new).double()
        th, f = B.force(T(p["y"]) - B.x, 1.0 - broken)
        deg = B.sum(torch.ones_like(broken)).clamp(min=1.0)
        return dict(bond_damage=broken, damage=B.sum(broken) / deg, near=None, theta=th, force=f)
    if kind == "network":
        return _exact_network(case, p, B, T)
    fixed = torch.zeros(3 * n, dtype=torch.bool, device=dev)
    fixed[torch.tensor(p["fixed"], device=dev)] = True
    fixed = fixed.reshape(n, 3)
    if kind == "tangent":
        return B.tangent(T(p["u"]), fixed)[0](T(p["w"]))
    if kind == "solve":
        apply, diag = B.tangent(T(p["u"]), fixed)
        return _cg(apply, diag, T(p["b"]))
    u = torch.zeros((n, 3), dtype=torch.float64, device=dev)
    length = case["nx"] * p["h"]
    for s in range(1, case["load_steps"] + 1):
        for ids, sign in ((p["left"], -0.5), (p["right"], 0.5)):
            ids = torch.tensor(ids, device=dev)
            u[ids] = 0.0
            u[ids, 0] = sign * p["strain"] * length * s / case["load_steps"]
        for _ in range(2 if s < case["load_steps"] else 4):
            r = torch.where(fixed, torch.zeros_like(u), B.force(u)[1] * B.vol[:, None])
            apply, diag = B.tangent(u, fixed)
            u = u + _cg(apply, diag, r, tol=1.0e-10)
    return dict(u=u, newton=None)


def _exact_network(case, p, B, T):
    """The network in FP64 (the timed one multiplies in BF16)."""
    par = T(p["params"]).requires_grad_(True)
    deg = B.sum(torch.ones_like(B.zeta))

    def layer(h, at, di, do):
        mean = torch.zeros_like(h).index_add_(0, B.i, h[B.j]) / deg.clamp(min=1.0)[:, None]
        ws, wn = par[at:at + di * do], par[at + di * do:at + 2 * di * do]
        return h @ ws.reshape(di, do) + mean @ wn.reshape(di, do) \
            + par[at + 2 * di * do:at + 2 * di * do + do]
    h = torch.tanh(layer(T(p["features"]), 0, 8, 32))
    h = torch.tanh(layer(h, 544, 32, 32))
    out = layer(h, 544 + 2080, 32, 3)
    if p["gout"] is None:
        return dict(out=out.detach())
    (out * T(p["gout"])).sum().backward()
    return dict(out=out.detach(), grad=par.grad)
