"""The work a user of flouhip has it do, as cases that can be timed and checked.

Every case is a dict of plain values.  Its "kind" says which public entry points one pass calls:

    march     timeintegrate from a copy of the initial state, a few fixed steps (a whole call:
              time loop, stages and the final domain check)
    cfl       timeintegrate with dt recomputed from the CFL condition before every step
              (get_max_dt inside), optionally with the Zhang & Shu stage limiter
    stages    one Runge-Kutta step stage by stage (rk_stage), as a host's own time loop does
    gradient  adjoint.gradient: a checkpointed forward run and its reverse sweep
    vjp       rhs_ and rhs_vjp of it: what an outer optimiser calls per rhs evaluation
    monitors  get_max_dt, integrate of every variable and both monitors on one state

Meshes are periodic boxes unless the case says otherwise.  `exact` restates the scheme in plain
torch FP64 (flux differencing on GLL nodes, the reference's operators by their formulas).
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flou.jl_amd"))

import flouhip as F  # noqa: E402
from flouhip import adjoint as A  # noqa: E402

GAMMA = 1.4
DEV = "cuda"


# ------------------------------------------------------------------------------ the cases
def listed():
    return [
        # The smallest run: the linear advection test problem (2-D, 16x16, N=4), a few steps per
        # call.  Launch and call latency are all of it.
        dict(name="advection_2d_small", kind="march", eq="advection", op="strong", nx=16, ny=16, n=5,
             precision="fp64", scheme="ssprk33", steps=10),
        # The Sod tube of the reference's test suite (1-D, 20 elements, N=3): entropy-conserving
        # split form, matrix dissipation, Dirichlet ends.
        dict(name="sod_1d", kind="march", eq="euler", op="split", tp="ch", surf="matrix", setup="sod", nx=20,
             n=4, precision="fp64", scheme="ork256", steps=10),
        # Shock capturing: the reference's Shockwave2D set-up on a finer mesh of odd size, the
        # hybrid subcell operator with the positivity limiter after every stage and CFL control.
        dict(name="shock_2d_hybrid", kind="cfl", eq="euler", op="hybrid", tp="ch", surf="matrix", setup="shock",
             nx=87, ny=25, n=6, precision="fp64", scheme="ork256", steps=4, limiter=True),
        # An ordinary production run in the reference's own precision: 2-D, ragged mesh, N=4,
        # dt from the CFL condition at every step (get_cfl_callback).
        dict(name="euler_2d_cfl", kind="cfl", eq="euler", op="split", tp="kg", surf="lxf", setup="smooth",
             nx=61, ny=43, n=5, precision="fp64", scheme="ck2n54", steps=4, limiter=False),
        # The FP32 2-D benchmark: Kennedy-Gruber, 256^2, N=7.
        dict(name="kg_2d_fp32", kind="stages", eq="euler", op="split", tp="kg", surf="lxf", setup="smooth",
             nx=256, ny=256, n=8, precision="fp32", scheme="ssprk33"),
        # The headline benchmark: 3-D Taylor-Green with noise, 64^3, N=5, one CK2N54 step, FP32.
        dict(name="tgv_3d_fp32", kind="stages", eq="euler", op="split", tp="ch", surf="lxf", setup="smooth",
             nx=64, ny=64, nz=64, n=6, precision="fp32", scheme="ck2n54"),
        # The same physics in FP64, the reference's own precision, on a ragged box.
        dict(name="tgv_3d_fp64", kind="stages", eq="euler", op="split", tp="ch", surf="lxf", setup="smooth",
             nx=37, ny=32, nz=41, n=6, precision="fp64", scheme="ck2n54"),
        # The curved 3-D benchmark: 32^3 warped hexahedra, N=6, one SSPRK33 step, FP32.
        dict(name="curved_3d_fp32", kind="stages", eq="euler", op="split", tp="ch", surf="lxf", setup="smooth",
             curved=True, nx=32, ny=32, nz=32, n=7, precision="fp32", scheme="ssprk33"),
        # A channel with inflow, outflow and slip walls in the strong form, FP32, odd sizes.
        dict(name="channel_3d_strong", kind="stages", eq="euler", op="strong", surf="lxf", setup="channel",
             nx=27, ny=19, nz=14, n=5, precision="fp32", scheme="ssprk33"),
        # The adjoint benchmark: 128^2, N=5, FP64, gradient over a few checkpointed steps.
        dict(name="gradient_2d_fp64", kind="gradient", eq="euler", op="split", tp="ch", surf="lxf", setup="smooth",
             nx=128, ny=128, n=6, precision="fp64", scheme="ssprk33", steps=4, every=2),
        # rhs and its vector-Jacobian product on the curved 3-D mesh, FP32.
        dict(name="vjp_curved_3d_fp32", kind="vjp", eq="euler", op="split", tp="ch", surf="lxf", setup="smooth",
             curved=True, nx=20, ny=20, nz=20, n=7, precision="fp32", scheme="ssprk33"),
        # What a run logs between steps: the CFL step, conserved integrals, energy and entropy.
        dict(name="monitors_3d", kind="monitors", eq="euler", op="split", tp="ch", surf="lxf", setup="smooth",
             nx=48, ny=48, nz=48, n=6, precision="fp64", scheme="ck2n54"),
    ]


# Range of the node count each kind of work is done at (total nodes, low and high), and the
# polynomial degrees; a draw takes one of the listed set-ups to another place of its range.
_RANGE = {
    "advection_2d_small": (400, 60000), "sod_1d": (32, 20000), "shock_2d_hybrid": (1200, 400000),
    "euler_2d_cfl": (1200, 800000), "kg_2d_fp32": (4000, 8000000), "tgv_3d_fp32": (8000, 50000000),
    "tgv_3d_fp64": (8000, 10000000), "curved_3d_fp32": (8000, 6000000), "channel_3d_strong": (4000, 4000000),
    "gradient_2d_fp64": (2000, 800000), "vjp_curved_3d_fp32": (8000, 2000000), "monitors_3d": (2000, 20000000),
}


_AXES = ("nx", "ny", "nz")


def _full(case):
    """The case with its elements per direction as a tuple "nel"."""
    return dict(case, nel=tuple(int(case[a]) for a in _AXES if a in case))


def draw(rng):
    base = rng.choice(listed())
    c = {k: v for k, v in base.items() if k != "name"}
    nd = sum(a in c for a in _AXES)
    c["n"] = rng.choice([4, 5, 6, 7, 8] if c["eq"] == "euler" else [3, 4, 5, 6, 7, 8])
    lo, hi = _RANGE[base["name"]]
    nodes = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    side = max(2.0, (nodes ** (1.0 / nd)) / c["n"])
    nel = [max(2, int(round(side * rng.uniform(0.75, 1.3)))) for _ in range(nd)]
    while nel[-1] > 2 and math.prod(nel) * c["n"] ** nd > hi:
        nel[-1] -= 1
    c.update(zip(_AXES, nel))
    if c["kind"] in ("stages", "vjp", "gradient", "monitors") and nd > 1:
        if c["op"] == "split" and not c.get("curved"):
            c["tp"] = rng.choice(["ch", "ch", "kg", "std"])
        if math.prod(nel) * c["n"] ** nd < 8000000:
            c["precision"] = rng.choice(["fp32", "fp64"])
    if c["kind"] in ("stages", "gradient", "cfl"):
        c["scheme"] = rng.choice(["ssprk33", "ck2n54", "ork256"])
    return c


# ------------------------------------------------------------------- plain FP64 operators
@functools.lru_cache(maxsize=None)
def _gll(n):
    """GLL nodes, weights and the derivative matrix on [-1, 1]."""
    c = np.zeros(n)
    c[-1] = 1.0
    P = np.polynomial.legendre.Legendre(c)
    x = np.concatenate([[-1.0], np.sort(P.deriv().roots().real), [1.0]])
    dP, ddP = P.deriv(), P.deriv(2)
    for _ in range(3):
        x[1:-1] -= dP(x[1:-1]) / ddP(x[1:-1])
    x = 0.5 * (x - x[::-1])
    w = 2.0 / (n * (n - 1) * P(x) ** 2)
    bw = np.array([1.0 / np.prod([x[i] - x[j] for j in range(n) if j != i]) for i in range(n)])
    D = np.array([[0.0 if i == j else bw[j] / bw[i] / (x[i] - x[j]) for j in range(n)] for i in range(n)])
    D[np.arange(n), np.arange(n)] = -D.sum(axis=1)
    return x, w, D


def _box(case):
    nd = len(case["nel"])
    s = case.get("setup")
    if s == "shock":
        return (-1.0, 0.0), (2.0, 1.0)
    if s == "sod":
        return (0.0,), (1.0,)
    if case.get("curved"):
        return (0.0,) * nd, (1.0,) * nd
    if s == "channel":
        return (0.0,) * nd, (2.0, 1.0, 1.0)[:nd]
    return (0.0,) * nd, (2.0 * math.pi,) * nd


def _coords(case):
    """Reference (unmapped) node coordinates, nd tensors of shape (*nel reversed, *n reversed)."""
    nd, n, nel = len(case["nel"]), case["n"], case["nel"]
    start, length = _box(case)
    xi = torch.tensor(_gll(n)[0], dtype=torch.float64, device=DEV)
    full = tuple(reversed(nel)) + (n,) * nd
    out = []
    for d in range(nd):
        e = torch.arange(nel[d], dtype=torch.float64, device=DEV)
        x = start[d] + (e[:, None] + (xi[None, :] + 1) / 2) * (length[d] / nel[d])
        shape = [1] * (2 * nd)
        shape[nd - 1 - d], shape[2 * nd - 1 - d] = nel[d], n
        out.append(x.reshape(shape).expand(full))
    return out


def _warp(x):
    s = 0.05
    for c in x:
        s = s * torch.sin(2 * math.pi * c)
    return [c + s for c in x]


def _cons(prim):
    rho, p = prim[0], prim[-1]
    u = prim[1:-1]
    kin = sum(c * c for c in u)
    return torch.stack([rho] + [rho * c for c in u] + [p / (GAMMA - 1) + rho * kin / 2])


def _shock_states():
    u0 = 2.0 * math.sqrt(GAMMA)
    m2, g = 4.0, GAMMA
    rho1 = m2 * (g + 1) / ((g - 1) * m2 + 2)
    p1 = (2 * g * m2 - (g - 1)) / (g + 1)
    return (1.0, u0, 0.0, 1.0), (rho1, u0 / rho1, 0.0, p1)


def _prim(v):
    """Primitive state as a conservative tuple."""
    return _cons(torch.tensor(v, dtype=torch.float64)).tolist()


INFLOW = (1.0, 0.4, 0.0, 0.0, 1.0)


def _initial(case, seed):
    """The initial state of a case in its precision, (nvars, ndofs)."""
    nd = len(case["nel"])
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    dtype = torch.float64 if case["precision"] == "fp64" else torch.float32
    x = _coords(case)
    start, length = _box(case)
    full = x[0].shape
    noise = torch.randn((nd + 2,) + tuple(full), generator=g, device=DEV, dtype=torch.float64)
    ph = (2 * math.pi * torch.rand(8, generator=g, device=DEV, dtype=torch.float64)).tolist()
    y = [2 * math.pi * (c - s) / l for c, s, l in zip(x, start, length)]
    if case["eq"] == "advection":
        Q = torch.ones(full, dtype=torch.float64, device=DEV)
        for k, c in enumerate(y):
            Q = Q * torch.exp(torch.sin(c + ph[k]))
        return (Q + 1e-3 * noise[0]).reshape(1, -1).to(dtype).contiguous()
    one = torch.ones(full, dtype=torch.float64, device=DEV)
    s = case["setup"]
    if s == "sod":
        left = x[0] < 0.5
        prim = torch.stack([torch.where(left, 1.0, 0.125) * one, 0 * one, torch.where(left, 100.0, 10.0) * one])
        prim = prim * (1 + 1e-3 * noise)
    elif s == "shock":
        a, b = _shock_states()
        left = x[0] < 0
        prim = torch.stack([torch.where(left, p, q) * one for p, q in zip(a, b)]) * (1 + 1e-3 * noise)
    elif s == "channel":
        bump = torch.sin(y[0] / 2) ** 2
        prim = torch.stack([one + 0.05 * bump * torch.cos(y[1] + ph[0]), 0.4 * one + 0.05 * bump * torch.sin(y[2] + ph[1]),
                            0.05 * torch.sin(y[1] / 2) * bump, 0.05 * bump * torch.cos(y[2] + ph[2]),
                            one + 0.05 * bump * torch.sin(y[1] + ph[3])])
        prim = prim + 1e-4 * noise
    else:
        # Taylor-Green like velocities on a smooth density and pressure, with noise
        u = [0.3 * torch.sin(y[0] + ph[0]) * torch.cos(y[1] + ph[1]), -0.3 * torch.cos(y[0] + ph[0]) * torch.sin(y[1] + ph[1])]
        if nd == 3:
            u = [c * torch.cos(y[2] + ph[2]) for c in u] + [0.1 * torch.sin(y[2] + ph[3]) * torch.cos(y[0] + ph[4])]
        rho = 1 + 0.1 * torch.sin(y[0] + y[1] + ph[5])
        p = 1 + 0.1 * torch.cos(y[0] - y[1] + ph[6])
        prim = torch.stack([rho * one] + u + [p * one]) + 1e-3 * noise
    return _cons(prim).reshape(nd + 2, -1).to(dtype).contiguous()


def _dt(case):
    """A fixed time step well inside the stability limit of every set-up."""
    start, length = _box(case)
    h = min(l / e for l, e in zip(length, case["nel"])) / case["n"]
    speed = {"sod": 16.0, "shock": 4.5}.get(case.get("setup"), 2.0) if case["eq"] == "euler" else 5.0
    return 0.08 * h / speed * (0.4 if case.get("curved") else 1.0)


def _cfl(case):
    return 0.08


# -------------------------------------------------------------------- handles and passes
_SOLVER = {"ssprk33": F.SSPRK33, "ck2n54": F.CarpenterKennedy2N54, "ork256": F.ORK256}
_TP = {"std": F.StdAverage, "ch": F.ChandrasekharAverage, "kg": F.KennedyGruber}


@functools.lru_cache(maxsize=1)
def _disc(key):
    """The discretisation of a case: a program builds it once and runs many states on it."""
    case = dict(key)
    nd, n = len(case["nel"]), case["n"]
    start, length = _box(case)
    std_t = {1: F.StdSegment, 2: F.StdQuad, 3: F.StdHex}[nd]
    b = F.LagrangeBasis("GLL", n)
    adv = case["eq"] == "advection"
    std = std_t(b, F.DGSEMrec(b), 1 if adv else nd + 2)
    mesh = F.CartesianMesh(nd, start, [s + l for s, l in zip(start, length)], case["nel"])
    s = case.get("setup")
    bcs = {}
    if s == "sod":
        def ends(_, x, *__):
            return _prim((1.0, 0.0, 100.0) if x[0] < 0.5 else (0.125, 0.0, 10.0))
        bcs = {"1": F.GenericBC(ends), "2": F.GenericBC(ends)}
    elif s == "shock":
        a, c = (_prim(v) for v in _shock_states())

        def ends(_, x, *__):
            return a if x[0] < 0 else c
        mesh.apply_periodicBCs(("3", "4"))
        bcs = {"1": F.GenericBC(ends), "2": F.GenericBC(ends)}
    elif s == "channel":
        mesh.apply_periodicBCs(("5", "6"))
        bcs = {"1": F.EulerInflowBC(_prim(INFLOW)), "2": F.EulerOutflowBC(), "3": F.EulerSlipBC(),
               "4": F.EulerSlipBC()}
    else:
        mesh.apply_periodicBCs(*[(str(2 * k + 1), str(2 * k + 2)) for k in range(nd)])
    if case.get("curved"):
        def mapping(X):
            return X + 0.05 * np.prod(np.sin(2 * np.pi * X), axis=1, keepdims=True)
        mesh.apply_mapping(mapping)
    eq = F.LinearAdvection(3.0, 4.0) if adv else F.EulerEquation(nd, GAMMA)
    surf = F.MatrixDissipation(F.ChandrasekharAverage(), 1.0) if case.get("surf") == "matrix" else \
        F.LxF(F.StdAverage(), 1.0)
    if case["op"] == "strong":
        op = F.StrongDivOperator(surf)
    elif case["op"] == "hybrid":
        op = F.HybridDivOperator(_TP[case["tp"]](), surf, 1.0)
    else:
        op = F.SplitDivOperator(_TP[case["tp"]](), surf)
    return F.MultielementDisc(mesh, std, eq, op, bcs, precision=case["precision"]), eq


def _key(case):
    return tuple(sorted((k, tuple(v) if isinstance(v, (list, tuple)) else v) for k, v in case.items() if k != "name"))


def _cotangent(case, seed, shape, dtype):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) + 77)
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float64).to(dtype)


def prepare(case, seed):
    case = _full(case)
    disc, eq = _disc(_key(case))
    Q0 = _initial(case, seed)
    st = dict(case=case, disc=disc, eq=eq, Q0=Q0, dt=_dt(case))
    kind = case["kind"]
    if kind == "march":
        st["solver"] = _SOLVER[case["scheme"]]()
    elif kind == "cfl":
        lim = F.get_limiter_callback(disc, eq, "zhang_shu", 1e-6) if case["limiter"] else None
        st["solver"] = _SOLVER[case["scheme"]](stage_limiter=lim)
        st["dt"] = F.get_max_dt(Q0, disc, eq, _cfl(case))
    elif kind == "stages":
        st["bufs"] = [disc.new_state() for _ in range(3)]
    elif kind == "vjp":
        st["dQ"], st["W"] = disc.new_state(), _cotangent(case, seed, Q0.shape, Q0.dtype)
    elif kind == "gradient":
        st["W"] = _cotangent(case, seed, Q0.shape, Q0.dtype)
        st["solver"] = _SOLVER[case["scheme"]]()
    elif kind == "monitors":
        st["ke"], st["ent"] = F.get_monitor(disc, eq, "kinetic_energy"), F.get_monitor(disc, eq, "entropy")
    return st


def run(st):
    case, disc, eq, Q0, dt = st["case"], st["disc"], st["eq"], st["Q0"], st["dt"]
    kind = case["kind"]
    if kind == "march":
        Q = Q0.clone()
        F.timeintegrate(Q, disc, eq, st["solver"], case["steps"] * dt, dt=dt)
        return Q
    if kind == "cfl":
        Q = Q0.clone()
        F.timeintegrate(Q, disc, eq, st["solver"], case["steps"] * dt, dt=2 * dt, cfl=_cfl(case))
        return Q
    if kind == "stages":
        code = _SOLVER[case["scheme"]].code
        a, b, c = st["bufs"]
        if case["scheme"] == "ssprk33":
            F.rk_stage(disc, code, 0, dt, Q0, a)
            F.rk_stage(disc, code, 1, dt, a, b, u_base=Q0)
            F.rk_stage(disc, code, 2, dt, b, c, u_base=Q0)
            return c
        cur, oth = Q0, a
        for s in range(5):
            F.rk_stage(disc, code, s, dt, cur, oth, reg=c)
            cur, oth = oth, (b if s == 0 else cur)
        return cur, c
    if kind == "vjp":
        F.rhs_(st["dQ"], Q0, F.EquationConfig(disc, eq))
        Qbar = torch.zeros_like(Q0)
        A.rhs_vjp(Qbar, st["W"], Q0, disc)
        return st["dQ"], Qbar
    if kind == "gradient":
        return A.gradient(disc, st["solver"], Q0, dt, case["steps"], lambda uT: st["W"],
                          checkpoint_every=case["every"], return_state=True)
    out = [F.get_max_dt(Q0, disc, eq, 0.5)]
    out += [F.integrate(Q0, disc, v) for v in range(disc.nvars)]
    return out + [st["ke"](Q0, disc, eq), st["ent"](Q0, disc, eq)]


def work(case):
    case = _full(case)
    nd, n = len(case["nel"]), case["n"]
    nv = 1 if case["eq"] == "advection" else nd + 2
    nn = math.prod(case["nel"]) * n ** nd
    s = 8 if case["precision"] == "fp64" else 4
    state = nn * nv * s
    geo = nn * (nd * nd + 1) * s if case.get("curved") else 0
    if case["eq"] == "advection":
        rhs = nn * nd * (2 * n + 4)
    elif case["op"] == "strong":
        rhs = nn * nd * (2 * n * nv + 25)
    else:
        pair = {"std": 25, "kg": 30, "ch": 45}[case["tp"]] + 4 * nv
        rhs = nn * nd * ((n - 1) / 2 * pair + 30)
        if case["op"] == "hybrid":
            rhs += nn * nd * 150
    nst = 3 if case["scheme"] == "ssprk33" else 5
    # states one step moves: inputs read once, outputs written once, stage by stage
    moved = 8 if nst == 3 else 19
    kind = case["kind"]
    if kind in ("march", "stages"):
        k = case.get("steps", 1)
        return {"bytes": k * (moved * state + nst * geo), "flops": k * nst * rhs}
    if kind == "cfl":
        k, lim = case["steps"], 2 * nst if case["limiter"] else 0
        return {"bytes": k * ((moved + 1 + lim) * state), "flops": k * (nst * rhs + 25 * nn)}
    if kind == "vjp":
        return {"bytes": 6 * state + 2 * geo, "flops": 3 * rhs}
    if kind == "gradient":
        # forward, recomputation of the segments that are not kept, reverse stages
        k = case["steps"]
        again = max(0, k - case["every"])
        fwd, rev = moved * state, (5 * nst + 2) * state
        return {"bytes": (k + again) * fwd + k * rev, "flops": (k + again) * nst * rhs + 2 * k * nst * rhs}
    return {"bytes": state * (1 + 1 + (nv - 1) / nv + 1), "flops": 60 * nn}


# -------------------------------------------------- the scheme in plain torch FP64 (exact)
def _geometry(case, x):
    """(Ja, J): contravariant vectors Ja[d][c] and J per node (floats on affine elements)."""
    nd, n = len(case["nel"]), case["n"]
    _, length = _box(case)
    if not case.get("curved"):
        h = [l / e / 2 for l, e in zip(length, case["nel"])]
        J = math.prod(h)
        return [[J / h[d] if c == d else 0.0 for c in range(nd)] for d in range(nd)], J
    D = torch.tensor(_gll(n)[2], dtype=torch.float64, device=DEV)

    def der(u, k):  # along reference direction k
        return torch.moveaxis(torch.tensordot(u, D, dims=([2 * nd - 1 - k], [1])), -1, 2 * nd - 1 - k)
    X = _warp(x)
    first = (Ellipsis,) + (slice(0, 1),) * nd
    X = [c - c[first] for c in X]
    dX = [[der(c, k) for k in range(nd)] for c in X]
    if nd == 2:
        Ja = [[dX[1][1], -dX[0][1]], [-dX[1][0], dX[0][0]]]
        return Ja, dX[0][0] * dX[1][1] - dX[0][1] * dX[1][0]
    Ja = [[None] * 3 for _ in range(3)]
    for c in range(3):
        m, l = (c + 1) % 3, (c + 2) % 3
        V = [X[l] * dX[m][k] for k in range(3)]
        Ja[0][c] = der(V[1], 2) - der(V[2], 1)
        Ja[1][c] = der(V[2], 0) - der(V[0], 2)
        Ja[2][c] = der(V[0], 1) - der(V[1], 0)
    a = [[dX[c][k] for c in range(3)] for k in range(3)]
    J = a[0][0] * (a[1][1] * a[2][2] - a[1][2] * a[2][1]) + a[0][1] * (a[1][2] * a[2][0] - a[1][0] * a[2][2]) + \
        a[0][2] * (a[1][0] * a[2][1] - a[1][1] * a[2][0])
    return Ja, J


def _pressure(Q):
    return (GAMMA - 1) * (Q[-1] - sum(m * m for m in Q[1:-1]) / (2 * Q[0]))


def _dot(a, b):
    return sum(p * q for p, q in zip(a, b) if not (isinstance(q, float) and q == 0.0))


def _flux(Q, nrm):
    p = _pressure(Q)
    un = _dot(Q[1:-1], nrm) / Q[0]
    return [Q[0] * un] + [m * un + p * c for m, c in zip(Q[1:-1], nrm)] + [(Q[-1] + p) * un]


def _logmean(a, b):
    xi = a / b
    f = (xi - 1) / (xi + 1)
    u = f * f
    near = u < 0.01
    fs = torch.where(near, torch.full_like(f, 0.5), f)
    Fl = torch.log(torch.where(near, torch.full_like(xi, 3.0), xi)) / (2 * fs)
    return (a + b) / (2 * torch.where(near, 1 + u / 3 + u * u / 5 + u * u * u / 7, Fl))


def _two_point(Qa, Qb, nrm, tp):
    ra, rb = Qa[0], Qb[0]
    ua, ub = [m / ra for m in Qa[1:-1]], [m / rb for m in Qb[1:-1]]
    pa, pb = _pressure(Qa), _pressure(Qb)
    if tp == "std":
        return [(p + q) / 2 for p, q in zip(_flux(Qa, nrm), _flux(Qb, nrm))]
    u = [(p + q) / 2 for p, q in zip(ua, ub)]
    un = _dot(u, nrm)
    if tp == "kg":
        p, m = (pa + pb) / 2, (ra + rb) / 2 * un
        return [m] + [m * c + p * k for c, k in zip(u, nrm)] + [m * (Qa[-1] / ra + Qb[-1] / rb) / 2 + p * un]
    ba, bb = ra / (2 * pa), rb / (2 * pb)
    rho, beta, p = _logmean(ra, rb), _logmean(ba, bb), (ra + rb) / (2 * (ba + bb))
    sq = sum(c * c for c in ua) + sum(c * c for c in ub)
    h = 1 / (2 * beta * (GAMMA - 1)) - sq / 4 + p / rho + sum(c * c for c in u)
    m = rho * un
    return [m] + [m * c + p * k for c, k in zip(u, nrm)] + [m * h]


def _entropy(Q):
    p = _pressure(Q)
    s = torch.log(p) - GAMMA * torch.log(Q[0])
    return [(GAMMA - s) / (GAMMA - 1) - sum(m * m for m in Q[1:-1]) / Q[0] / (2 * p)] + [m / p for m in Q[1:-1]] + [-Q[0] / p]


def _matrix_flux(Ql, Qr, d):
    """Chandrasekhar average with matrix dissipation along axis d (Winters et al., 2017)."""
    nd = len(Ql) - 2
    order = [d] + [k for k in range(nd) if k != d]
    L = [Ql[0]] + [Ql[1 + k] for k in order] + [Ql[-1]]
    R = [Qr[0]] + [Qr[1 + k] for k in order] + [Qr[-1]]
    Fn = _two_point(L, R, [1.0] + [0.0] * (nd - 1), "ch")
    pl, pr = _pressure(L), _pressure(R)
    ul, ur = [m / L[0] for m in L[1:-1]], [m / R[0] for m in R[1:-1]]
    um = [(p + q) / 2 for p, q in zip(ul, ur)]
    v2 = 2 * sum(c * c for c in um) - (sum(c * c for c in ul) + sum(c * c for c in ur)) / 2
    bl, br = L[0] / (2 * pl), R[0] / (2 * pr)
    rho, beta, p = _logmean(L[0], R[0]), _logmean(bl, br), (L[0] + R[0]) / (2 * (bl + br))
    a = torch.sqrt(GAMMA * p / rho)
    h = GAMMA / (2 * beta) / (GAMMA - 1) + v2 / 2
    dW = [p_ - q_ for p_, q_ in zip(_entropy(L), _entropy(R))]
    one, zero, u, nv = torch.ones_like(a), torch.zeros_like(a), um[0], nd + 2
    cols = [[one, u - a] + um[1:] + [h - u * a], [one, u] + um[1:] + [v2 / 2]]
    for k in range(1, nd):
        cols.append([zero, zero] + [one if j == k else zero for j in range(1, nd)] + [um[k]])
    cols.append([one, u + a] + um[1:] + [h + u * a])
    lam = [torch.abs(u - a)] + [torch.abs(u)] * nd + [torch.abs(u + a)]
    T = [rho / (2 * GAMMA), (GAMMA - 1) * rho / GAMMA] + [p] * (nd - 1) + [rho / (2 * GAMMA)]
    for c, l, t in zip(cols, lam, T):
        s = l * t * sum(c[j] * dW[j] for j in range(nv)) / 2
        Fn = [f + s * c[i] for i, f in enumerate(Fn)]
    out = [Fn[0]] + [None] * nd + [Fn[-1]]
    for i, k in enumerate(order):
        out[1 + k] = Fn[1 + i]
    return out


def _lxf(Ql, Qr, nrm):
    """Rusanov flux along nrm (not unit), scaled by its length."""
    if all(isinstance(c, float) for c in nrm):
        ln = math.sqrt(sum(c * c for c in nrm))
    else:
        ln = torch.sqrt(sum(c * c for c in nrm))
    speeds = [torch.abs(_dot(Q[1:-1], nrm) / Q[0]) + ln * torch.sqrt(GAMMA * _pressure(Q) / Q[0]) for Q in (Ql, Qr)]
    lam = torch.maximum(*speeds)
    return [(f + g) / 2 + lam * (p - q) / 2 for f, g, p, q in zip(_flux(Ql, nrm), _flux(Qr, nrm), Ql, Qr)]


def _ends(case, d, side, own):
    """Exterior state at the box's end of axis d, or None where the axis is periodic."""
    s = case.get("setup")
    if s == "sod":
        v = _prim((1.0, 0.0, 100.0) if side == 0 else (0.125, 0.0, 10.0))
    elif s == "shock" and d == 0:
        v = _prim(_shock_states()[side])
    elif s == "channel" and d == 0:
        if side == 1:
            return own
        v = _prim(INFLOW)
    elif s == "channel" and d == 1:
        return [-q if k == 2 else q for k, q in enumerate(own)]
    else:
        return None
    return [torch.full_like(own[0], c) for c in v]


def _rhs(case, Q, geo):
    """dQ/dt of Q (nv, *nel reversed, *n reversed), differentiable."""
    nd, n = len(case["nel"]), case["n"]
    _, w, D = _gll(n)
    Ja, J = geo
    adv = case["eq"] == "advection"
    out = [[] for _ in range(Q.shape[0])]
    total = None
    for d in range(nd):
        ax, ex = 2 * nd - 1 - d, nd - 1 - d  # node and element axis of one variable
        q = [[Q[v].select(ax, i) for v in range(Q.shape[0])] for i in range(n)]
        M = [[c if isinstance(c, float) else c.select(ax, i) for c in Ja[d]] for i in range(n)]
        if adv:
            an = Ja[d][d] * (3.0, 4.0)[d]
            f = [[an * q[i][0]] for i in range(n)]
        elif case["op"] == "strong":
            f = [_flux(q[i], M[i]) for i in range(n)]
        rows = [None] * n

        def add(i, c, F_):
            rows[i] = [c * t for t in F_] if rows[i] is None else [r + c * t for r, t in zip(rows[i], F_)]
        if adv or case["op"] == "strong":
            for i in range(n):
                for k in range(n):
                    if D[i, k] != 0.0:
                        add(i, -D[i, k], f[k])
        else:
            pairs = {}
            for i in range(n):
                for j in range(i + 1, n):
                    nrm = [(a + b) / 2 for a, b in zip(M[i], M[j])]
                    pairs[i, j] = _two_point(q[i], q[j], nrm, case["tp"])
            if case["op"] == "split":
                for (i, j), F_ in pairs.items():
                    add(i, -2 * D[i, j], F_)
                    add(j, -2 * D[j, i], F_)
            else:
                W = [_entropy(s) for s in q]
                for s in range(1, n):
                    Fb = None
                    for (l, k), F_ in pairs.items():
                        if l < s <= k:
                            t = [2 * w[l] * D[l, k] * c for c in F_]
                            Fb = t if Fb is None else [a + b for a, b in zip(Fb, t)]
                    Fv = [c * Ja[d][d] for c in _matrix_flux(q[s - 1], q[s], d)]
                    b = sum((r - l) * (x - y) for l, r, x, y in zip(W[s - 1], W[s], Fb, Fv))
                    root = torch.sqrt(b * b + 1.0)
                    de = torch.clamp((root - b) / root, min=0.5)
                    Fx = [(1 - de) * y + de * x for x, y in zip(Fb, Fv)]
                    add(s - 1, -1 / w[s - 1], Fx)
                    add(s, 1 / w[s], Fx)
        # faces: left state = last node of the element below, right state = own first node
        right = q[0]
        left = [torch.roll(t, 1, dims=ex) for t in q[n - 1]]
        lo, hi = [t.narrow(ex, 0, 1) for t in q[0]], [t.narrow(ex, t.shape[ex] - 1, 1) for t in q[n - 1]]
        el, er = (None, None) if adv else (_ends(case, d, 0, lo), _ends(case, d, 1, hi))
        top = [t.narrow(ex, 0, 1) for t in right]
        if el is not None:
            left = [torch.cat([g, t.narrow(ex, 1, t.shape[ex] - 1)], dim=ex) for g, t in zip(el, left)]
        nrm = [c if isinstance(c, float) else c for c in M[0]]

        def surface(l, r, m):
            if adv:
                return [an * (l[0] + r[0]) / 2 + abs(an) * (l[0] - r[0]) / 2]
            if case["surf"] == "matrix":
                return [c * Ja[d][d] for c in _matrix_flux(l, r, d)]
            return _lxf(l, r, m)
        Fl = surface(left, right, nrm)
        Fr = [torch.roll(t, -1, dims=ex) for t in Fl]
        if er is not None:
            end = surface(hi, er, [c if isinstance(c, float) else c.narrow(ex, c.shape[ex] - 1, 1) for c in M[n - 1]])
            Fr = [torch.cat([t.narrow(ex, 0, t.shape[ex] - 1), g], dim=ex) for t, g in zip(Fr, end)]
        if adv or case["op"] == "strong":
            Fl = [a - b for a, b in zip(Fl, f[0])]
            Fr = [a - b for a, b in zip(Fr, f[n - 1])]
        add(0, 1 / w[0], Fl)
        add(n - 1, -1 / w[n - 1], Fr)
        part = torch.stack([torch.stack([rows[i][v] for i in range(n)], dim=ax) for v in range(Q.shape[0])])
        total = part if total is None else total + part
    return total / J


_CK = ([0.0, -567301805773 / 1357537059087, -2404267990393 / 2016746695238, -3550918686646 / 2091501179385,
        -1275806237668 / 842570457699],
       [1432997174477 / 9575080441755, 5161836677717 / 13612068292357, 1720146321549 / 2090206949498,
        3134564353537 / 4481467310338, 2277821191437 / 14882151754819])
_ORK = ([0.0, -1.0, -1.55798, -1.0, -0.45031], [0.2, 0.83204, 0.6, 0.35394, 0.2])


def _step(case, Q, dt, geo, after=lambda u: u):
    if case["scheme"] == "ssprk33":
        a = after(Q + dt * _rhs(case, Q, geo))
        b = after((3 * Q + a + dt * _rhs(case, a, geo)) / 4)
        return after((Q + 2 * b + 2 * dt * _rhs(case, b, geo)) / 3), None
    As, Bs = _CK if case["scheme"] == "ck2n54" else _ORK
    reg = None
    for a, b in zip(As, Bs):
        L = dt * _rhs(case, Q, geo)
        reg = L if reg is None else a * reg + L
        Q = after(Q + b * reg)
    return Q, reg


def _weights(case, J):
    nd, n = len(case["nel"]), case["n"]
    w = torch.tensor(_gll(n)[1], dtype=torch.float64, device=DEV)
    W = torch.ones((n,) * nd, dtype=torch.float64, device=DEV)
    for k in range(nd):
        shape = [1] * nd
        shape[k] = n
        W = W * w.reshape(shape)
    return W * J


def _limit(case, Q, minval=1e-6):
    nd = len(case["nel"])
    axes = tuple(range(nd, 2 * nd))
    _, length = _box(case)
    W = _weights(case, math.prod(l / e / 2 for l, e in zip(length, case["nel"])))
    vol = math.prod(l / e for l, e in zip(length, case["nel"]))

    def mean(t):
        return (W * t).sum(dim=axes, keepdim=True) / vol
    qm = [mean(t) for t in Q]

    def pull(t, m, th):
        return torch.where(th <= 1, th * (t - m) + m, t)
    lo = Q[0].amin(dim=axes, keepdim=True)
    th = torch.abs((qm[0] - torch.clamp(qm[0], max=minval)) / (qm[0] - lo))
    Q = [pull(Q[0], qm[0], th)] + list(Q[1:])
    p = _pressure(Q)
    pm = mean(p)
    th = torch.abs((pm - torch.clamp(pm, max=minval)) / (pm - p.amin(dim=axes, keepdim=True)))
    return torch.stack([pull(t, m, th) for t, m in zip(Q, qm)])


def _max_dt(case, Q, cfl, J):
    nd, n = len(case["nel"]), case["n"]
    if isinstance(J, float):
        dx = (J * 2.0 ** nd / n ** nd) ** (1.0 / nd)
    else:
        axes = tuple(range(nd, 2 * nd))
        dx = (_weights(case, J).sum(dim=axes, keepdim=True) / n ** nd) ** (1.0 / nd)
    speed = torch.sqrt(sum(m * m for m in Q[1:-1])) / Q[0] + torch.sqrt(GAMMA * _pressure(Q) / Q[0])
    return float((cfl * dx / speed).min())


def exact(case, seed):
    case = _full(case)
    nd, n = len(case["nel"]), case["n"]
    Q0 = _initial(case, seed)
    dtype = Q0.dtype
    Q = Q0.to(torch.float64).reshape((Q0.shape[0],) + tuple(reversed(case["nel"])) + (n,) * nd)
    geo = _geometry(case, _coords(case))
    dt, kind = _dt(case), case["kind"]

    def flat(t):
        return t.reshape(t.shape[0], -1)
    if kind == "march":
        for _ in range(case["steps"]):
            Q = _step(case, Q, dt, geo)[0]
        return flat(Q)
    if kind == "cfl":
        d0 = _max_dt(case, Q, _cfl(case), geo[1])
        t, tf = 0.0, case["steps"] * d0
        after = (lambda u: _limit(case, u)) if case["limiter"] else (lambda u: u)
        while t < tf * (1 - 1e-14):
            step = min(_max_dt(case, Q, _cfl(case), geo[1]), min(2 * d0, tf - t))
            Q = _step(case, Q, step, geo, after)[0]
            t += step
        return flat(Q)
    if kind == "stages":
        out, reg = _step(case, Q, dt, geo)
        return flat(out) if reg is None else (flat(out), flat(reg))
    if kind in ("vjp", "gradient"):
        W = _cotangent(case, seed, Q0.shape, dtype).to(torch.float64).reshape(Q.shape)
        Q.requires_grad_(True)
        if kind == "vjp":
            out = _rhs(case, Q, geo)
        else:
            out = Q
            for _ in range(case["steps"]):
                out = _step(case, out, dt, geo)[0]
        bar, = torch.autograd.grad(out, Q, W)
        out = out.detach()
        return (flat(out), flat(bar)) if kind == "vjp" else (flat(bar), flat(out))
    wq = _weights(case, geo[1])
    ent = -Q[0] * (torch.log(_pressure(Q)) - GAMMA * torch.log(Q[0])) / (GAMMA - 1)
    ke = sum(m * m for m in Q[1:-1]) / (2 * Q[0])
    return [_max_dt(case, Q, 0.5, geo[1])] + [float((wq * t).sum()) for t in Q] + [float((wq * ke).sum()),
                                                                                     float((wq * ent).sum())]
