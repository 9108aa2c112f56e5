"""The measured workloads: what a program that uses this package has it do.

Five kinds of work, each through the public entry points:

  step2d    Solver (2D): a rollout of whole TVD-RK2 / RK2 steps from a given
            state to the state after them
  step3d    the same in 3D, ideal or resistive
  ensemble  Ensemble: uneven 2D grids advanced together
  adjoint   Adjoint: forward with checkpoints, then the reverse pass (2D, and
            3D resistive with the resistivity gradient)
  routines  openmhd_amd.api: the reference's subroutines one by one on device
            arrays, as a driver written like its main program calls them (one
            Runge-Kutta stage: u2v, limiter, face patch, flux_solver, set_dt,
            rk_tvd21, bc, glm_ss2)

Sizes are those of the repository's configurations (Orszag-Tang 200^2 and
512^2, Kelvin-Helmholtz 4096^2, an uneven Kelvin-Helmholtz ensemble with sides
from 64, the 512x256x256 resistive Harris sheet) and odd ones between them.
A rollout's pass starts from the state it is given each time, so passes repeat.

`exact` restates the scheme in plain torch float64 (autograd for the reverse
pass), written from the scheme's formulas and independent of the package.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import openmhd_amd as om
from openmhd_amd import api

DEV = "cuda"
F64 = torch.float64
GAMMA = 5.0 / 3.0
ETA = (1.0e-3, 1.0e-2, 2.0)  # eta0, eta1, w of the localized resistivity


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _step2d(name, problem, nx, ny, steps, lim, flux=3, rk=0, mode="host"):
    return dict(name=name, kind="step2d", problem=problem, nx=nx, ny=ny, nz=0, steps=steps, lim=lim, flux=flux, rk=rk,
                mode=mode)


def listed():
    return [
        # the smallest grid of the ensemble configuration run alone: launch and round-trip latency per step
        _step2d("kh_64", "kh", 64, 64, 10, 1),
        # the Orszag-Tang acceptance grid (MC limiter, periodic), the default host-dt loop
        _step2d("ot_200", "ot", 200, 200, 20, 2),
        # an ordinary grid with ragged sides, the other integrator, Koren slopes and the LHLLD flux
        _step2d("kh_1030x517_lhlld", "kh", 1030, 517, 10, 4, flux=4, rk=1, mode="device"),
        # an ordinary production grid, device dt replayed from a graph
        _step2d("ot_1000_graph", "ot", 1000, 1000, 10, 2, mode="graph"),
        # the Kelvin-Helmholtz benchmark grid
        _step2d("kh_4096", "kh", 4096, 4096, 10, 1, mode="device"),
        # a parameter scan: uneven grids advanced together
        dict(name="ensemble_48", kind="ensemble", members=48, smin=64, smax=768, steps=20, lim=1, graph=True),
        # a 3D periodic run of ordinary, ragged size
        dict(name="ideal3d_130x70x50", kind="step3d", problem="modes", nx=130, ny=70, nz=50, steps=5, lim=2, flux=3,
             rk=0, mode="host"),
        # the 3D resistive reconnection grid
        dict(name="harris3d_512", kind="step3d", problem="harris", nx=512, ny=256, nz=256, steps=2, lim=1, flux=3, rk=0,
             mode="host"),
        # gradient with respect to the initial state on the 512^2 adjoint grid
        dict(name="adjoint2d_512", kind="adjoint", problem="ot", nx=512, ny=512, nz=0, steps=10, every=5, lim=2),
        # gradient of a resistive 3D run, resistivity parameters included
        dict(name="adjoint3d_192x96x80", kind="adjoint", problem="harris", nx=192, ny=96, nz=80, steps=2, every=2,
             lim=1),
        # the reference-style driver on the Orszag-Tang grid: per-call latency
        dict(name="routines_200", kind="routines", nx=200, ny=200, nz=0, lim=2, flux=3),
        # the same on a 3D block: memory traffic of the separate routines
        dict(name="routines_160x128x120", kind="routines", nx=160, ny=128, nz=120, lim=1, flux=3),
    ]


def draw(rng):
    def log(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    lim = rng.choice((1, 1, 2, 2, 3, 4))
    kind = rng.choice(("step2d", "step2d", "step2d", "ensemble", "step3d", "step3d", "adjoint", "adjoint", "routines"))
    if kind == "step2d":
        return dict(kind=kind, problem=rng.choice(("kh", "ot")), nx=log(64, 3600), ny=log(64, 3600), nz=0,
                    steps=rng.randint(5, 12), lim=lim, flux=rng.choice((3, 3, 3, 4)), rk=rng.choice((0, 0, 1)),
                    mode=rng.choice(("host", "device", "graph")))
    if kind == "ensemble":
        return dict(kind=kind, members=rng.randint(4, 48), smin=64, smax=log(128, 768), steps=rng.randint(5, 20),
                    lim=lim, graph=rng.random() < 0.5)
    if kind == "step3d":
        return dict(kind=kind, problem=rng.choice(("modes", "harris")), nx=log(48, 320), ny=log(24, 200),
                    nz=log(16, 200), steps=rng.randint(1, 4), lim=lim, flux=3, rk=rng.choice((0, 0, 1)), mode="host")
    if kind == "adjoint":
        steps = rng.randint(2, 8)
        if rng.random() < 0.5:
            return dict(kind=kind, problem="ot", nx=log(96, 640), ny=log(96, 640), nz=0, steps=steps,
                        every=rng.randint(1, steps), lim=lim)
        return dict(kind=kind, problem="harris", nx=log(48, 192), ny=log(24, 96), nz=log(16, 80), steps=2,
                    every=rng.randint(1, 2), lim=lim)
    if rng.random() < 0.5:
        return dict(kind=kind, nx=log(64, 2000), ny=log(64, 2000), nz=0, lim=lim, flux=rng.choice((3, 3, 4)))
    return dict(kind=kind, nx=log(32, 160), ny=log(24, 128), nz=log(16, 120), lim=lim, flux=3)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) & 0x7FFFFFFF)


def _conserved(ro, vx, vy, vz, p, bx, by, bz, psi):
    en = 0.5 * (ro * (vx * vx + vy * vy + vz * vz) + (bx * bx + by * by + bz * bz)) + p / (GAMMA - 1)
    return torch.stack([ro * vx, ro * vy, ro * vz, en, ro, bx, by, bz, psi + 0 * en])


def _smooth(seed, n, grids, modes=4):
    """n smooth random fields of amplitude about 1: a few periodic modes each."""
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(n):
        f = 0.0
        for _ in range(modes):
            arg = rng.uniform(0, 2 * math.pi)
            for g in grids:
                arg = arg + float(rng.integers(-4, 5)) * g
            f = f + float(rng.uniform(0.2, 0.5)) * torch.sin(arg)
        out.append(f)
    return out


def _angles(n, shape, axis):
    """Cell centres of one axis as an angle in [0, 2 pi), shaped to broadcast."""
    a = (torch.arange(n, dtype=F64, device=DEV) + 0.5) * (2 * math.pi / n)
    return a.reshape([n if k == axis else 1 for k in range(len(shape))])


def _initial(case, seed):
    """(W, dx, origin): interior state W(9, [nz,] ny, nx) on the device."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    problem = case["problem"]
    shape = (nz, ny, nx) if nz else (ny, nx)
    one = torch.ones(shape, dtype=F64, device=DEV)
    if problem == "kh":  # shear layer between walls, seeded noise near it
        dx = 40.0 / nx
        y = ((torch.arange(ny, dtype=F64, device=DEV) + 0.5) * dx - 0.5 * ny * dx)[:, None]
        noise = 1.0e-3 * torch.randn(shape, dtype=F64, device=DEV, generator=_gen(seed))
        vy = torch.where(y.abs() < 2.0, noise, 0 * noise)
        z = 0 * one
        return _conserved(one, 0.5 * torch.tanh(y) * one, vy, z, 1.04 * one, 0.2 * one, z, one, z), dx, (0.0, 0.0)
    ax = [_angles(n, shape, k) for k, n in enumerate(shape)]
    if problem == "harris":  # current sheet between y walls, seeded velocity noise, smooth modes in the other fields
        dx = 0.125
        y = ((torch.arange(ny, dtype=F64, device=DEV) + 0.5) * dx - 0.5 * ny * dx)[None, :, None]
        ro = (0.2 + torch.cosh(y) ** -2 / 0.2) * one
        g = _gen(seed)
        v = [1.0e-3 * torch.randn(shape, dtype=F64, device=DEV, generator=g) for _ in range(3)]
        b = [1.0e-2 * f * one for f in _smooth(seed, 6, ax)]
        return (_conserved(ro * (1 + b[3]), v[0], v[1], v[2], 0.1 * ro * (1 + b[4]), torch.tanh(y) + b[0], b[1], b[2],
                           0.1 * b[5]), dx,
                (-0.5 * nx * dx, -0.5 * ny * dx))
    # Orszag-Tang in the plane (2D "ot", 3D "modes") with smooth modes in every field
    dx = 2 * math.pi / nx
    X, Y = ax[-1], ax[-2]
    s = _smooth(seed, 9, ax)
    a = 0.05
    return (_conserved(GAMMA ** 2 * (1 + a * s[0]), -torch.sin(Y) + a * s[1], torch.sin(X) + a * s[2], a * s[3] * one,
                       GAMMA * (1 + a * s[4]), -torch.sin(Y) + a * s[5], torch.sin(2 * X) + a * s[6], a * s[7] * one,
                       0.01 * s[8] * one), dx, (0.0, 0.0))


def _walls(case):
    """Per axis: 'periodic' or 'wall' (the y walls of the shear layer and the sheet)."""
    return ("periodic", "wall" if case["problem"] in ("kh", "harris") else "periodic", "periodic")


def _resistive(case):
    return ETA if case["problem"] == "harris" else None


def _solver(case, dx, origin):
    return om.Solver(case["nx"], case["ny"], dx, nz=case["nz"], cfl=0.4, lm_type=case["lim"],
                     flux_type=case.get("flux", 3), time_type=case.get("rk", 0), bc=_walls(case),
                     resistivity=_resistive(case), origin=origin)


def _members(case, seed):
    rng = np.random.default_rng(case["members"] * 1009 + case["smax"])
    span = math.log(case["smin"]), math.log(case["smax"])
    sides = [[int(round(math.exp(rng.uniform(*span)))) for _ in range(2)] for _ in range(case["members"])]
    return [dict(problem="kh", nx=a, ny=b, nz=0, seed=int(seed) * 64 + m) for m, (a, b) in enumerate(sides)]


def _fortran(W, wall_y):
    """The reference's array U(ix, jx[, kx], 9), column-major with ghosts, of an interior state."""
    nd = W.dim() - 1
    U = torch.empty(tuple(n + 2 for n in W.shape[1:][::-1]) + (9,), dtype=F64, device=DEV)
    U = torch.empty_strided(U.shape, [int(np.prod(U.shape[:k])) for k in range(nd + 1)], dtype=F64, device=DEV)
    P = W
    for axis in range(nd, 0, -1):
        P = _pad(P, axis, 1, wall_y and axis == nd - 1)
    U.copy_(P.permute(*range(nd, 0, -1), 0))
    return U


def prepare(case, seed):
    kind = case["kind"]
    if kind == "ensemble":
        mem = _members(case, seed)
        init = [_initial(m, m["seed"]) for m in mem]
        e = om.Ensemble([om.make_config(m["nx"], m["ny"], i[1], cfl=0.4, lm_type=case["lim"], bc=("periodic", "wall"))
                         for m, i in zip(mem, init)])
        U = [_fortran(i[0], True) for i in init]
        for k, u in enumerate(U):
            e.upload(k, u)
        e.set_mode(device_dt=case["graph"], graph=case["graph"])
        return dict(case=case, ens=e, U=U, out=[torch.empty_like(u) for u in U])
    if kind == "routines":
        return _prepare_routines(case, seed)
    W, dx, origin = _initial(case, seed)
    s = _solver(case, dx, origin)
    st = dict(case=case, solver=s, W=W, out=torch.empty_like(W))
    if kind == "adjoint":
        st["adj"] = om.Adjoint(s, case["steps"], case["every"])
        st["lam"] = _seed_adjoint(W, seed)
        st["grad"] = torch.empty_like(W)
    elif case["mode"] != "host":
        s.set_state(W)
        s.set_mode(device_dt=True, graph=case["mode"] == "graph")
    return st


def _seed_adjoint(W, seed):
    """dL/dW(T) of a generic scalar: one random value per entry."""
    return torch.randn(W.shape, dtype=F64, device=DEV, generator=_gen(seed + 77))


def _prepare_routines(case, seed):
    W, dx, _ = _initial(dict(case, problem="modes"), seed)
    U = _fortran(W, False)
    shp = tuple(U.shape[:-1])

    def planes(n):
        st = [int(np.prod(shp[:k])) for k in range(len(shp) + 1)]
        return torch.empty_strided(shp + (n,), st, dtype=F64, device=DEV).zero_()

    return dict(case=case, U=U, V=planes(4), U1=planes(9), VL=planes(9), VR=planes(9),
                flux=[planes(9) for _ in range(len(shp))], dx=dx)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(st):
    kind = st["case"]["kind"]
    if kind == "ensemble":
        e = st["ens"]
        for k, u in enumerate(st["U"]):
            e.upload(k, u)
        e.step(st["case"]["steps"])
        for k, u in enumerate(st["out"]):
            om.lib.omhd_batch_download(e.h, k, ctypes.cast(ctypes.c_void_p(u.data_ptr()),
                                                           ctypes.POINTER(ctypes.c_double)), None)
        return st["out"]
    if kind == "routines":
        return _run_routines(st)
    s = st["solver"]
    s.set_state(st["W"])
    if kind == "adjoint":
        st["adj"].forward()
        s.get_state(st["out"])
        st["adj"].backward(st["lam"], st["grad"])
        eta = st["adj"].eta_grad() if st["case"]["problem"] == "harris" else None
        return [st["out"], st["grad"]] + ([] if eta is None else [eta])
    s.step(st["case"]["steps"])
    return s.get_state(st["out"])


def _run_routines(st):
    case, U, V, U1, VL, VR, dx = st["case"], st["U"], st["V"], st["U1"], st["VL"], st["VR"], st["dx"]
    shp = U.shape[:-1]
    ix, jx, kx = (tuple(shp) + (1,))[:3]
    nd = len(shp)
    api.u2v(U, V, ix, jx, kx)
    ch, dt = api.set_dt(U, V, dx, 0.4, ix, jx, kx, nd)
    for d in range(nd):
        for m in range(9):
            api.limiter(V[..., m] if m < 4 else U[..., m], VL[..., m], VR[..., m], ix, jx, d + 1, case["lim"], kx)
        api.periodic_patch(VL, VR, ix, jx, d + 1, kx)
        api.flux_solver(st["flux"][d], VL, VR, ch, ix, jx, d + 1, case["flux"], kx)
    f = st["flux"]
    api.rk_tvd21(U, U1, f[0], f[1], dt, dx, ix, jx, f[2] if nd == 3 else None, kx)
    api.bc(U1, ix, jx, kx)
    api.glm_ss2(U1, ch, dt, ix, jx, kx)
    return [V, U1] + f


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "ensemble":
        cells = sum(m["nx"] * m["ny"] for m in _members(case, 0))
        return {"bytes": 144.0 * cells * case["steps"], "flops": 1770.0 * cells * case["steps"]}
    nd = 3 if case["nz"] else 2
    cells = case["nx"] * case["ny"] * max(1, case["nz"])
    if kind == "routines":  # each routine reads its arrays once and writes its results once
        return {"bytes": cells * (104.0 + 104 + nd * (9 * 24 + 216) + 144 + 72 * nd + 16), "flops": cells * nd * 420.0}
    per_step = 885.0 * nd  # the scheme's operations per cell and step: two stages of nd interfaces
    if kind == "adjoint":  # forward; then the states and the adjoint read and written per step
        return {"bytes": 432.0 * cells * case["steps"], "flops": 4 * per_step * cells * case["steps"]}
    return {"bytes": 144.0 * cells * case["steps"], "flops": per_step * cells * case["steps"]}  # read U^n, write U^{n+1}


# ---------------------------------------------------------------------------
# the scheme in plain torch float64
# ---------------------------------------------------------------------------
def _wall_sign():
    """Slots negated in a wall's mirror: the normal velocity and By of the shear layer's tables."""
    s = torch.ones(9, dtype=F64, device=DEV)
    s[1] = s[6] = -1.0
    return s


def _pad(W, axis, g, wall, sign=None):
    """g ghost cells along one axis: periodic images, or mirrors with signs."""
    n = W.shape[axis]
    if not wall:
        return torch.cat([W.narrow(axis, n - g, g), W, W.narrow(axis, 0, g)], axis)
    s = (_wall_sign() if sign is None else sign).reshape([-1] + [1] * (W.dim() - 1))
    return torch.cat([s * W.narrow(axis, 0, g).flip(axis), W, s * W.narrow(axis, n - g, g).flip(axis)], axis)


def _prims(U):
    v = [U[m] / U[4] for m in range(3)]
    rv2 = v[0] * U[0] + v[1] * U[1] + v[2] * U[2]
    B2 = U[5] * U[5] + U[6] * U[6] + U[7] * U[7]
    return torch.stack(v + [(GAMMA - 1) * (U[3] - 0.5 * (rv2 + B2))] + [U[m] for m in range(4, 9)])


def _limited(wm, w0, wp, lim):
    """(right state of the lower face, left state of the upper face)."""
    a, b = w0 - wm, wp - w0
    same = torch.where((a > 0) & (b > 0), 1.0, torch.where((a < 0) & (b < 0), -1.0, 0.0))
    lo = torch.minimum(a.abs(), b.abs())
    if lim == 1:
        g = 0.5 * same * lo
        return w0 - g, w0 + g
    if lim == 2:
        g = same * torch.minimum(lo, 0.25 * (wp - wm).abs())
        return w0 - g, w0 + g
    if lim == 3:
        g = torch.where(a * b <= 0, 0 * a, a * b / torch.where(a * b <= 0, 1 + 0 * a, a + b))
        return w0 - g, w0 + g
    r = same * torch.minimum(lo, ((2 * a + b) / 6.0).abs())
    l = same * torch.minimum(lo, ((a + 2 * b) / 6.0).abs())
    return w0 - r, w0 + l


def _side(S, vn, bn):
    """Conserved state (9), flux (9), fast speed^2, total pressure and v.B of one side."""
    v2 = S[0] * S[0] + S[1] * S[1] + S[2] * S[2]
    B2 = S[5] * S[5] + S[6] * S[6] + S[7] * S[7]
    vB = S[0] * S[5] + S[1] * S[6] + S[2] * S[7]
    U = [S[4] * S[0], S[4] * S[1], S[4] * S[2], 0.5 * (S[4] * v2 + B2) + S[3] / (GAMMA - 1)] + [S[m] for m in range(4, 9)]
    pt = S[3] + 0.5 * B2
    F = [S[4] * S[vn] * S[m] - S[bn] * S[5 + m] for m in range(3)]
    F[vn] = F[vn] + pt
    F += [(U[3] + pt) * S[vn] - vB * S[bn], S[4] * S[vn]] + [S[vn] * S[5 + m] - S[bn] * S[m] for m in range(3)]
    F[bn] = 0 * S[4]

    def fast2(gp):
        A = gp + B2
        return (A + torch.sqrt(torch.clamp(A * A - 4 * gp * S[bn] * S[bn], min=0.0))) / (2 * S[4])

    return U, F, fast2(GAMMA * S[3]), pt, vB, fast2(S[4] * v2) if not S[4].requires_grad else None


def _riemann(L, R, ch, d, flux):
    """HLLD (3, with its HLLC-G fallback) or LHLLD (4) flux along axis d (0 x, 1 y, 2 z)."""
    vn, t = d, ((d + 1) % 3, (d + 2) % 3)
    bn = 5 + d
    UL, FL, fL, ptL, vBL, kL = _side(L, vn, bn)
    UR, FR, fR, ptR, vBR, kR = _side(R, vn, bn)
    c = torch.sqrt(torch.maximum(fL, fR))
    aL, aR = torch.minimum(L[vn], R[vn]) - c, torch.maximum(L[vn], R[vn]) + c
    h = 1.0 / (aR - aL)
    Uh = [h * (aR * UR[m] - aL * UL[m] - FR[m] + FL[m]) for m in range(8)]
    aM, hb = Uh[vn] / Uh[4], Uh[bn]
    dL, dR = aL - L[vn], aR - R[vn]
    if flux == 4:
        chi = torch.clamp(torch.maximum(kL, kR) / torch.maximum(fL, fR), max=1.0)
        psi = 2 * torch.sqrt(chi) - chi
        pt = (R[4] * ptL * dR - L[4] * ptR * dL + psi * L[4] * R[4] * dR * dL * (R[vn] - L[vn])) / (R[4] * dR - L[4] * dL)
        fallback = torch.zeros_like(aM, dtype=torch.bool)
    else:
        pt = ptL + L[4] * dL * (aM - L[vn])
    roL, roR = L[4] * dL / (aL - aM), R[4] * dR / (aR - aM)
    sL, sR = torch.sqrt(roL), torch.sqrt(roR)
    aL1, aR1 = aM - hb.abs() / sL, aM + hb.abs() / sR
    if flux == 3:
        fallback = (aL >= aM - 1.001 * (hb.abs() / sL)) | (aM + 1.001 * (hb.abs() / sR) >= aR)

    def energy(a, S, U, p, vB, vt, bt):
        return ((a - S[vn]) * U[3] - p * S[vn] + pt * aM + hb * (vB - aM * hb - vt[0] * bt[0] - vt[1] * bt[1])) / (a - aM)

    def star(a, da, S, U, p, vB, ro):
        den = S[4] * da * (a - aM) - hb * hb
        f = 1.0 / torch.where(fallback, 1 + 0 * den, den)
        bt = [S[5 + m] * f * (S[4] * (da * da) - hb * hb) for m in t]
        vt = [S[m] - f * hb * S[5 + m] * (aM - S[vn]) for m in t]
        return vt, bt, energy(a, S, U, p, vB, vt, bt)

    def state(ro, vt, bt, en):
        s = [None] * 9
        s[vn], s[t[0]], s[t[1]], s[3], s[4] = ro * aM, ro * vt[0], ro * vt[1], en, ro
        s[5 + t[0]], s[5 + t[1]] = bt
        return s

    vL, bL, eL = star(aL, dL, L, UL, ptL, vBL, roL)
    vR, bR, eR = star(aR, dR, R, UR, ptR, vBR, roR)
    S1L, S1R = state(roL, vL, bL, eL), state(roR, vR, bR, eR)
    sg = torch.where(hb >= 0, 1.0, -1.0)
    fs = 1.0 / (sL + sR)
    at = [fs * (sL * vL[q] + sR * vR[q] + (bR[q] - bL[q]) * sg) for q in (0, 1)]
    bt = [fs * (sL * bR[q] + sR * bL[q] + sL * sR * (vR[q] - vL[q]) * sg) for q in (0, 1)]
    e2L = eL - sL * (vL[0] * bL[0] + vL[1] * bL[1] - at[0] * bt[0] - at[1] * bt[1]) * sg
    e2R = eR + sR * (vR[0] * bR[0] + vR[1] * bR[1] - at[0] * bt[0] - at[1] * bt[1]) * sg
    S2L, S2R = state(roL, at, bt, e2L), state(roR, at, bt, e2R)
    if flux == 3:
        av = [Uh[m] / Uh[4] for m in t]
        ub = [Uh[5 + m] for m in t]
        gL = state(roL, av, ub, energy(aL, L, UL, ptL, vBL, av, ub))
        gR = state(roR, av, ub, energy(aR, R, UR, ptR, vBR, av, ub))
    F = [None] * 9
    left = aM >= 0
    for m in [0, 1, 2, 3, 4, 5 + t[0], 5 + t[1]]:
        two = torch.where(left, aL1 * S2L[m] - (aL1 - aL) * S1L[m] - aL * UL[m] + FL[m],
                          aR1 * S2R[m] - (aR1 - aR) * S1R[m] - aR * UR[m] + FR[m])
        f = torch.where(aL1 >= 0, aL * (S1L[m] - UL[m]) + FL[m],
                        torch.where(aR1 <= 0, aR * (S1R[m] - UR[m]) + FR[m], two))
        if flux == 3:
            if m < 5:
                g = torch.where(left, aL * (gL[m] - UL[m]) + FL[m], aR * (gR[m] - UR[m]) + FR[m])
            else:
                g = h * (aR * FL[m] - aL * FR[m] + aL * aR * (R[m] - L[m]))
            f = torch.where(fallback, g, f)
        F[m] = torch.where(aL >= 0, FL[m], torch.where(aR <= 0, FR[m], f))
    F[bn] = 0.5 * ((L[8] + R[8]) - ch * (R[bn] - L[bn]))
    F[8] = 0.5 * (ch * ch * (L[bn] + R[bn]) - ch * (R[8] - L[8]))
    return F


def _interfaces(W, axis, wall, lim):
    """Left and right states of the n+1 faces of an axis."""
    n = W.shape[axis]
    P = _pad(W, axis, 2, wall)
    gR, gL = _limited(P.narrow(axis, 0, n + 2), P.narrow(axis, 1, n + 2), P.narrow(axis, 2, n + 2), lim)
    L, R = gL.narrow(axis, 0, n + 1), gR.narrow(axis, 1, n + 1)
    if wall:  # a wall face's outer state mirrors its inner one
        s = _wall_sign().reshape([-1] + [1] * (W.dim() - 1))
        L = torch.cat([s * R.narrow(axis, 0, 1), L.narrow(axis, 1, n)], axis)
        R = torch.cat([R.narrow(axis, 0, n), s * L.narrow(axis, n, 1)], axis)
    return L, R


def _eta_faces(case, dx, origin, eta):
    """eta at the x-, y- and z-face centres, shaped (1, ny, nx+1), (1, ny+1, nx), (1, ny, nx); and its largest value."""
    xs = []
    for o, n in zip(origin, (case["nx"], case["ny"])):
        c = [o - dx / 2]
        for _ in range(n + 1):
            c.append(c[-1] + dx)
        xs.append(torch.tensor(c, dtype=F64, device=DEV))

    def at(x, y):
        r2 = x[None, :] * x[None, :] + y[:, None] * y[:, None]
        return eta[0] + eta[1] * torch.exp(-r2 / (eta[2] * eta[2]))

    x, y = xs
    faces = [at(x + 0.5 * dx, y), at(x, y + 0.5 * dx), at(x, y)]
    top = max(float(f.max()) for f in faces)
    return [faces[0][None, 1:-1, :-1], faces[1][None, :-1, 1:-1], faces[2][None, 1:-1, 1:-1]], top


def _add_resistive(F, W, d, eta_dx, walls):
    """The resistive flux at the faces of axis d (0 x, 1 y, 2 z) of a 3D state: F[3], and the two transverse B."""
    B = W
    for k in range(3):
        B = _pad(B, 3 - k, 1, walls[k] == "wall")
    q1, q2, tn = 5 + (d + 2) % 3, 5 + (d + 1) % 3, 5 + d
    a1, a2 = (d + 2) % 3, (d + 1) % 3  # axes of the transverse differences of J1 and J2

    def at(m, shift):  # slot m at the face's lower cell, moved by `shift` cells per axis
        v = B[m]
        for k in range(3):
            ax = 2 - k
            n = v.shape[ax] - 2
            v = v.narrow(ax, (0 if k == d else 1) + shift.get(k, 0), n + 1 if k == d else n)
        return v

    def cross(a):
        return 0.25 * (at(tn, {a: 1}) + at(tn, {a: 1, d: 1}) - at(tn, {a: -1}) - at(tn, {a: -1, d: 1}))

    J1 = -(at(q1, {d: 1}) - at(q1, {})) + cross(a1)
    J2 = (at(q2, {d: 1}) - at(q2, {})) - cross(a2)
    F[3] = F[3] + 0.5 * eta_dx * (J1 * (at(q1, {}) + at(q1, {d: 1})) - J2 * (at(q2, {}) + at(q2, {d: 1})))
    F[q1] = F[q1] + eta_dx * J1
    F[q2] = F[q2] - eta_dx * J2


def _fluxes(U, case, ch, walls, eta=None, dx=1.0):
    """Per axis: the 9 flux components at its n+1 faces."""
    W = _prims(U)
    out = []
    for d in range(U.dim() - 1):
        axis = U.dim() - 1 - d
        L, R = _interfaces(W, axis, walls[d] == "wall", case["lim"])
        F = _riemann(L, R, ch, d, case.get("flux", 3))
        if eta is not None:
            _add_resistive(F, U, d, eta[d] / dx, walls)
        out.append(torch.stack(F))
    return out


def _difference(fluxes):
    s = 0.0
    for d, F in enumerate(fluxes):
        axis = F.dim() - 1 - d
        n = F.shape[axis] - 1
        s = s + F.narrow(axis, 0, n) - F.narrow(axis, 1, n)
    return s


def _speed(U):
    W = _prims(U)
    B2 = U[5] * U[5] + U[6] * U[6] + U[7] * U[7]
    gp = GAMMA * W[3]
    s, top = gp + B2, 0.0
    for d in range(U.dim() - 1):
        f = torch.sqrt((s + torch.sqrt(torch.clamp(s * s - 4 * gp * (U[5 + d] * U[5 + d]), min=0.0))) / (2 * U[4]))
        top = max(top, float((W[d].abs() + f).max()))
    return top


def _damp(U, f):
    return torch.cat([U[:8], f * U[8:]])


def _advance(U, case, dt, ch, dx, walls, eta):
    f = math.exp(-0.5 * dt * ch / 0.2)
    U = _damp(U, f)

    def D(X):
        return _difference(_fluxes(X, case, ch, walls, eta, dx))

    if case.get("rk", 0) == 0:
        U1 = U + dt / dx * D(U)
        U = 0.5 * (U + U1 + dt / dx * D(U1))
    else:
        U = U + dt / dx * D(U + 0.5 * dt / dx * D(U))
    return _damp(U, f)


def _dt(U, dx, top_eta):
    ch = _speed(U)
    dt = 0.4 * dx / ch
    return (dt if top_eta is None else min(dt, 0.5 * 0.4 * (dx * dx) / top_eta)), ch


def _rollout(U, case, steps, dx, origin):
    """The state after `steps` steps, and the (dt, ch) sequence taken."""
    walls, eta, top, seq = _walls(case), None, None, []
    if _resistive(case):
        eta, top = _eta_faces(case, dx, origin, ETA)
    for _ in range(steps):
        seq.append(_dt(U, dx, top))
        U = _advance(U, case, *seq[-1], dx, walls, eta)
    return U, seq


def exact(case, seed):
    kind = case["kind"]
    if kind == "ensemble":
        out = []
        for m in _members(case, seed):
            W, dx, origin = _initial(m, m["seed"])
            W, _ = _rollout(W, dict(m, lim=case["lim"]), case["steps"], dx, origin)
            out.append(_fortran(W, True))
        return out
    if kind == "routines":
        return _exact_routines(case, seed)
    W, dx, origin = _initial(case, seed)
    WT, seq = _rollout(W, case, case["steps"], dx, origin)
    return WT if kind != "adjoint" else _exact_adjoint(case, seed, W, WT, seq, dx, origin)


def _exact_adjoint(case, seed, W, WT, seq, dx, origin):
    """Reverse mode by autograd, one step at a time, with the (dt, ch) sequence held fixed."""
    walls, lam = _walls(case), _seed_adjoint(W, seed)
    states, eta = [W], None
    prm = torch.tensor(ETA, dtype=F64, device=DEV, requires_grad=True)
    geta = torch.zeros_like(prm)
    if _resistive(case):
        eta = _eta_faces(case, dx, origin, ETA)[0]
    for dt, ch in seq[:-1]:
        states.append(_advance(states[-1], case, dt, ch, dx, walls, eta))
    for U, (dt, ch) in zip(states[::-1], seq[::-1]):
        U = U.detach().requires_grad_(True)
        if eta is not None:
            eta = _eta_faces(case, dx, origin, prm)[0]
        out = _advance(U, case, dt, ch, dx, walls, eta)
        got = torch.autograd.grad(out, [U] if eta is None else [U, prm], lam)
        lam = got[0]
        if eta is not None:
            geta = geta + got[1]
    return [WT, lam] + ([] if eta is None else [geta.detach().cpu().numpy()])


def _exact_routines(case, seed):
    """Interior of what one stage computes; faces and ghosts the routines leave alone are zero."""
    c = dict(case, problem="modes")
    W, dx, _ = _initial(c, seed)
    walls = ("periodic",) * 3
    nd = W.dim() - 1
    dt, ch = _dt(W, dx, None)
    flux = _fluxes(W, c, ch, walls)
    U1 = _damp(W + dt / dx * _difference(flux), math.exp(-0.5 * dt * ch / 0.2))
    V = _fortran(_prims(W), False)[..., :4].contiguous()
    shp = tuple(n + 2 for n in W.shape[1:])
    whole = []
    for d, F in enumerate(flux):  # face c+1/2 is stored at cell c's place: 1..n-1 of its axis, interior of the others
        G = torch.zeros((9,) + shp, dtype=F64, device=DEV)
        part = G
        for k in range(nd):
            axis = nd - k
            part = part.narrow(axis, 0 if k == d else 1, F.shape[axis])
        part.copy_(F)
        whole.append(G.permute(*range(nd, 0, -1), 0).contiguous())
    return [V, _fortran(U1, False)] + whole
