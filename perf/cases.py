"""The work whose speed is followed: what programs have this framework do,
through its public entry points, over the sizes they do it at.

Six kinds of program:

  box       a resident periodic 3D simulation: `steps` RK2 steps at the CFL dt,
            then the state as device tensors
  plane     the same in 2D (x-y problems such as Orszag-Tang)
  outflow   a 3D box with outflow sides, its state read back to host arrays
  patches   many periodic cubes advanced together, each with its own dt, read
            back to host arrays
  gradient  a rollout of `steps` fixed-dt steps and its reverse pass
  advance   one AdvanceStep through the C interface on a program's own ghosted
            host arrays, dt by the CFL rule

Inputs are seeded random fields: density and pressure about 1, subsonic
turbulent velocity and a divergence-free field from an edge potential, as the
benchmark's state, on boxes of any shape.
"""

from __future__ import annotations

import ctypes
import math
import random

import numpy as np
import torch

from pluto_amd import adjoint, native, plutoabi, problems

GAMMA = 5.0 / 3.0
CFL, CFL_VAR = 0.4, 1.1
SOLVERS = {"hlld": native.SOLVER_HLLD, "hll": native.SOLVER_HLL, "hllc": native.SOLVER_HLLC,
           "tvdlf": native.SOLVER_TVDLF}
PRECISION = {"fp64": native.PGPU_PREC_FP64, "fp32": native.PGPU_PREC_FP32_FLUX,
             "fast": native.PGPU_PREC_FP64_FAST}
F64 = torch.float64
# FLOPs of one zone-update: IEEE add, multiply, divide and square root of the
# 3D HLLD + UCT_HLL step, counted in the oracle's arithmetic
FLOPS_3D = 3476.0
FLOPS_2D = 2100.0


def _box(name, nx, ny, nz, steps, precision="fp64", solver="hlld", emf="uct_hll"):
    c = dict(kind="box", nx=nx, ny=ny, nz=nz, steps=steps, precision=precision, solver=solver,
             emf=emf)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the benchmark's box: the ordinary production size of one GPU's share
        _box("box_256", 256, 256, 256, 4),
        # small enough that launches and the march along a row set the time:
        # parameter studies, tests, coarse runs
        _box("box_32", 32, 32, 32, 16),
        # odd extents along every axis: domains sized by the problem
        _box("box_131x93x77", 131, 93, 77, 8),
        # rows wider than 256 cells, the largest box here
        _box("box_384x288x320", 384, 288, 320, 2),
        # the FP32-flux precision
        _box("box_256_fp32", 256, 256, 256, 4, precision="fp32"),
        # the tolerance-mode FP64 flux
        _box("box_160_fast", 160, 160, 160, 6, precision="fast"),
        # another Riemann solver and the EMF average that PLUTO's
        # configurations choose most after the default
        _box("box_128_hllc_contact", 128, 128, 128, 8, solver="hllc", emf="uct_contact"),
        # 2D problems
        dict(name="plane_512", kind="plane", nx=512, ny=512, steps=16),
        # non-periodic sides: the ghosted box, ghost zones refilled each stage
        dict(name="outflow_128", kind="outflow", nx=128, ny=128, nz=128, steps=16),
        # AMR-like patches of the benchmark's edges
        dict(name="patches_96", kind="patches", count=96, edges="16,24,32,48,64", steps=24),
        # the gradient of a short rollout (variational problems)
        dict(name="gradient_128", kind="gradient", nx=128, ny=128, nz=128, steps=4),
        # a PLUTO program calling the library in place of its own AdvanceStep
        dict(name="advance_128", kind="advance", nx=128, ny=128, nz=128),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: every kind, sizes spread over their
    logarithm, half of the extents left as they fall (odd ones among them)
    and half rounded to a multiple of 8."""
    def size(lo, hi):
        n = _log_int(rng, lo, hi)
        return n if rng.random() < 0.5 else max(lo, n // 8 * 8)

    kind = rng.choice(["box"] * 5 + ["plane", "outflow", "patches", "gradient", "advance"])
    if kind == "box":
        nx, ny, nz = size(16, 400), size(16, 320), size(16, 320)
        while nx * ny * nz > 34_000_000:
            ny, nz = max(16, ny * 3 // 4), max(16, nz * 3 // 4)
        steps = max(1, min(16, 60_000_000 // (nx * ny * nz)))
        precision = rng.choice(["fp64", "fp64", "fp64", "fp32", "fast"])
        solver, emf = "hlld", "uct_hll"
        if precision == "fp64" and rng.random() < 0.5:
            solver = rng.choice(list(SOLVERS))
            emf = rng.choice(["arithmetic", "uct0", "uct_contact", "uct_hll"])
        return _box(None, nx, ny, nz, steps, precision, solver, emf)
    if kind == "plane":
        return dict(kind=kind, nx=size(48, 1024), ny=size(48, 1024), steps=rng.randint(4, 16))
    if kind == "outflow":
        return dict(kind=kind, nx=size(16, 144), ny=size(16, 128), nz=size(16, 128),
                    steps=rng.randint(4, 16))
    if kind == "patches":
        edges = rng.choice(["16,24,32,48,64", "8,12,16,20,24", "16,32", "15,21,24,33,40", "64"])
        return dict(kind=kind, count=rng.randint(8, 80), edges=edges, steps=rng.randint(4, 24))
    if kind == "gradient":
        return dict(kind=kind, nx=size(16, 136), ny=size(16, 120), nz=size(16, 120),
                    steps=rng.randint(1, 5))
    return dict(kind=kind, nx=size(16, 128), ny=size(16, 128), nz=size(16, 128))


# ---------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------

def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _field(rng, shape, shift=(0.0, 0.0, 0.0), modes=None, kmax=6, dims=3):
    """A random field of 40 plane waves of the unit box, amplitude |k|^-2,
    sampled at cell centres displaced by shift (in cells)."""
    nz, ny, nx = shape
    k, ph, amp = modes if modes is not None else _modes(rng, kmax, dims)
    dev = _device()

    def pos(n, s):
        return (torch.arange(n, dtype=F64, device=dev) + 0.5 + s) / n

    k = torch.as_tensor(k, dtype=F64, device=dev)
    ph = torch.as_tensor(ph, dtype=F64, device=dev)
    amp = torch.as_tensor(amp, dtype=F64, device=dev)
    az = 2 * math.pi * pos(nz, shift[2])[:, None] * k[None, :, 2]
    ay = 2 * math.pi * pos(ny, shift[1])[:, None] * k[None, :, 1] + ph
    ax = 2 * math.pi * pos(nx, shift[0])[None, :] * k[:, 0, None]
    zy = (az[:, None, :] + ay[None, :, :]).reshape(nz * ny, -1)
    left = torch.cat([zy.cos() * amp, -zy.sin() * amp], 1)
    return (left @ torch.cat([ax.cos(), ax.sin()], 0)).reshape(shape)


def _modes(rng, kmax, dims):
    k = []
    while len(k) < 40:
        v = rng.integers(-kmax, kmax + 1, 3)
        if dims == 2:
            v[2] = 0
        if 1 <= math.sqrt(float(v @ v)) <= kmax:
            k.append(v)
    k = np.array(k, dtype=np.float64)
    amp = rng.standard_normal(40) / np.sum(k * k, axis=1)
    return k, rng.uniform(0.0, 2 * math.pi, 40), amp


def _curl(a, d, dims):
    """Face fields from the edge potentials a = (ax, ay, az)."""
    def dif(f, ax):
        return f - torch.roll(f, 1, ax)
    x, y, z = -1, -2, -3
    bx, by = dif(a[2], y) / d[1], -dif(a[2], x) / d[0]
    if dims == 2:
        return torch.stack([bx, by, torch.zeros_like(bx)])
    bx = bx - dif(a[1], z) / d[2]
    by = by + dif(a[0], z) / d[2]
    return torch.stack([bx, by, dif(a[1], x) / d[0] - dif(a[0], y) / d[1]])


def _average(b, dims):
    """Cell-centred field of periodic faces."""
    out = [0.5 * (b[a] + torch.roll(b[a], 1, -1 - a)) for a in range(3)]
    if dims == 2:
        out[2] = torch.zeros_like(out[2])
    return out


def _initial(shape, seed, dims=3, smooth=False):
    """(prim [8,nz,ny,nx], faces [3,nz,ny,nx], spacing) on the unit box.
    smooth: a weak perturbation of rho = p = 1, B = (1,0,0)."""
    rng = np.random.default_rng([int(seed), dims, *shape])
    d = tuple(1.0 / n for n in (shape[2], shape[1], shape[0]))
    kmax = 3 if smooth else 6
    f = [_field(rng, shape, kmax=kmax, dims=dims) for _ in range(5)]
    f = [(x - x.mean()) / x.std() for x in f]
    amp = 0.05 if smooth else 0.5 / math.sqrt(3.0)
    shifts = ((0.0, 0.5, 0.5), (0.5, 0.0, 0.5), (0.5, 0.5, 0.0))
    b = _curl([_field(rng, shape, s, kmax=kmax, dims=dims) for s in shifts], d, dims)
    b = b * ((0.1 if smooth else 0.5) / b.square().sum(0).mean().sqrt())
    if smooth:
        b[0] += 1.0
    v = [amp * x for x in f[2:]]
    if dims == 2:
        v[2] = torch.zeros_like(v[2])
    rho = 1.0 + (0.05 if smooth else 0.1) * f[0]
    p = torch.ones_like(rho) if smooth else 1.0 + 0.05 * f[1]
    return torch.stack([rho, *v, *_average(b, dims), p]), b.contiguous(), d


def _shape(case):
    return (case.get("nz", 1), case["ny"], case["nx"])


def _first_dt(prim, d, dims):
    """A CFL-limited first step from the fast speeds of the state."""
    a2 = GAMMA * prim[7] / prim[0]
    c2 = (prim[4:7].square().sum(0)) / prim[0]
    c = (a2 + c2).sqrt()
    inv = sum((prim[1 + a].abs() + c) / d[a] for a in range(dims))
    return 0.8 * CFL * dims / float(inv.max())


def _patch_edges(case, seed):
    r = random.Random(case["count"])    # the same patches for every seed
    kinds = [int(e) for e in case["edges"].split(",")]
    return [r.choice(kinds) for _ in range(case["count"])]


def _host(prim, b, dims=3):
    p, f = prim.cpu().numpy(), b.cpu().numpy()
    return problems.MHDState(p, f[0], f[1], f[2], dims, (1.0, 1.0, 1.0))


def _dp(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))


# ---------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------

class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.case, s.kind = case, case["kind"]
    lib = native.lib()
    if s.kind == "patches":
        edges = _patch_edges(case, seed)
        s.batch = native.Batch(edges, GAMMA)
        zones = sum(n ** 3 for n in edges)
        s.prim, s.faces = np.ones(8 * zones), np.ones(3 * zones)   # the patches one after another
        s.views, dts, o = [], [], 0
        for p, n in enumerate(edges):
            prim, b, d = _initial((n, n, n), seed * 4099 + p)
            s.batch.set_patch(p, _host(prim, b))
            dts.append(_first_dt(prim, d, 3))
            z = n ** 3
            s.views.append((s.prim[8 * o:8 * (o + z)],
                            s.faces[3 * o:3 * (o + z)].reshape(3, z)))
            o += z
        s.batch.set_dt(min(dts), CFL, CFL_VAR)
        return s
    shape, dims = _shape(case), 2 if s.kind == "plane" else 3
    prim, b, d = _initial(shape, seed, dims, smooth=s.kind == "gradient")
    dt = _first_dt(prim, d, dims)
    if s.kind in ("box", "plane"):
        s.dom = native.Domain(shape, dims, d if dims == 3 else (d[0], d[1], 1.0), GAMMA,
                              precision=PRECISION[case.get("precision", "fp64")],
                              solver=SOLVERS[case.get("solver", "hlld")],
                              emf_average=native.EMF_AVERAGES[case.get("emf", "uct_hll")])
        s.dom.set_dt(dt, CFL, CFL_VAR)
        torch.cuda.synchronize()
        native.check(lib.pgpu_set_state_device(s.dom.h, ctypes.c_void_p(prim.data_ptr()),
                                               ctypes.c_void_p(b.data_ptr())))
        s.dom.sync()
        s.prim, s.faces = prim, b          # the program's tensors: its output from now on
    elif s.kind == "outflow":
        s.dom = native.Domain(shape, 3, d, GAMMA, bounds=["outflow"] * 6)
        s.dom.set_state(_host(prim, b))
        s.dom.set_dt(dt, CFL, CFL_VAR)
        s.prim, s.faces = np.ones((8,) + shape), np.ones((3,) + shape)
    elif s.kind == "gradient":
        s.stepper = adjoint.Stepper(shape, d, 0.5 * dt, GAMMA)
        s.prim, s.faces = prim.requires_grad_(True), b.requires_grad_(True)
        rng = torch.Generator(device=prim.device).manual_seed(int(seed) + 1)
        s.weights = [torch.randn(x.shape, generator=rng, dtype=F64, device=x.device)
                     for x in (prim, b)]
    else:
        s.lib = plutoabi.load_abi(native.LIB_PATH)
        s.box = plutoabi.PlutoBox(_host(prim, b))
        s.solver = ctypes.cast(s.lib.HLLD_Solver, ctypes.c_void_p).value
        s.lib.SetSolver(b"hlld")
        s.dt = dt
    return s


def run(s):
    if s.kind in ("box", "plane"):
        s.dom.run(s.case["steps"])
        native.check(native.lib().pgpu_get_state_device(
            s.dom.h, ctypes.c_void_p(s.prim.data_ptr()), ctypes.c_void_p(s.faces.data_ptr())))
        return {"prim": s.prim, "faces": s.faces}
    if s.kind == "outflow":
        s.dom.run(s.case["steps"])
        native.check(native.lib().pgpu_get_state(s.dom.h, _dp(s.prim), _dp(s.faces[0]),
                                                 _dp(s.faces[1]), _dp(s.faces[2])))
        return {"prim": s.prim, "faces": s.faces}
    if s.kind == "patches":
        s.batch.run(s.case["steps"])
        for p, (prim, faces) in enumerate(s.views):
            native.check(native.lib().pgpu_batch_get_patch(
                s.batch.h, p, _dp(prim), _dp(faces[0]), _dp(faces[1]), _dp(faces[2])))
        return {"prim": s.prim, "faces": s.faces}
    if s.kind == "gradient":
        out = adjoint.rollout(s.prim, s.faces, s.stepper, s.case["steps"])
        grad = torch.autograd.grad(out, (s.prim, s.faces), s.weights)
        return {"prim": out[0].detach(), "faces": out[1].detach(), "d_prim": grad[0],
                "d_faces": grad[1]}
    # one step of a PLUTO program's loop: AdvanceStep, then the next dt by the CFL rule
    ctypes.c_double.in_dll(s.lib, "g_dt").value = s.dt
    ctypes.c_double.in_dll(s.lib, "g_maxMach").value = 0.0
    s.box.dts.invDt_hyp = 0.0
    if s.lib.AdvanceStep(ctypes.byref(s.box.data), s.solver, ctypes.byref(s.box.dts),
                         ctypes.byref(s.box.grid)) != 0:
        raise RuntimeError("AdvanceStep failed")
    s.dt = min(CFL / s.box.dts.invDt_hyp, CFL_VAR * s.dt)
    return _advanced(s.box, s.dt)


def _advanced(box, dt):
    """The box's interior cells and their upper faces, in its own arrays."""
    nz, ny, nx = box.st.shape
    g = box.ng
    return {"prim": box.vc[:, g:g + nz, g:g + ny, g:g + nx],
            "bx": box.vs[0][g:g + nz, g:g + ny, g + 1:g + 1 + nx],
            "by": box.vs[1][g:g + nz, g + 1:g + 1 + ny, g:g + nx],
            "bz": box.vs[2][g + 1:g + 1 + nz, g:g + ny, g:g + nx], "dt": dt}


def work(case):
    """320 bytes per zone-update (a read and a write of the eight variables by
    the first stage, a read of the stage's input and of the step's input and a
    write by the second), the state out; the reverse of a step as three
    steps' arithmetic and twice its traffic."""
    kind = case["kind"]
    if kind == "patches":
        zones = sum(n ** 3 for n in _patch_edges(case, 0))
    else:
        zones = case["nx"] * case["ny"] * case.get("nz", 1)
    steps = case.get("steps", 1)
    flops = FLOPS_2D if kind == "plane" else FLOPS_3D
    if kind == "gradient":
        return {"bytes": zones * (steps * 3 * 320 + 4 * 88), "flops": zones * steps * 4 * flops}
    return {"bytes": zones * (steps * 320 + 88 * (2 if kind == "advance" else 1)),
            "flops": zones * steps * flops}


def tolerance(case):
    # about four times and more what this file's plain 64-bit steps (below),
    # which take sums and quotients in other orders, differ by over a pass:
    # FP64 states 9e-16 (24 steps), FP32 flux 5e-8 (16 steps), gradients
    # 3e-12 (their terms cancel; the reverse pass contracts multiply-adds)
    if case.get("precision") == "fp32":
        return {"rel": 2.5e-7, "max": 2e-5}
    if case["kind"] == "gradient":
        return {"rel": 5e-11, "max": 1e-8}
    return {"rel": 1e-14, "max": 1e-11}


# ---------------------------------------------------------------------
# the same steps in plain 64-bit torch
# ---------------------------------------------------------------------
# Arrays are [..., nz, ny, nx]; axis a (0 x, 1 y, 2 z) is dimension -1-a.
# U and V: lists of eight arrays (rho, x, y, z momenta or velocities, Bx, By,
# Bz, energy or pressure); b: the three face fields.

def _at(f, a, n):
    """f at n cells further along axis a."""
    return torch.roll(f, -n, -1 - a)


def _mc(dp, dm, strict):
    lim = 2.0 * torch.where(dp.abs() < dm.abs(), dp, dm)
    cen = 0.5 * (dp + dm)
    s = torch.where(cen.abs() < lim.abs(), cen, lim)
    return torch.where(dp * dm > 0 if strict else dp * dm >= 0, s, torch.zeros_like(s))


def _slope(f, a, strict):
    return _mc(_at(f, a, 1) - f, f - _at(f, a, -1), strict)


def _cons(V):
    rho, v, B, p = V[0], V[1:4], V[4:7], V[7]
    E = p / (GAMMA - 1) + 0.5 * (rho * sum(x * x for x in v) + sum(x * x for x in B))
    return [rho, *[rho * x for x in v], *B, E]


def _prim(U):
    v = [m / U[0] for m in U[1:4]]
    kin = 0.5 * (sum(m * x for m, x in zip(U[1:4], v)) + sum(x * x for x in U[4:7]))
    return [U[0], *v, *U[4:7], (GAMMA - 1) * (U[7] - kin)]


def _flux(V, U, n):
    """Ideal MHD flux along axis n, the total pressure in the normal momentum."""
    v, B = V[1:4], V[4:7]
    pt = V[7] + 0.5 * sum(x * x for x in B)
    F = [U[1 + n]] + [v[n] * U[1 + a] - B[n] * B[a] for a in range(3)]
    F[1 + n] = F[1 + n] + pt
    F += [v[n] * B[a] - B[n] * v[a] for a in range(3)]
    F.append((U[7] + pt) * v[n] - B[n] * sum(x * y for x, y in zip(v, B)))
    return F, pt


def _fast(V, n):
    a2 = GAMMA * V[7] / V[0]
    bn2 = V[4 + n] ** 2 / V[0]
    s = a2 + sum(x * x for x in V[4:7]) / V[0]
    bt2 = sum(V[4 + a] ** 2 for a in range(3) if a != n) / V[0]
    return (0.5 * (s + ((a2 - bn2 - bt2) ** 2 + 4.0 * a2 * bt2).sqrt())).sqrt()


def _pick(c, x, y):
    return [torch.where(c, p, q) for p, q in zip(x, y)]


def _riemann(solver, VL, VR, n):
    """Flux (8), SL, SR and the signal speed of the interfaces along axis n."""
    t, b = [a for a in range(3) if a != n]
    UL, UR = _cons(VL), _cons(VR)
    FL, pL = _flux(VL, UL, n)
    FR, pR = _flux(VR, UR, n)
    if solver == "tvdlf":
        M = [0.5 * (x + y) for x, y in zip(VL, VR)]
        c = M[1 + n].abs() + _fast(M, n)
        return [0.5 * (f + g - c * (y - x)) for f, g, x, y in zip(FL, FR, UL, UR)], -c, c, c
    cL, cR = _fast(VL, n), _fast(VR, n)
    SL = torch.minimum(VL[1 + n] - cL, VR[1 + n] - cR)
    SR = torch.maximum(VL[1 + n] + cL, VR[1 + n] + cR)
    w = 1.0 / (SR - SL)
    Fh = [(SR * f - SL * g + SL * SR * (y - x)) * w for f, g, x, y in zip(FL, FR, UL, UR)]
    if solver == "hll":
        F = Fh
    else:
        Uh = [(SR * y - SL * x + f - g) * w for f, g, x, y in zip(FL, FR, UL, UR)]
        star = _hllc if solver == "hllc" else _hlld
        F = star(n, t, b, VL, VR, UL, UR, FL, FR, pL, pR, SL, SR, Uh, Fh)
    F = _pick(SL >= 0, FL, _pick(SR <= 0, FR, F))
    return F, SL, SR, torch.maximum(SL.abs(), SR.abs())


def _hllc(n, t, b, VL, VR, UL, UR, FL, FR, pL, pR, SL, SR, Uh, Fh):
    """Li (2005)."""
    S = Uh[1 + n] / Uh[0]
    B = Uh[4:7]
    ps = Fh[1 + n] + B[n] ** 2 - Fh[0] * S
    vB = sum(m * x for m, x in zip(Uh[1:4], B)) / Uh[0]
    out = []
    for V, U, F, pt, Sk in ((VL, UL, FL, pL, SL), (VR, UR, FR, pR, SR)):
        d, e = Sk - V[1 + n], 1.0 / (Sk - S)
        Us = [None] * 8
        Us[0] = U[0] * d * e
        Us[1 + n] = Us[0] * S
        for a in (t, b):
            Us[1 + a] = (U[1 + a] * d - (B[n] * B[a] - V[4 + n] * V[4 + a])) * e
        Us[4:7] = B
        Us[7] = (U[7] * d + ps * S - pt * V[1 + n] - B[n] * vB
                 + V[4 + n] * sum(x * y for x, y in zip(V[1:4], V[4:7]))) * e
        out.append([f + Sk * (s - u) for f, s, u in zip(F, Us, U)])
    return _pick(S >= 0, out[0], out[1])


def _hlld(n, t, b, VL, VR, UL, UR, FL, FR, pL, pR, SL, SR, Uh, Fh):
    """Miyoshi & Kusano (2005); where an Alfven wave meets an outer one the
    fast star states hold the single-state field and no rotation."""
    Bn = Uh[4 + n]
    sg = torch.where(Bn > 0, 1.0, -1.0).to(F64)
    dL, dR = SL - VL[1 + n], SR - VR[1 + n]
    q = 1.0 / (dR * UR[0] - dL * UL[0])
    SM = (dR * UR[1 + n] - dL * UL[1 + n] - pR + pL) * q
    ps = (dR * UR[0] * pL - dL * UL[0] * pR
          + VL[0] * VR[0] * dR * dL * (VR[1 + n] - VL[1 + n])) * q
    side = []
    for V, U, pt, Sk, d, sgn in ((VL, UL, pL, SL, dL, -1.0), (VR, UR, pR, SR, dR, 1.0)):
        rho = U[0] * d / (Sk - SM)
        root = rho.sqrt()
        S1 = SM + sgn * Bn.abs() / root
        side.append((V, U, pt, Sk, d, rho, root, S1))
    (lo, hi) = ((s[7], s[3]) for s in side)
    flat = ((lo[0] - lo[1]) < 1e-4 * (SM - lo[1])) | ((hi[0] - hi[1]) > -1e-4 * (hi[1] - SM))
    star = []
    for V, U, pt, Sk, d, rho, root, S1 in side:
        k = (U[0] * d * d - Bn * Bn) / torch.where(flat, torch.ones_like(d),
                                                 U[0] * d * (Sk - SM) - Bn * Bn)
        Us = [None] * 8
        Us[0], Us[1 + n], Us[4 + n] = rho, rho * SM, Bn
        vs = {}
        for a in (t, b):
            Us[4 + a] = torch.where(flat, Uh[4 + a], U[4 + a] * k)
            vs[a] = V[1 + a] - Bn / (U[0] * d) * (Us[4 + a] - U[4 + a])
            Us[1 + a] = rho * vs[a]
        vB = V[1 + n] * Bn + V[1 + t] * U[4 + t] + V[1 + b] * U[4 + b]
        vBs = SM * Bn + vs[t] * Us[4 + t] + vs[b] * Us[4 + b]
        Us[7] = (d * U[7] - pt * V[1 + n] + ps * SM + Bn * (vB - vBs)) / (Sk - SM)
        star.append((Us, vs, vBs, root, torch.where(flat, SM, S1)))
    (Ul, vl, el, rl, S1L), (Ur, vr, er, rr, S1R) = star
    i = 1.0 / (rl + rr)
    mid = []
    vm = {a: (rl * vl[a] + rr * vr[a] + (Ur[4 + a] - Ul[4 + a]) * sg) * i for a in (t, b)}
    Bm = {a: (rl * Ur[4 + a] + rr * Ul[4 + a] + rl * rr * (vr[a] - vl[a]) * sg) * i
          for a in (t, b)}
    em = SM * Bn + sum(vm[a] * Bm[a] for a in (t, b))
    for Us, e, r, s in ((Ul, el, rl, -1.0), (Ur, er, rr, 1.0)):
        Um = [None] * 8
        Um[0], Um[1 + n], Um[4 + n] = Us[0], Us[1 + n], Bn
        for a in (t, b):
            Um[1 + a], Um[4 + a] = Us[0] * vm[a], Bm[a]
        Um[7] = Us[7] + s * r * (e - em) * sg
        mid.append(Um)
    fl = [f + SL * (s - u) for f, s, u in zip(FL, Ul, UL)]
    fr = [f + SR * (s - u) for f, s, u in zip(FR, Ur, UR)]
    gl = [f + S1L * (m - s) for f, m, s in zip(fl, mid[0], Ul)]
    gr = [f + S1R * (m - s) for f, m, s in zip(fr, mid[1], Ur)]
    return _pick(S1L >= 0, fl, _pick(S1R <= 0, fr, _pick(SM >= 0, gl, gr)))


def _edge_emf(c, emf, V, b, faces):
    """EMF on the edges along axis c: E_c = v_q b_p - v_p b_q, p, q the next axes."""
    p, q = (c + 1) % 3, (c + 2) % 3
    if emf == "uct_hll":
        (SLp, SRp, dp), (SLq, SRq, dq) = faces[p]["hll"], faces[q]["hll"]
        ap, am = torch.maximum(SRp, _at(SRp, q, 1)), torch.maximum(SLp, _at(SLp, q, 1))
        cp, cm = torch.maximum(SRq, _at(SRq, p, 1)), torch.maximum(SLq, _at(SLq, p, 1))
        sp, sq = _slope(b[p], q, False), _slope(b[q], p, False)
        bS, bN = b[p] + 0.5 * sp, _at(b[p] - 0.5 * sp, q, 1)
        bW, bE = b[q] + 0.5 * sq, _at(b[q] - 0.5 * sq, p, 1)

        def corner(x, y, bp, bq):
            vq = V[1 + q] + 0.5 * (x * dp[q] + y * dq[q])
            vp = V[1 + p] + 0.5 * (x * dp[p] + y * dq[p])
            vq, vp = (_at(_at(v, p, int(x < 0)), q, int(y < 0)) for v in (vq, vp))
            return vq * bp - vp * bq

        e = ap * cp * corner(1, 1, bS, bW) + am * cp * corner(-1, 1, bS, bE) \
            + am * cm * corner(-1, -1, bN, bE) + ap * cm * corner(1, -1, bN, bW)
        return e / ((ap + am) * (cp + cm)) - cp * cm * (bN - bS) / (cp + cm) \
            + ap * am * (bE - bW) / (ap + am)
    fp, fq = -faces[p]["flux"][4 + q], faces[q]["flux"][4 + p]
    cell = V[1 + q] * V[4 + p] - V[1 + p] * V[4 + q]
    if emf == "uct0":
        fp = 2.0 * fp - 0.5 * (cell + _at(cell, p, 1))
        fq = 2.0 * fq - 0.5 * (cell + _at(cell, q, 1))
    e = fp + _at(fp, q, 1) + fq + _at(fq, p, 1)
    if emf == "uct_contact":
        def up(f, s, a):
            g = _at(f, a, 1)
            return torch.where(s > 1e-6, f, torch.where(s < -1e-6, g, 0.5 * (f + g)))
        mp, mq = faces[p]["flux"][0], faces[q]["flux"][0]
        e = e + up(fq - cell, mp, p) + up(fp - cell, mq, q)
        e = e - up(_at(cell, p, 1) - fp, _at(mq, p, 1), q)
        e = e - up(_at(cell, q, 1) - fq, _at(mp, q, 1), p)
    return 0.25 * e


def _stage(V, b, U, dt, d, dims, solver, emf):
    """U + dt L(V, b), the faces after dt, and the cells' signal rates."""
    rate, out, faces = 0.0, list(U), [None] * 3
    for a in range(dims):
        s = [_slope(x, a, True) for x in V]
        VL = [x + 0.5 * y for x, y in zip(V, s)]
        VR = [_at(x - 0.5 * y, a, 1) for x, y in zip(V, s)]
        VL[4 + a] = VR[4 + a] = b[a]
        F, SL, SR, c = _riemann(solver, VL, VR, a)
        faces[a] = {"hll": ((-SL).clamp(min=0), SR.clamp(min=0), s[1:4]), "flux": F}
        out = [u - dt / d[a] * (f - _at(f, a, -1)) for u, f in zip(out, F)]
        rate = rate + 0.5 * (c + _at(c, a, -1)) / d[a]
    E = [_edge_emf(c, emf, V, b, faces) if dims == 3 or c == 2 else None for c in range(3)]
    new = []
    for a in range(3):
        p, q = (a + 1) % 3, (a + 2) % 3
        f = b[a]
        if dims == 3 or a < 2:
            if E[q] is not None and p < dims:
                f = f - dt / d[p] * (E[q] - _at(E[q], p, -1))
            if E[p] is not None and q < dims:
                f = f + dt / d[q] * (E[p] - _at(E[p], q, -1))
        new.append(f)
    return out, new, rate


def _with_field(U, b, dims):
    B = [0.5 * (b[a] + _at(b[a], a, -1)) for a in range(3)]
    if dims == 2:
        B[2] = torch.zeros_like(B[2])
    return _prim([*U[:4], *B, U[7]])


def _step(V, b, dt, d, dims=3, solver="hlld", emf="uct_hll", ghosts=None):
    if ghosts:
        V, b = ghosts(V, b)
    U0 = _cons(V)
    U, b1, rate = _stage(V, b, U0, dt, d, dims, solver, emf)
    V1 = _with_field(U, b1, dims)
    if ghosts:
        V1, b1 = ghosts(V1, b1)
    U, b2, _ = _stage(V1, b1, U, dt, d, dims, solver, emf)
    b2 = [0.5 * (x + y) for x, y in zip(b, b2)]
    U = [0.5 * (x + y) for x, y in zip(U0, U)]
    return _with_field(U, b2, dims), b2, rate / dims


def _outflow(n, d):
    """Ghost fill of a block of n + 5 cells per axis whose interior starts at
    cell 3: zero gradient for all but the normal face field, which keeps the
    ghost cells' divergence zero."""
    def fill(V, b):
        V, b = [x.clone() for x in V], [x.clone() for x in b]
        for a in range(3):
            lo, hi = 3, 3 + n[a]
            m = [x.movedim(-1 - a, 0) for x in V]
            f = [x.movedim(-1 - a, 0) for x in b]
            for x in m + [f[c] for c in range(3) if c != a]:
                x[:lo] = x[lo]
                x[hi:] = x[hi - 1]
            div = sum((b[c] - _at(b[c], c, -1)) / d[c] for c in range(3) if c != a) * d[a]
            div = div.movedim(-1 - a, 0)
            for k in (2, 1):
                f[a][k - 1] = f[a][k] + div[k]
            for k in (hi, hi + 1):
                f[a][k] = f[a][k - 1] - div[k]
            for k in (1, 2, hi, hi + 1):
                m[4 + a][k] = 0.5 * (f[a][k] + f[a][k - 1])
        return V, b
    return fill


def _march(V, b, dt, d, steps, dims=3, solver="hlld", emf="uct_hll", ghosts=None, inside=None):
    """steps CFL steps; dt of shape [..., 1, 1, 1]."""
    for _ in range(steps):
        V, b, rate = _step(V, b, dt, d, dims, solver, emf, ghosts)
        rate = rate[inside] if inside else rate
        dt = torch.minimum(CFL / rate.amax((-1, -2, -3), keepdim=True), CFL_VAR * dt)
    return V, b, dt


def exact(case, seed):
    kind = case["kind"]
    if kind == "patches":
        return _exact_patches(case, seed)
    shape, dims = _shape(case), 2 if kind == "plane" else 3
    prim, b, d = _initial(shape, seed, dims, smooth=kind == "gradient")
    dt = torch.tensor(_first_dt(prim, d, dims), dtype=F64, device=prim.device).reshape(1, 1, 1)
    if kind == "gradient":
        return _exact_gradient(case, prim, b, 0.5 * dt, d, seed)
    with torch.no_grad():
        steps = case.get("steps", 1)
        if kind == "outflow":
            n = (case["nx"], case["ny"], case["nz"])
            at = (slice(None),) + tuple(slice(3, 3 + n[a]) for a in (2, 1, 0))
            V, f = (torch.ones((x.shape[0],) + tuple(m + 5 for m in shape), dtype=F64,
                               device=x.device) for x in (prim, b))
            V[at], f[at] = prim, b
            for a in range(3):                 # the lower face: image of the last one
                x, y = (z[a].movedim(-1 - a, 0) for z in (f, b))
                x[2][tuple(s for c, s in zip((2, 1, 0), at[1:]) if c != a)] = y[-1]
            V, f, dt = _march(list(V), list(f), dt, d, steps, ghosts=_outflow(n, d), inside=at[1:])
            return {"prim": torch.stack(V)[at], "faces": torch.stack(f)[at]}
        V, f, dt = _march(list(prim), list(b), dt, d, steps, dims, case.get("solver", "hlld"),
                          case.get("emf", "uct_hll"))
        if kind == "advance":
            return {"prim": torch.stack(V), "bx": f[0], "by": f[1], "bz": f[2], "dt": float(dt)}
        return {"prim": torch.stack(V), "faces": torch.stack(f)}


def _exact_patches(case, seed):
    edges = _patch_edges(case, seed)
    start = {}
    dts = []
    for p, n in enumerate(edges):
        prim, b, d = _initial((n, n, n), seed * 4099 + p)
        dts.append(_first_dt(prim, d, 3))
        start.setdefault(n, []).append((p, prim, b))
    out = [None] * len(edges)
    with torch.no_grad():
        for n, group in start.items():
            V = list(torch.stack([g[1] for g in group], 1))
            b = list(torch.stack([g[2] for g in group], 1))
            dt = torch.full((len(group), 1, 1, 1), min(dts), dtype=F64, device=V[0].device)
            V, b, dt = _march(V, b, dt, (1.0 / n,) * 3, case["steps"])
            V, b = torch.stack(V), torch.stack(b)
            for i, (p, _, _) in enumerate(group):
                out[p] = (V[:, i].reshape(-1).cpu().numpy(), b[:, i].reshape(-1).cpu().numpy())
    return {"prim": np.concatenate([o[0] for o in out]),
            "faces": np.concatenate([o[1] for o in out])}


def _exact_gradient(case, prim, b, dt, d, seed):
    from torch.utils.checkpoint import checkpoint
    prim, b = prim.requires_grad_(True), b.requires_grad_(True)
    rng = torch.Generator(device=prim.device).manual_seed(int(seed) + 1)
    weights = [torch.randn(x.shape, generator=rng, dtype=F64, device=x.device) for x in (prim, b)]

    def step(V, f):
        V, f, _ = _step(list(V), list(f), dt, d)
        return torch.stack(V), torch.stack(f)

    V = torch.cat([prim[:4], torch.stack(_average(b, 3)), prim[7:]])
    f = b
    for _ in range(case["steps"]):
        V, f = checkpoint(step, V, f, use_reentrant=False)
    g = torch.autograd.grad((V, f), (prim, b), weights, allow_unused=True)
    return {"prim": V.detach(), "faces": f.detach(), "d_prim": g[0], "d_faces": g[1]}
