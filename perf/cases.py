"""The level-set work whose speed is tracked: what a program built on this package asks of it.

Every case is one pass through the public entry points, as a time loop calls them: one TVD-RK3 step with its
ghost fills (fused stages or the reference's own call sequence), a stretch of narrow-band motion between two
rebuilds of the band, or the gradient of a loss through a few steps.  Fields live on the GPU and the library works
on torch's current stream without waiting after each call, as a time loop sets it up once.

``exact`` restates the same schemes in plain torch in 64 bits.
"""
from __future__ import annotations

import math
import random

import torch

from lsmlib_amd.adjoint import NormalMotionAdjoint, autograd_functions
from lsmlib_amd.solver import DropInChain, Grid, NarrowBandRun, Solver, curvature_corrected_dt

G = 3  # ghost layers: the reach of HJ-WENO5
CFL = 0.5
BAND_STEPS = 10  # steps between two rebuilds of a narrow band
VMAX = 1.3  # the largest speed of speed_field


def listed():
    return [
        # a quick look on a coarse grid, stepped thousands of times: latency and launches count
        dict(name="deform_64_f32", kind="step", rhs="deform", path="fused", dtype="f32", nx=64, ny=64, nz=64),
        # reinitialization of a non-distance function as the reference's drivers run it: one call per derivative,
        # term and stage, in double precision
        dict(name="reinit_chain_128_f64", kind="step", rhs="reinit", path="chain", dtype="f64", nx=128, ny=128, nz=128),
        # motion by a speed that varies in space on a box cut to the object: no size a multiple of anything
        dict(name="normal_ragged_f32", kind="step", rhs="normal", path="fused", dtype="f32", nx=203, ny=149, nz=97),
        # advection by a velocity that a flow solver left in memory, double precision, ragged
        dict(name="velocity_ragged_f64", kind="step", rhs="velocity", path="fused", dtype="f64", nx=301, ny=203, nz=157),
        # advection, normal speed and curvature together through the reference's call sequence, with its CFL steps
        dict(name="motion_chain_256_f64", kind="motion", dtype="f64", nx=256, ny=256, nz=256),
        # the production grid: one step of the deformation flow in single and in double precision, and one
        # pseudo-step of the reinitialization that follows every few of them
        dict(name="deform_512_f32", kind="step", rhs="deform", path="fused", dtype="f32", nx=512, ny=512, nz=512),
        dict(name="deform_512_f64", kind="step", rhs="deform", path="fused", dtype="f64", nx=512, ny=512, nz=512),
        dict(name="reinit_512_f32", kind="step", rhs="reinit", path="fused", dtype="f32", nx=512, ny=512, nz=512),
        # a narrow band: rebuild it, then ten steps, through the fused band stages and through the reference's
        # call sequence
        dict(name="band_512_f32", kind="band", path="fused", dtype="f32", n=512),
        dict(name="band_chain_256_f64", kind="band", path="chain", dtype="f64", n=256),
        # shape matching: the loss and its gradients with respect to the initial shape and the speed
        dict(name="gradient_256_f32", kind="gradient", dtype="f32", nx=256, ny=256, nz=256, steps=6, every=3),
        # the planar twins: one reinitialization pseudo-step of an image-sized grid
        dict(name="plane_1024_f64", kind="plane", dtype="f64", nx=1024, ny=1024),
    ]


def _around(rng, size):
    """A size near `size`, odd as often as even."""
    return max(16, int(size * rng.uniform(0.75, 1.3333)))


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "step", "chain", "motion", "band", "gradient", "plane"])
    dtype = rng.choice(["f32", "f64"])
    if kind == "plane":
        s = _log(rng, 64, 3000)
        return dict(kind="plane", dtype=dtype, nx=_around(rng, s), ny=_around(rng, s))
    if kind == "band":
        path = rng.choice(["fused", "chain"])
        return dict(kind="band", path=path, dtype=dtype, n=int(_log(rng, 64, 400 if path == "fused" else 256)))
    if kind == "gradient":
        s = _log(rng, 32, 200)
        return dict(kind="gradient", dtype=dtype, nx=_around(rng, s), ny=_around(rng, s), nz=_around(rng, s),
                    steps=rng.randint(2, 6), every=3)
    if kind == "motion":
        s = _log(rng, 32, 220)
        return dict(kind="motion", dtype="f64", nx=_around(rng, s), ny=_around(rng, s), nz=_around(rng, s))
    if kind == "chain":
        s = _log(rng, 32, 260)
        return dict(kind="step", rhs=rng.choice(["reinit", "normal", "velocity"]), path="chain", dtype=dtype,
                    nx=_around(rng, s), ny=_around(rng, s), nz=_around(rng, s))
    s = _log(rng, 32, 420)
    return dict(kind="step", rhs=rng.choice(["deform", "velocity", "normal", "reinit"]), path="fused", dtype=dtype,
                nx=_around(rng, s), ny=_around(rng, s), nz=_around(rng, s))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
BC = {"deform": "signed_linear", "velocity": "signed_linear", "reinit": "linear", "normal": "periodic"}


def _grid(case):
    n = (case["nx"], case["ny"], case["nz"])
    if case.get("rhs") == "reinit":
        return Grid(n, lo=(-1.0,) * 3, hi=(1.0,) * 3, centred=True)
    return Grid(n)


def _axes(grid):
    """Coordinates of the ghost box as broadcastable (z, y, x) tensors."""
    x, y, z = (torch.as_tensor(grid.axis(d), device="cuda") for d in range(3))
    return x[None, None, :], y[None, :, None], z[:, None, None]


def _spheres(grid, rng, count, centre, radius):
    x, y, z = _axes(grid)
    out = None
    for _ in range(count):
        c = [rng.uniform(*centre) for _ in range(3)]
        r = rng.uniform(*radius)
        d = torch.sqrt((x - c[0]) ** 2 + (y - c[1]) ** 2 + (z - c[2]) ** 2) - r
        out = d if out is None else torch.minimum(out, d)
    return out.contiguous()


def _speed_field(grid, rng):
    """1 + 0.3 tanh(g), g a few low Fourier modes: a speed in (0.7, 1.3) that varies in space."""
    x, y, z = _axes(grid)
    g = 0.0
    for _ in range(4):
        k = [rng.randint(1, 4) for _ in range(3)]
        g = g + rng.uniform(0.3, 1.0) * torch.cos(2 * math.pi * (k[0] * x + k[1] * y + k[2] * z) + rng.uniform(0, 6.28))
    return (1.0 + 0.3 * torch.tanh(g)).contiguous()


def _velocity(grid, rng):
    x, y, z = _axes(grid)
    p = [rng.uniform(0, 2 * math.pi) for _ in range(3)]
    full = torch.zeros(grid.shape, dtype=torch.float64, device="cuda")
    return [(0.5 * torch.sin(2 * math.pi * a + q) + full).contiguous() for a, q in ((y, p[0]), (z, p[1]), (x, p[2]))]


def _inputs(case, seed):
    """phi (and what else the equation needs), in the case's precision."""
    rng = random.Random(seed)
    dtype = torch.float64 if case["dtype"] == "f64" else torch.float32
    inp = {}
    if case["kind"] == "plane":
        nx, ny = case["nx"], case["ny"]
        h = (2.0 / nx, 2.0 / ny)
        c = [rng.uniform(-0.1, 0.1) for _ in range(2)]
        x = -1.0 + h[0] * (torch.arange(-G, nx + G, dtype=torch.float64, device="cuda") + 0.5)[None, :]
        y = -1.0 + h[1] * (torch.arange(-G, ny + G, dtype=torch.float64, device="cuda") + 0.5)[:, None]
        d = torch.sqrt((x - c[0]) ** 2 + (y - c[1]) ** 2) - 0.5
        inp["phi"] = (d * (1 + 0.1 * torch.sin(3 * math.pi * x) * torch.sin(3 * math.pi * y))).to(dtype).contiguous()
        return inp
    if case["kind"] == "band":
        g = Grid((case["n"],) * 3)
        inp["phi"] = _spheres(g, rng, 64, (0.1, 0.9), (0.03, 0.1)).to(dtype)
        return inp
    g = _grid(case)
    rhs = case.get("rhs")
    if case["kind"] == "gradient":
        c = [rng.uniform(0.45, 0.55) for _ in range(3)]
        x, y, z = _axes(g)
        d = torch.sqrt((x - c[0]) ** 2 + (y - c[1]) ** 2 + (z - c[2]) ** 2)
        # the run carries its leaves in double precision; the engine works in the case's
        inp["phi0"] = (d - 0.2).to(dtype).double()
        inp["target"] = (d - 0.2 - 1.5 * g.dx[0]).to(dtype)
        inp["V"] = _speed_field(g, rng).to(dtype).double()
        return inp
    if case["kind"] == "motion" or rhs == "velocity":
        inp["phi"] = _spheres(g, rng, 32, (0.15, 0.85), (0.04, 0.12)).to(dtype)
        inp["vel"] = [v.to(dtype) for v in _velocity(g, rng)]
    elif rhs == "deform":
        inp["phi"] = _spheres(g, rng, 1, (0.32, 0.38), (0.14, 0.16)).to(dtype)
        inp["t"] = rng.uniform(0.0, 1.2)
    elif rhs == "normal":
        inp["phi"] = _spheres(g, rng, 1, (0.45, 0.55), (0.15, 0.25)).to(dtype)
        inp["V"] = _speed_field(g, rng).to(dtype)
    else:
        c = [rng.uniform(-0.1, 0.1) for _ in range(3)]
        x, y, z = _axes(g)
        d = torch.sqrt((x - c[0]) ** 2 + (y - c[1]) ** 2 + (z - c[2]) ** 2) - 0.5
        w = torch.sin(3 * math.pi * x) * torch.sin(3 * math.pi * y) * torch.sin(3 * math.pi * z)
        inp["phi"] = (d * (1 + 0.1 * w)).to(dtype).contiguous()
    return inp


def _dt(case, grid):
    inv = [1.0 / h for h in grid.dx]
    if case["kind"] == "gradient" or case.get("rhs") == "normal":
        return CFL / (VMAX * sum(inv))
    if case.get("rhs") == "deform":
        return CFL / (2 * inv[0] + inv[1] + inv[2])
    if case.get("rhs") == "velocity":
        return CFL / (0.5 * sum(inv))
    return CFL * min(grid.dx)


def _factors(t, dt):
    """cos(pi t / 3) of the deformation field at the three stage times."""
    return [math.cos(math.pi * s / 3.0) for s in (t, t + dt, t + 0.5 * dt)]


def _on_torch_stream(lib):
    lib.set_stream(torch.cuda.current_stream().cuda_stream, synchronous=False)


def prepare(case, seed):
    inp = _inputs(case, seed)
    s = dict(case=case, inp=inp)
    if case["kind"] == "plane":
        from lsmlib_amd.lib import load
        lib = load(case["dtype"])
        _on_torch_stream(lib)
        s["api"] = lib.api
        s["buf"] = [torch.zeros_like(inp["phi"]) for _ in range(9)]
        _fill_plane(s, inp["phi"])
        return s
    if case["kind"] == "band":
        import numpy as np
        run = NarrowBandRun(case["n"], precision=case["dtype"], fused=case["path"] == "fused",
                            phi0=np.zeros(Grid((case["n"],) * 3).shape))
        _on_torch_stream(run.solver.lib)
        run.solver.fill_ghosts(inp["phi"])
        s["run"] = run
        return s
    grid = _grid(case)
    s["grid"], s["dt"] = grid, _dt(case, grid)
    if case["kind"] == "gradient":
        eng = NormalMotionAdjoint(grid, case["dtype"], case["steps"], dt=s["dt"], checkpoint_every=case["every"])
        _on_torch_stream(eng.solver.lib)
        s["engine"] = eng
        inp["phi0"].requires_grad_(True)
        inp["V"].requires_grad_(True)
        return s
    bc = "periodic" if case["kind"] == "motion" else BC[case["rhs"]]
    sol = Solver(grid, case["dtype"], bc=bc)
    _on_torch_stream(sol.lib)
    s["solver"] = sol
    sol.fill_ghosts(inp["phi"])
    s["work"] = (sol.field(), sol.field())
    s["out"] = sol.field()
    if case["kind"] == "motion":
        s["chain"] = DropInChain(sol)
        s["kappa"], s["gmag"] = sol.field(), sol.field()
        s["cg"] = [sol.field() for _ in range(3)]
    elif case["path"] == "chain":
        s["chain"] = DropInChain(sol)
        if case["rhs"] == "normal":
            s["vel"] = inp["V"]
    elif case["rhs"] == "deform":
        sol.deform_tables()
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(state):
    return {"step": _run_step, "motion": _run_motion, "band": _run_band, "gradient": _run_gradient,
            "plane": _run_plane}[state["case"]["kind"]](state)


def _run_step(s):
    """phi(n+1) from phi(n) by one TVD-RK3 step, ghosts filled; phi(n) is kept."""
    case, sol, dt, phi, (p1, p2), out = s["case"], s["solver"], s["dt"], s["inp"]["phi"], s["work"], s["out"]
    rhs = case["rhs"]
    if case["path"] == "fused":
        if rhs == "deform":
            stage, per = sol.stage_deform, [dict(c=c) for c in _factors(s["inp"]["t"], dt)]
        elif rhs == "velocity":
            stage, per = sol.stage_advect, [dict(vel=s["inp"]["vel"])] * 3
        elif rhs == "normal":
            stage, per = sol.stage_normal, [dict(vn_field=s["inp"]["V"])] * 3
        else:
            stage, per = sol.stage_reinit, [{}] * 3
        stage(p1, phi, None, 1, dt, **per[0])
        sol.fill_ghosts(p1)
        stage(p2, p1, phi, 2, dt, **per[1])
        sol.fill_ghosts(p2)
        stage(out, p2, phi, 3, dt, **per[2])
        sol.fill_ghosts(out)
        return out
    ch = s["chain"]
    if rhs == "reinit":
        f = ch.rhs_reinit
    elif rhs == "velocity":
        f = lambda u: ch.rhs_advect(u, vel=s["inp"]["vel"])  # noqa: E731
    else:
        f = lambda u: _rhs_normal_field(s, u)  # noqa: E731
    return _rk3_chain(s, f, dt)


def _rhs_normal_field(s, u):
    g, a, ch = s["grid"], s["solver"].lib.api, s["chain"]
    gb, fb, G6 = g.gb, g.fb, ch.grads
    a.lsm3dhjweno5(G6[0], G6[1], G6[2], gb, G6[3], G6[4], G6[5], gb, u, gb, ch.d1, gb, fb, *g.dx)
    a.lsm3dzerooutlevelseteqnrhs(ch.rhs, gb)
    a.lsm3daddnormalveltermtolserhs(ch.rhs, gb, G6[0], G6[1], G6[2], gb, G6[3], G6[4], G6[5], gb, s["vel"], gb, fb)


def _rk3_chain(s, f, dt):
    g, sol, ch, a = s["grid"], s["solver"], s["chain"], s["solver"].lib.api
    phi, (p1, p2), out = s["inp"]["phi"], s["work"], s["out"]
    gb, fb = g.gb, g.fb
    f(phi)
    a.lsm3dtvdrk3stage1(p1, gb, phi, gb, ch.rhs, gb, fb, dt)
    sol.fill_ghosts(p1)
    f(p1)
    a.lsm3dtvdrk3stage2(p2, gb, p1, gb, phi, gb, ch.rhs, gb, fb, dt)
    sol.fill_ghosts(p2)
    f(p2)
    a.lsm3dtvdrk3stage3(out, gb, p2, gb, phi, gb, ch.rhs, gb, fb, dt)
    sol.fill_ghosts(out)
    return out


CURV = 0.02  # V = 1 - CURV * curvature


def _run_motion(s):
    g, ch, a, C = s["grid"], s["chain"], s["solver"].lib.api, s["cg"]
    gb, fb, G6, vel, kap, gm = g.gb, g.fb, ch.grads, s["inp"]["vel"], s["kappa"], s["gmag"]

    def weno(u):
        a.lsm3dhjweno5(G6[0], G6[1], G6[2], gb, G6[3], G6[4], G6[5], gb, u, gb, ch.d1, gb, fb, *g.dx)

    def rhs(u):
        a.lsm3dcentralgradorder2(C[0], C[1], C[2], gb, u, gb, fb, *g.dx)
        a.lsm3dgradientmagnitude(C[0], C[1], C[2], gm, gb, fb)
        a.lsm3dcomputemeancurvatureorder2(kap, gb, u, gb, C[0], C[1], C[2], gm, gb, fb, *g.dx)
        ch.rhs_advect(u, vel=vel)
        weno(u)
        a.lsm3daddconstnormalveltermtolserhs(ch.rhs, gb, G6[0], G6[1], G6[2], gb, G6[3], G6[4], G6[5], gb, 1.0, fb)
        a.lsm3daddconstprecomputedcurvtermtolserhs(ch.rhs, gb, kap, gb, gm, gb, CURV, fb)

    dt_adv = a.lsm3dcomputestableadvectiondt(None, vel[0], vel[1], vel[2], gb, fb, *g.dx, CFL)
    weno(s["inp"]["phi"])
    dt_n = a.lsm3dcomputestableconstnormalveldt(None, 1.0, G6[0], G6[1], G6[2], gb, G6[3], G6[4], G6[5], gb, fb,
                                                *g.dx, CFL)
    dt = curvature_corrected_dt(min(dt_adv, dt_n), g, CURV, CFL)
    return {"phi": _rk3_chain(s, rhs, dt), "dt": dt}


def _run_band(s):
    r = s["run"]
    r.phi.copy_(s["inp"]["phi"])  # a run starts from the field it is given
    r.nsteps, r.dts, r.band_sizes = 0, [], []
    for _ in range(BAND_STEPS):
        r.step()
    # the lists' lengths follow the field; their first part is one of every band (the marks hold all of its points)
    first = 16 * s["case"]["n"] ** 2
    return {"phi": r.phi, "dt": list(r.dts), "marks": r.nb, "index": [a[:first] for a in (r.ix, r.iy, r.iz)],
            "levels": [int(v) for v in r.n_lo] + [int(v) for v in r.n_hi]}


def _run_gradient(s):
    Evolve, Mismatch = autograd_functions()
    inp, eng, eps = s["inp"], s["engine"], 1.5 * s["grid"].dx[0]
    loss = Mismatch.apply(Evolve.apply(inp["phi0"], inp["V"], eng), inp["target"], eng.solver, eps)
    gphi, gv = torch.autograd.grad(loss, (inp["phi0"], inp["V"]))
    return {"loss": loss.detach(), "phi0": gphi, "V": gv}


def _plane_boxes(case):
    nx, ny = case["nx"], case["ny"]
    return (-G, nx - 1 + G, -G, ny - 1 + G), (0, nx - 1, 0, ny - 1), (2.0 / nx, 2.0 / ny)


def _fill_plane(s, u):
    gb, fb, _ = _plane_boxes(s["case"])
    for face in range(4):
        s["api"].lsm2dsignedlinearextrapolation(u, gb, fb, face)


def _run_plane(s):
    a, phi = s["api"], s["inp"]["phi"]
    xp, yp, xm, ym, rhs, d1, p1, p2, out = s["buf"]
    gb, fb, h = _plane_boxes(s["case"])
    dt = CFL * min(h)

    def f(u):
        a.lsm2dhjweno5(xp, yp, gb, xm, ym, gb, u, gb, d1, gb, fb, *h)
        a.lsm2dcomputereinitializationeqnrhs(rhs, gb, u, gb, u, gb, xp, yp, gb, xm, ym, gb, fb, *h, 0)

    f(phi)
    a.lsm2dtvdrk3stage1(p1, gb, phi, gb, rhs, gb, fb, dt)
    _fill_plane(s, p1)
    f(p1)
    a.lsm2dtvdrk3stage2(p2, gb, p1, gb, phi, gb, rhs, gb, fb, dt)
    _fill_plane(s, p2)
    f(p2)
    a.lsm2dtvdrk3stage3(out, gb, p2, gb, phi, gb, rhs, gb, fb, dt)
    _fill_plane(s, out)
    return out


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
WENO = 73  # operations of one HJ-WENO5 reconstruction


def work(case):
    """Bytes: each array argument of each call read or written once.  Operations: the reconstructions and what
    combines them."""
    b = 8 if case["dtype"] == "f64" else 4
    if case["kind"] == "plane":
        cells = case["nx"] * case["ny"]
        return {"bytes": 3 * cells * b * (5 + 6) + cells * b * 8, "flops": 3 * cells * (4 * WENO + 30)}
    if case["kind"] == "band":
        cells, level0 = case["n"] ** 3, 38 * case["n"] ** 2
        build = cells * (b + 1) + 12 * 2 * level0
        stage = level0 * (13 + 3 * b)
        if case["path"] == "chain":
            stage = level0 * (8 * 13 + (7 + 1 + 8 + 3 + 4) * b)
        return {"bytes": build + BAND_STEPS * (3 * stage + level0 * (13 + 7 * b)),
                "flops": BAND_STEPS * 3 * level0 * (6 * WENO + 30)}
    cells = case["nx"] * case["ny"] * case["nz"]
    if case["kind"] == "gradient":
        # a stage reads phi and the speed (and phi at the start of the step) and writes one field; its reverse reads
        # phi, the speed and the incoming gradient and updates three
        return {"bytes": case["steps"] * cells * b * ((3 + 4 + 4) + 3 * (3 + 2 * 3)),
                "flops": case["steps"] * 3 * cells * (6 * WENO + 6 * 3 * WENO)}
    if case["kind"] == "motion":
        stage = 4 + 4 + 6 + 7 + 1 + 8 + 7 + 8 + 4
        return {"bytes": cells * b * (3 * stage + 3 + 4 + 4 + 3 + 7 + 6), "flops": 3 * cells * (9 * WENO + 110)}
    sides = 6 if case["rhs"] in ("normal", "reinit") else 3
    flops = 3 * cells * (sides * WENO + 20)
    if case["path"] == "fused":
        extra = {"deform": 0, "reinit": 0, "normal": 1, "velocity": 3}[case["rhs"]]
        return {"bytes": cells * b * (2 + 3 + 3 + 3 * extra), "flops": flops}
    rhs = {"reinit": 7 + 8, "normal": 7 + 1 + 9, "velocity": 7 + 1 + 8}[case["rhs"]]
    return {"bytes": cells * b * (3 * rhs + 3 + 4 + 4), "flops": flops}


def tolerance(case):
    """About four times what another order of the same sums showed over these ranges: the 64-bit restatement below, and
    in single precision the library's second set of stage kernels and the chain against the fused stages.  A cell where
    the upwind side or a Godunov branch hangs on a rounding differs by more than the rest: "max"."""
    if case["kind"] == "gradient":  # measured 1.5e-13 / 2.5e-11 and 1.2e-4 / 1.6e-2
        return {"rel": 6e-13, "max": 1e-10} if case["dtype"] == "f64" else {"rel": 5e-4, "max": 6e-2}
    if case["dtype"] == "f64":  # measured 3.9e-16 / 1.1e-14
        return {"rel": 1.6e-15, "max": 5e-14, "differ": 0.0}
    return {"rel": 1e-6, "max": 4e-5, "differ": 0.0}  # measured 2.7e-7 / 9.8e-6


# ---------------------------------------------------------------------------
# The same in plain torch in 64 bits
# ---------------------------------------------------------------------------
def _weno5(v1, v2, v3, v4, v5):
    m = v1 * v1
    for v in (v2, v3, v4, v5):
        m = torch.maximum(m, v * v)
    eps = 1e-6 * m + 1e-36
    p1 = v1 / 3 - 7 * v2 / 6 + 11 * v3 / 6
    p2 = -v2 / 6 + 5 * v3 / 6 + v4 / 3
    p3 = v3 / 3 + 5 * v4 / 6 - v5 / 6
    s1 = 13 / 12 * (v1 - 2 * v2 + v3) ** 2 + 0.25 * (v1 - 4 * v2 + 3 * v3) ** 2
    s2 = 13 / 12 * (v2 - 2 * v3 + v4) ** 2 + 0.25 * (v2 - v4) ** 2
    s3 = 13 / 12 * (v3 - 2 * v4 + v5) ** 2 + 0.25 * (3 * v3 - 4 * v4 + v5) ** 2
    a1, a2, a3 = 0.1 / (s1 + eps) ** 2, 0.6 / (s2 + eps) ** 2, 0.3 / (s3 + eps) ** 2
    return (a1 * p1 + a2 * p2 + a3 * p3) / (a1 + a2 + a3)


def _shift(u, dim, s, n):
    """u at offset s along one axis of the ghosted array, the interior of the others."""
    for d in range(u.dim()):
        o = G + (s if d == dim else 0)
        u = u.narrow(d, o, n[d])
    return u


def _diffs(u, dim, h, n):
    f = [_shift(u, dim, s, n) for s in range(-3, 4)]
    return [(f[q + 1] - f[q]) / h for q in range(6)]  # D(-2) .. D(3)


def _sides(u, dim, h, n):
    d = _diffs(u, dim, h, n)
    return _weno5(d[5], d[4], d[3], d[2], d[1]), _weno5(d[0], d[1], d[2], d[3], d[4])


def _upwind(u, dim, h, n, v, tol):
    d = _diffs(u, dim, h, n)
    pos = v > 0
    w = _weno5(*(torch.where(pos, d[q], d[5 - q]) for q in range(5)))
    return torch.where(v.abs() < tol, torch.zeros_like(w), w)


def _inner(u):
    for d in range(u.dim()):
        u = u.narrow(d, G, u.shape[d] - 2 * G)
    return u


def _extend(core, kind):
    """The ghosted array around interior values: faces along x, then y, then z."""
    u = core
    for d in range(core.dim() - 1, -1, -1):
        m = u.shape[d]
        if kind == "periodic":
            u = torch.cat([u.narrow(d, m - G, G), u, u.narrow(d, 0, G)], d)
            continue
        shape = [1] * u.dim()
        shape[d] = G
        dist = torch.arange(1, G + 1, dtype=u.dtype, device=u.device).reshape(shape)
        ends = []
        for e, i in ((0, 1), (m - 1, m - 2)):
            pb, pin = u.narrow(d, e, 1), u.narrow(d, i, 1)
            slope = pb - pin if kind == "linear" else torch.where(pb < 0, -1.0, 1.0) * (pb - pin).abs()
            ends.append(pb + slope * dist)
        u = torch.cat([ends[0].flip(d), u, ends[1]], d)
    return u


def _godunov(pos, sides):
    g = 0.0
    for p, m in sides:
        up = torch.maximum(m.clamp(min=0) ** 2, p.clamp(max=0) ** 2)
        dn = torch.maximum(m.clamp(max=0) ** 2, p.clamp(min=0) ** 2)
        g = g + torch.where(pos, up, dn)
    return g


def _safe_sqrt(g):
    return torch.where(g > 0, torch.sqrt(torch.where(g > 0, g, torch.ones_like(g))), torch.zeros_like(g))


def _normal_rhs(u, V, h, n):
    return -V * _safe_sqrt(_godunov(V > 0, [_sides(u, d, h[d], n) for d in range(len(n))]))


def _reinit_rhs(u, h, n, tol, strict):
    s = _inner(u)
    n2 = 0.0
    for d in range(len(n)):
        p, m = _sides(u, d, h[d], n)
        up = torch.maximum((-p).clamp(min=0), m.clamp(min=0))
        dn = torch.maximum(p.clamp(min=0), (-m).clamp(min=0))
        n2 = n2 + torch.where(s > 0, up, dn) ** 2
    sgn = s / torch.sqrt(s * s + n2 * max(h) ** 2)
    r = sgn * (1 - torch.sqrt(n2))
    on = s.abs() > tol if strict else s.abs() >= tol
    return torch.where(on, r, torch.zeros_like(r))


def _rk3(u0, rhs, dt, kind):
    c0 = _inner(u0)
    u1 = _extend(c0 + dt * rhs(u0, 0), kind)
    u2 = _extend(0.75 * c0 + 0.25 * (_inner(u1) + dt * rhs(u1, 1)), kind)
    return _extend(c0 / 3 + 2 / 3 * (_inner(u2) + dt * rhs(u2, 2)), kind)


def exact(case, seed):
    inp = _inputs(case, seed)
    tol = 1e-11 if case["dtype"] == "f64" else 1e-5  # the zero tolerance of the library's two precisions
    if case["kind"] == "plane":
        h = (2.0 / case["ny"], 2.0 / case["nx"])
        n = (case["ny"], case["nx"])
        u = _extend(_inner(inp["phi"].double()), "signed_linear")
        return _rk3(u, lambda v, k: _reinit_rhs(v, h, n, tol, True), CFL * min(h), "signed_linear")
    if case["kind"] == "band":
        return _exact_band(case, inp["phi"].double())
    g = _grid(case)
    h, n = g.dx[::-1], g.n[::-1]  # (z, y, x), as the arrays
    dt = _dt(case, g)
    if case["kind"] == "gradient":
        return _exact_gradient(case, inp, g, h, n, dt)
    if case["kind"] == "motion":
        return _exact_motion(inp, g, h, n, tol)
    kind = BC[case["rhs"]]
    u = _extend(_inner(inp["phi"].double()), kind)
    if case["rhs"] == "reinit":
        return _rk3(u, lambda v, k: _reinit_rhs(v, h, n, tol, False), dt, kind)
    if case["rhs"] == "normal":
        V = _inner(inp["V"].double())
        return _rk3(u, lambda v, k: _normal_rhs(v, V, h, n), dt, kind)
    if case["rhs"] == "velocity":
        vels = [[_inner(v.double()) for v in inp["vel"]]] * 3
    else:
        x, y, z = (a.narrow(d, G, a.shape[d] - 2 * G) for a, d in zip(_axes(g), (2, 1, 0)))
        A = [torch.sin(math.pi * a) ** 2 for a in (x, y, z)]
        B = [torch.sin(2 * math.pi * a) for a in (x, y, z)]
        base = (2 * A[0] * B[1] * B[2], -B[0] * A[1] * B[2], -B[0] * B[1] * A[2])
        vels = [[c * v for v in base] for c in _factors(inp["t"], dt)]

    def advect(w, k):
        r = 0.0
        for d in range(3):
            v = vels[k][2 - d]
            r = r - v * _upwind(w, d, h[d], n, v, tol)
        return r

    return _rk3(u, advect, dt, kind)


def _exact_motion(inp, g, h, n, tol):
    u = _extend(_inner(inp["phi"].double()), "periodic")
    vel = [_inner(v.double()) for v in inp["vel"]]
    one = torch.ones(n, dtype=torch.float64, device=u.device)
    sides = [_sides(u, d, h[d], n) for d in range(3)]
    w = [torch.maximum(p.abs(), m.abs()) for p, m in sides]
    nrm = torch.sqrt(sum(a * a for a in w) + max(h) ** 2)
    dt_n = CFL / (float((sum(a / q for a, q in zip(w, h)) / nrm).max()) + 1e-36)
    dt_a = CFL / (float(sum(v.abs() / q for v, q in zip(vel, g.dx)).max()) + 1e-36)
    dt = curvature_corrected_dt(min(dt_a, dt_n), g, CURV, CFL)

    def rhs(v, k):
        r = 0.0
        for d in range(3):
            r = r - vel[2 - d] * _upwind(v, d, h[d], n, vel[2 - d], tol)
        r = r + _normal_rhs(v, one, h, n)

        def at(o):  # v at offset o = (dz, dy, dx)
            w = v
            for d in range(3):
                w = w.narrow(d, G + o[d], n[d])
            return w

        def e(d, s=1):
            return tuple(s if q == d else 0 for q in range(3))

        c = at((0, 0, 0))
        D = [(at(e(d)) - at(e(d, -1))) / (2 * h[d]) for d in range(3)]
        H = {}
        for a in range(3):
            H[a, a] = (at(e(a)) - 2 * c + at(e(a, -1))) / h[a] ** 2
            for b in range(a):
                o = [tuple(p if q == a else m if q == b else 0 for q in range(3)) for p in (1, -1) for m in (1, -1)]
                H[a, b] = H[b, a] = (at(o[0]) - at(o[1]) - at(o[2]) + at(o[3])) / (4 * h[a] * h[b])
        q2 = [torch.where(t * t < 1e-8, torch.zeros_like(t), t * t) for t in D]
        gm = torch.sqrt(sum(q2))
        gm = torch.where(gm < 1e-8, torch.zeros_like(gm), gm)
        num = 0.0
        for a in range(3):
            for b in range(3):
                if a != b:
                    num = num + H[a, a] * D[b] ** 2 - H[a, b] * D[a] * D[b]
        den = gm ** 3
        kap = torch.where(den < tol, torch.zeros_like(den), num / torch.where(den < tol, torch.ones_like(den), den))
        return r + CURV * kap * gm

    return {"phi": _rk3(u, rhs, dt, "periodic"), "dt": dt}


def _exact_band(case, phi):
    """Motion with speed 1 of the points |phi| < 6 dx of the field the band was built from, the rest frozen, the
    speed cut off smoothly between 3 dx and 6 dx."""
    n, h = case["n"], 1.0 / case["n"]
    beta, gamma = 3 * h, 6 * h
    phi = _extend(_inner(phi), "signed_linear")
    N = n + 2 * G
    inside = torch.zeros_like(phi, dtype=torch.bool)
    inside[G:-G, G:-G, G:-G] = _inner(phi).abs() < gamma
    at = inside.reshape(-1).nonzero()[:, 0]
    del inside
    strides = (N * N, N, 1)
    last = [(at // st) % N == N - 1 - G for st in strides]  # the last interior cell along each axis

    def sides(u):
        u, out = u.reshape(-1), []
        for st, end in zip(strides, last):
            f = [u[at + s * st] for s in range(-3, 4)]
            d = [(f[q + 1] - f[q]) for q in range(6)]
            # the difference over the last ghost cell is outside the layer where first differences are formed
            d[5] = torch.where(end, torch.full_like(d[5], 1e10), d[5])
            d = [q / h for q in d]
            out.append((_weno5(d[5], d[4], d[3], d[2], d[1]), _weno5(d[0], d[1], d[2], d[3], d[4])))
        return out

    def rhs(u, sd):
        r = -torch.sqrt(_godunov(torch.ones_like(sd[0][0], dtype=torch.bool), sd))
        a = u.reshape(-1)[at].abs()
        cut = (a - gamma) ** 2 * (2 * a + gamma - 3 * beta) / (gamma - beta) ** 3
        cut = torch.where(a <= beta, torch.ones_like(a), torch.where(a <= gamma, cut, torch.zeros_like(a)))
        return cut * r

    dts = []
    for _ in range(BAND_STEPS):
        sd = sides(phi)
        w = [torch.maximum(p.abs(), m.abs()) for p, m in sd]
        dt = CFL / (float((sum(w) / h / torch.sqrt(sum(a * a for a in w) + h * h)).max()) + 1e-36)
        dts.append(dt)
        c0 = phi.reshape(-1)[at]
        u = phi
        for k in range(3):
            r = rhs(u, sd if k == 0 else sides(u))
            uc = u.reshape(-1)[at]
            v = (c0 + dt * r, 0.75 * c0 + 0.25 * (uc + dt * r), c0 / 3 + 2 / 3 * (uc + dt * r))[k]
            nxt = phi.clone()
            nxt.reshape(-1)[at] = v
            u = _extend(_inner(nxt), "signed_linear")
        phi = u
    return {"phi": phi, "dt": dts, "marks": None, "index": [None] * 3, "levels": [None] * 8}


def _exact_gradient(case, inp, g, h, n, dt):
    eps, dV = 1.5 * g.dx[0], g.dx[0] * g.dx[1] * g.dx[2]

    def H(v):
        mid = 0.5 * (1 + v / eps + torch.sin(math.pi * v / eps) / math.pi)
        return torch.where(v < -eps, torch.zeros_like(v), torch.where(v > eps, torch.ones_like(v), mid))

    V = _inner(inp["V"])
    c = _inner(inp["phi0"])
    weights = ((0.0, 1.0), (0.75, 0.25), (1 / 3, 2 / 3))

    def stage(u, start, V, k):
        a, b = weights[k]
        return a * start + b * (u + dt * _normal_rhs(_extend(u, "periodic"), V, h, n))

    kept = []
    for _ in range(case["steps"]):
        start, u = c, c
        for k in range(3):
            kept.append((u, start))
            u = stage(u, start, V, k)
        c = u
    c = c.detach().requires_grad_(True)
    loss = ((H(c) - H(_inner(inp["target"].double()))) ** 2).sum() * dV
    lam, = torch.autograd.grad(loss, c)
    lam_v, carry = torch.zeros_like(V), torch.zeros_like(c)
    for q in range(len(kept) - 1, -1, -1):
        k = q % 3
        u, start, Vk = (t.detach().requires_grad_(True) for t in (kept[q][0], kept[q][1], V))
        du, ds, dv = torch.autograd.grad(stage(u, start, Vk, k), (u, start, Vk), lam)
        lam_v += dv
        carry = carry + ds
        lam = du
        if k == 0:
            lam, carry = lam + carry, torch.zeros_like(c)

    def ghosted(t):
        return torch.nn.functional.pad(t, (G,) * 6)

    return {"loss": loss.detach(), "phi0": ghosted(lam), "V": ghosted(lam_v)}
