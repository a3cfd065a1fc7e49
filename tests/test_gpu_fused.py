"""Fused WENO5 + RHS + RK stage kernels against the drop-in chain (GPU) and
the oracle chain (CPU).  FP64: bitwise.  FP32: error bounds against FP64."""
import numpy as np
import pytest

import harness as H

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def solvers():
    from lsmlib_amd.solver import Grid, Solver
    g = Grid((22, 19, 17), lo=(0, 0, 0), hi=(1.1, 0.95, 0.85))
    return g, Solver(g, "f64", bc="signed_linear"), Solver(g, "f32", bc="signed_linear")


def _phi(g, seed=3):
    from lsmlib_amd.solver import phi_spheres_min
    phi, _ = phi_spheres_min(g, seed, 4, (0.2, 0.8), (0.1, 0.25))
    rng = np.random.default_rng(seed)
    return phi + 0.02 * rng.standard_normal(phi.shape)  # rough enough to switch WENO weights


def _oracle_stage(g, phi_np, phin_np, stage, dt, kind, vel=None, vn=0.8, phi0=None):
    """Oracle drop-in chain for one stage on host arrays."""
    o = H.oracle()
    gb, fb = g.gb, g.fb
    G = [np.zeros(g.shape) for _ in range(6)]
    d1, rhs, out = np.zeros(g.shape), np.zeros(g.shape), np.zeros(g.shape)
    if kind == "advect":
        o.lsm3dupwindhjweno5(G[0], G[1], G[2], gb, phi_np, gb, vel[0], vel[1], vel[2], gb, d1, gb, fb, *g.dx)
        o.lsm3dzerooutlevelseteqnrhs(rhs, gb)
        o.lsm3daddadvectiontermtolserhs(rhs, gb, G[0], G[1], G[2], gb, vel[0], vel[1], vel[2], gb, fb)
    else:
        o.lsm3dhjweno5(G[0], G[1], G[2], gb, G[3], G[4], G[5], gb, phi_np, gb, d1, gb, fb, *g.dx)
        if kind == "normal":
            o.lsm3dzerooutlevelseteqnrhs(rhs, gb)
            o.lsm3daddconstnormalveltermtolserhs(rhs, gb, G[0], G[1], G[2], gb, G[3], G[4], G[5], gb, vn, fb)
        else:
            o.lsm3dcomputereinitializationeqnrhs(rhs, gb, phi_np, gb, phi0 if phi0 is not None else phi_np, gb,
                                                 G[0], G[1], G[2], gb, G[3], G[4], G[5], gb, fb, *g.dx,
                                                 1 if phi0 is not None else 0)
    out[...] = 0.0
    if stage == 1:
        o.lsm3dtvdrk3stage1(out, gb, phi_np, gb, rhs, gb, fb, dt)
    elif stage == 2:
        o.lsm3dtvdrk3stage2(out, gb, phi_np, gb, phin_np, gb, rhs, gb, fb, dt)
    else:
        o.lsm3dtvdrk3stage3(out, gb, phi_np, gb, phin_np, gb, rhs, gb, fb, dt)
    return out


@pytest.mark.parametrize("kind", ["normal", "reinit", "reinit_phi0", "advect"])
@pytest.mark.parametrize("stage", [1, 2, 3])
def test_fused_stage_fp64_bitwise_vs_oracle(solvers, kind, stage):
    g, s64, _ = solvers
    phi_np = _phi(g)
    phin_np = _phi(g, 5)
    dt = 0.3 * g.dx[0]
    us, uc = s64.field(phi_np), s64.field(phin_np)
    out = s64.field(np.zeros(g.shape))
    vel = phi0 = None
    if kind == "normal":
        s64.stage_normal(out, us, uc, stage, dt, vn=-0.8)
        ref = _oracle_stage(g, phi_np, phin_np, stage, dt, "normal", vn=-0.8)
    elif kind.startswith("reinit"):
        phi0 = s64.field(phin_np) if kind == "reinit_phi0" else None
        s64.stage_reinit(out, us, uc, stage, dt, phi0=phi0)
        ref = _oracle_stage(g, phi_np, phin_np, stage, dt, "reinit", phi0=phin_np if phi0 is not None else None)
    else:
        c = 0.7
        vel = s64.deform_velocity(c)  # the same device function the fused kernel evaluates
        s64.stage_deform(out, us, uc, stage, dt, c)
        ref = _oracle_stage(g, phi_np, phin_np, stage, dt, "advect", vel=[s64.host(v) for v in vel])
    got = s64.host(out)
    gi, ri = g.interior(got), g.interior(ref)
    bad = np.argwhere(gi != ri)
    assert len(bad) == 0, "differs at %d cells, first %s: %r vs %r" % (
        len(bad), bad[0].tolist(), gi[tuple(bad[0])], ri[tuple(bad[0])])


@pytest.mark.parametrize("kind", ["normal", "advect", "reinit"])
def test_fused_rk3_step_fp64_equals_dropin_chain(solvers, kind):
    from lsmlib_amd.solver import DropInChain
    g, s64, _ = solvers
    phi_np = _phi(g)
    a, b = s64.field(phi_np), s64.field(phi_np)
    s64.fill_ghosts(a)
    s64.fill_ghosts(b)
    wa = (s64.field(), s64.field())
    wb = (s64.field(), s64.field())
    chain = DropInChain(s64)
    dt = 0.4 * g.dx[0]
    for step in range(3):
        if kind == "normal":
            s64.rk3_fused(a, wa, s64.stage_normal, dt, vn=1.0)
            chain.rk3(b, wb, chain.rhs_normal, dt, vn=1.0)
        elif kind == "advect":
            c = np.cos(np.pi * step * dt / 3.0)
            vel = s64.deform_velocity(c)
            s64.rk3_fused(a, wa, s64.stage_deform, dt, c=c)
            chain.rk3(b, wb, chain.rhs_advect, dt, vel=vel)
        else:
            s64.rk3_fused(a, wa, s64.stage_reinit, dt)
            chain.rk3(b, wb, chain.rhs_reinit, dt)
    s64.lib.check()
    ha, hb = s64.host(a), s64.host(b)
    assert np.array_equal(ha, hb), np.abs(ha - hb).max()


@pytest.mark.parametrize("kernels", [1, 2])
@pytest.mark.parametrize("kind", ["normal", "advect", "reinit"])
def test_fused_fp32_close_to_fp64(solvers, kind, kernels):
    """Both FP32 kernel sets (1: a WENO5 window per cell, the default; 2: each
    position's terms shared between cells) within 2e-5 of FP64 after five
    steps."""
    import ctypes
    g, s64, s32 = solvers
    from lsmlib_amd.solver import phi_sphere
    phi_np = phi_sphere(g, (0.5, 0.45, 0.42), 0.3)
    if kind == "reinit":
        phi_np = 1.7 * phi_np  # |grad phi| = 1.7: the reinitialization RHS is O(1)
    select = s32.lib.fn("lsmhip_set_fused_f32_kernels", [ctypes.c_int])
    prev = select(kernels)
    res = []
    for s in (s64, s32):
        a = s.field(phi_np)
        s.fill_ghosts(a)
        w = (s.field(), s.field())
        for step in range(5):
            if kind == "normal":
                s.rk3_fused(a, w, s.stage_normal, 0.4 * g.dx[0], vn=1.0)
            elif kind == "reinit":
                s.rk3_fused(a, w, s.stage_reinit, 0.4 * g.dx[0])
            else:
                s.rk3_fused(a, w, s.stage_deform, 0.4 * g.dx[0], c=1.0)
        s.lib.check()
        res.append(g.interior(s.host(a)))
    assert select(prev) == kernels
    # FP32 storage and arithmetic: relative-to-O(1) errors of a few ulp per step
    assert np.abs(res[0] - res[1]).max() < 2e-5


# Tiles of 64 x 8 cells and chunks of planes: single cells, one cell past a tile, and grids that the chunk rule cuts
# into one plane, a few planes and its longest chunks (with a shorter last one).
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n", [(1, 1, 1), (3, 2, 5), (64, 8, 4), (65, 9, 7), (72, 17, 33), (130, 70, 101), (520, 270, 66)])
@pytest.mark.parametrize("kind", ["normal", "reinit", "advect"])
def test_stage_does_not_depend_on_the_chunks(prec, n, kind):
    """The chunks that the library takes from the grid's size against chunks of 64 planes: the same bits in FP64.  In
    FP32 the advection kernel's unrolled planes and its last ones may contract different products: each derivative,
    bounded by the largest difference, moves by some 50 roundings (a reconstruction's operations, its weights moving
    four times as much as their terms), dt |v| / dx <= 0.2 times that enters, over three axes."""
    import torch
    from lsmlib_amd.solver import Grid, Solver
    g = Grid(n, hi=tuple(0.05 * v for v in n))
    s = Solver(g, prec)
    gen = torch.Generator(device="cuda").manual_seed(7)
    us, uc = (torch.randn(g.shape, dtype=s.dtype, device="cuda", generator=gen) for _ in range(2))
    dt = 0.1 * g.dx[0]

    def run(stage):
        out = s.field()
        if kind == "normal":
            s.stage_normal(out, us, uc, stage, dt, vn=-0.8)
        elif kind == "reinit":
            s.stage_reinit(out, us, uc, stage, dt)
        else:
            s.stage_deform(out, us, uc, stage, dt, 0.7)
        return out

    chunk = s.lib.cdll.lsmhip_set_fused_kchunk
    for stage in (1, 2, 3):
        a = run(stage)
        chunk(64)
        try:
            b = run(stage)
        finally:
            chunk(0)
        assert torch.isfinite(a).all()
        if prec == "f64":
            assert torch.equal(a, b), "stage %d" % stage
        else:
            bound = 3 * 0.2 * 4 * 50 * 2.0 ** -24 * 2 * float(us.abs().max())
            assert float((a - b).abs().max()) <= bound, "stage %d" % stage


# Rows whose last tile holds 1, 8 and 9 cells (the waves that compute for lanes past the row's end), and speeds that
# change sign or vanish inside a wave (the waves that pick their side per lane).
@pytest.mark.parametrize("nx", [1, 8, 65, 72, 73])
@pytest.mark.parametrize("signs", ["minus", "plus", "mixed", "one lane", "zero"])
def test_fp64_advection_by_lane_is_bitwise_the_oracle(nx, signs):
    from lsmlib_amd.solver import Grid, Solver
    g = Grid((nx, 5, 4), hi=(0.1 * nx, 0.45, 0.4))
    s = Solver(g, "f64")
    rng = np.random.default_rng(nx)
    phi, phin = rng.standard_normal(g.shape), rng.standard_normal(g.shape)
    vel = [np.abs(rng.standard_normal(g.shape)) + 0.1 for _ in range(3)]
    if signs == "minus":
        vel = [-v for v in vel]
    elif signs == "mixed":
        vel = [np.where(rng.random(g.shape) < 0.4, -v, np.where(rng.random(g.shape) < 0.1, 0.0, v)) for v in vel]
    elif signs == "one lane":
        for v in vel:
            v[:, :, g.g + nx // 2] *= -1.0
            v[:, :, g.g] = 1e-12
    elif signs == "zero":
        vel = [v * 1e-13 for v in vel]
    ref = _oracle_stage(g, phi, phin, 2, 0.03, "advect", vel=vel)
    out = s.field()
    s.stage_advect(out, s.field(phi), s.field(phin), 2, 0.03, [s.field(v) for v in vel])
    s.lib.check()
    got = s.host(out)
    assert np.array_equal(g.interior(got), g.interior(ref))
    # the drop-in's upwinded derivatives on the same lanes
    gb, fb, G = g.gb, g.fb, [s.field() for _ in range(4)]
    o = [np.zeros(g.shape) for _ in range(4)]
    s.lib.api.lsm3dupwindhjweno5(G[0], G[1], G[2], gb, s.field(phi), gb, *[s.field(v) for v in vel], gb, G[3], gb, fb,
                                 *g.dx)
    H.oracle().lsm3dupwindhjweno5(o[0], o[1], o[2], gb, phi, gb, *vel, gb, o[3], gb, fb, *g.dx)
    for a, b in zip(G[:3], o[:3]):
        assert np.array_equal(g.interior(s.host(a)), g.interior(b))


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("pattern", ["zero waves", "one lane", "mixed"])
def test_fp32_advection_of_a_cell_does_not_depend_on_its_wave(axis, pattern):
    """Speeds along one axis that are positive, negative, below the zero tolerance (both signs) or exactly zero: waves
    without a speed, with one, and of every kind take different routes, and each cell has the value it has where all
    speeds are of its own kind: without a speed the same bits; with one, the routes may contract different products, and
    the derivative, bounded by the largest difference, moves by some 50 roundings (as above, four times for the
    weights), of which dt |v| / dx enters."""
    from lsmlib_amd.solver import Grid, Solver
    g = Grid((130, 17, 9), hi=(1.3, 0.17, 0.09))
    s = Solver(g, "f32")
    rng = np.random.default_rng(axis)
    phi, phin = (s.field(rng.standard_normal(g.shape)) for _ in range(2))
    size = np.abs(rng.standard_normal(g.shape)) + 0.1
    kind = rng.integers(-1, 2, g.shape)
    if pattern == "zero waves":
        kind[:, ::2, :] = 0
        kind[:, :, :g.g + 64] = 0
    elif pattern == "one lane":
        kind[...] = 0
        kind[:, :, g.g::64] = -1
        kind[:, :, g.g + 63::64] = 1
    tiny = np.where(rng.random(g.shape) < 0.5, rng.choice([-1e-16, 1e-16], g.shape), 0.0)

    def stage(speed):
        vel = [s.field() for _ in range(3)]
        vel[axis] = s.field(speed)
        out = s.field()
        s.stage_advect(out, phi, phin, 3, 0.003, vel)
        s.lib.check()
        return g.interior(s.host(out))

    got = stage(np.where(kind == 0, tiny, kind * size))
    inner = g.interior(kind)
    bound = 0.003 * size.max() / 0.01 * 4 * 50 * 2.0 ** -24 * 2 * float(phi.abs().max())
    assert bound < 1e-3
    for k in (-1, 0, 1):
        d = np.abs(got - stage(k * size))[inner == k]
        assert d.max() <= (bound if k else 0.0), k


# A few planes over 384 tiles and more: 2, 3 and 4 planes a chunk, in one and in several rounds of 512 blocks, and the
# sizes on either side of that rule.
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n", [(512, 384, 3), (449, 385, 4), (576, 512, 4), (512, 512, 6), (512, 384, 8), (512, 384, 9),
                               (448, 432, 4)])
def test_thin_grids_do_not_depend_on_the_chunks(prec, n):
    test_stage_does_not_depend_on_the_chunks(prec, n, "reinit")
    test_stage_does_not_depend_on_the_chunks(prec, n, "advect")
