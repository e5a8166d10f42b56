"""The Jacobi PCG iteration in one kernel (k_cg_iter) at the sizes where its layout can go
wrong: one block, ragged ends, one list slot more or less than a workgroup's share, the
change to the form that loads after the sums (more than 512 workgroups), several slots
to a wave (more than 1024), and the iteration budget at a restart.

Bars: the FP64 oracle's pressure where it is quick (1e-6, the bar of the other projection
tests), and on larger open tanks the multigrid solve of the same system to a residual of
1e-11.  There the velocities' bound is the FP32 storage of the pressure: each of the two
pressures of a face is off by up to 2^-24 max|p| in either solve, which the face update
multiplies by (dt / dx) beta, at most (dt / dx) / rho_g.
"""
import numpy as np
import pytest

import pfflip_amd as G
import pyoracle as O
from _helpers import phase, rel_err, scene

pytestmark = pytest.mark.gpu


def _context(shape, kind, seed=5):
    nx, ny, nz = shape
    dx, x, y, z, t = scene(kind, nx, seed=seed, ny=ny, nz=nz)
    rng = np.random.default_rng(seed)
    u, v, w = (rng.normal(scale=0.3, size=len(x)).astype(np.float32) for _ in range(3))
    ctx = G.Context(nx, ny, nz, dx)
    ctx.upload(x, y, z, u, v, w, t)
    oph = phase()
    return dx, ctx, O.Particles(x, y, z, u, v, w, t), oph, G.Phase(oph.rho_l, oph.rho_g, oph.alpha_phi, oph.rho_tilde_0)


def _grid_half(ctx, gph, dt=1e-3):
    ctx.mark_cells()
    ctx.p2g(gph, 1.0)
    ctx.save_velocity()
    ctx.apply_gravity(dt, -9.81)
    ctx.apply_walls()


@pytest.mark.parametrize("shape,kind", [((4, 4, 4), O.SCENE_RT), ((5, 3, 9), O.SCENE_RT), ((17, 18, 6), O.SCENE_RT),
                                        ((24, 25, 13), O.SCENE_BUBBLE), ((33, 12, 30), O.SCENE_DAMBREAK)])
def test_matches_the_oracle(shape, kind):
    print(f"[cg] {shape} {kind}", flush=True)
    dx, ctx, ps, oph, gph = _context(shape, kind)
    g = O.Grid(*shape, dx, faithful=False)
    g.mark_cells(ps)
    g.p2g(ps, oph, 1.0)
    g.apply_gravity(1e-3, -9.81)
    g.apply_walls()
    _grid_half(ctx, gph)
    st = ctx.project(gph, 1e-3, G.default_solve_cfg(G.STOP_REL2, 1e-9, 20000))
    ost = g.project(oph, 1e-3, 20000, 1e-12, 0.0, O.STOP_REL2)
    assert st.converged == 1 and st.breakdown == 0 and st.true_rel_residual <= 1e-9
    assert st.fluid_cells == ost.fluid_cells
    assert rel_err(ctx.field(G.FIELD_P), g.dense(O.P)) < 1e-6
    for f in range(3):
        assert rel_err(ctx.field(f), g.dense(f)) < 1e-5


def _workgroups(ctx):
    """of the iteration: sixteen listed blocks each, a multiple of 8, at most 1024"""
    m = np.asarray(ctx.field(G.FIELD_MARKER)) == 1  # FLUID
    m = np.pad(m.reshape(ctx.dims(G.FIELD_MARKER)[::-1]), [(0, -n % 4) for n in ctx.dims(G.FIELD_MARKER)[::-1]])
    z, y, x = (n // 4 for n in m.shape)
    listed = int(m.reshape(z, 4, y, 4, x, 4).any(axis=(1, 3, 5)).sum())
    return min(-(-listed // 128) * 8, 1024)


# up to 512 workgroups the row loads come before the sums, above after them; at the cap of
# 1024 (17,576 blocks) some waves take two slots; ragged grids on each side
@pytest.mark.parametrize("shape,groups", [((72, 72, 72), 224), ((84, 83, 82), 360), ((101, 35, 34), 88),
                                          ((80, 133, 80), 504), ((82, 130, 81), 528), ((105, 171, 103), 1024)])
def test_matches_multigrid_on_larger_grids(shape, groups):
    print(f"[cg] {shape}", flush=True)
    dx, ctx, _, _, gph = _context(shape, O.SCENE_BUBBLE)
    ctx.mark_cells()
    assert _workgroups(ctx) == groups
    faces = []
    for pre in (G.PRECOND_JACOBI, G.PRECOND_MULTIGRID):
        _grid_half(ctx, gph)
        st = ctx.project(gph, 1e-3, G.default_solve_cfg(G.STOP_REL2, 1e-11, 20000, pre))
        assert st.converged == 1 and st.true_rel_residual <= 1e-11 and st.fallback_used == 0
        faces.append([ctx.field(f) for f in range(3)])
    bound = 4 * (1e-3 / dx) / gph.rho_g * 2.0 ** -24 * np.abs(ctx.field(G.FIELD_P)).max()
    for a, b in zip(*faces):
        assert np.abs(a - b).max() < bound


def test_separate_kernels_match_multigrid():
    """85,184 listed blocks: the range in which the iteration takes the separate kernels"""
    n = 176
    gph = G.Phase(10.0, 1.0, 1.0, 1.0)  # (from rest: a lower pressure leaves a lower bound)
    gph.rho_tilde_0 = G.calibrate_rho_tilde0(gph, 1.0)
    ctx = G.Context(n, n, n, 1.0 / n)
    ctx.scene(G.SCENE_RT, 3)
    faces = []
    for pre in (G.PRECOND_JACOBI, G.PRECOND_MULTIGRID):
        _grid_half(ctx, gph)
        st = ctx.project(gph, 1e-3, G.default_solve_cfg(G.STOP_REL2, 1e-11, 20000, pre))
        assert st.converged == 1 and st.true_rel_residual <= 1e-11 and st.fallback_used == 0
        faces.append([ctx.field(f) for f in range(3)])
    bound = 4 * (1e-3 * n) / gph.rho_g * 2.0 ** -24 * np.abs(ctx.field(G.FIELD_P)).max()
    for a, b in zip(*faces):
        assert np.abs(a).max() > 100 * bound and np.abs(a - b).max() < bound


@pytest.mark.parametrize("budget", [1, 2, 60])
def test_stops_at_the_iteration_budget(budget):
    _, ctx, _, _, gph = _context((32, 20, 32), O.SCENE_RT)
    _grid_half(ctx, gph)
    cfg = G.default_solve_cfg(G.STOP_REL2, 1e-12, budget)
    st = ctx.project(gph, 1e-3, cfg)
    assert st.iterations == budget and st.converged == 0
    assert np.isfinite(ctx.field(G.FIELD_P)).all()
    # and the same context solves to the end afterwards, as a fresh one does
    _grid_half(ctx, gph)
    again = ctx.project(gph, 1e-3, G.default_solve_cfg(G.STOP_REL2, 1e-9, 20000))
    p = ctx.field(G.FIELD_P)
    _, fresh, _, _, _ = _context((32, 20, 32), O.SCENE_RT)
    _grid_half(fresh, gph)
    st = fresh.project(gph, 1e-3, G.default_solve_cfg(G.STOP_REL2, 1e-9, 20000))
    assert again.converged == 1 and again.iterations == st.iterations
    assert np.array_equal(p, fresh.field(G.FIELD_P))


def test_check_every_does_not_change_the_result():
    ps = []
    for every in (1, 7, 64):
        _, ctx, _, _, gph = _context((40, 30, 20), O.SCENE_RT)
        _grid_half(ctx, gph)
        cfg = G.default_solve_cfg(G.STOP_REL2, 1e-9, 20000)
        cfg.check_every = every
        st = ctx.project(gph, 1e-3, cfg)
        assert st.converged == 1
        ps.append((st.iterations, ctx.field(G.FIELD_P)))
    assert all(n == ps[0][0] and np.array_equal(p, ps[0][1]) for n, p in ps)
