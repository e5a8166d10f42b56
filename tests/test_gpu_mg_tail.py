"""The multigrid cycle's small levels in one workgroup (k_mg_tail): grids whose first tail
level is the coarsest, has one block, has exactly 64 blocks or just more (the level above
keeps the row kernels), ragged and elongated hierarchies, and every sweep count the tail
takes (one sweep keeps the separate kernels).

Bar: the projection to a relative FP64 residual of 1e-10 agrees with the Jacobi solve of
the same open tank in far fewer iterations, without the fallback that a wrong cycle ends
in.  The velocities' bound: the pressure is stored in FP32, so each of the two pressures of
a face is off by up to 2^-24 max|p| in either solve, which the face update multiplies by
(dt / dx) beta, at most (dt / dx) / rho_g: 4 (dt / dx) / rho_g 2^-24 max|p| on a face.
"""
import numpy as np
import pytest

import pfflip_amd as G
import pyoracle as O
from _helpers import phase, scene

pytestmark = pytest.mark.gpu


def _solve(shape, pre, sweeps=None):
    nx, ny, nz = shape
    dx, x, y, z, t = scene(O.SCENE_BUBBLE, nx, seed=3, ny=ny, nz=nz)
    rng = np.random.default_rng(3)
    u, v, w = (rng.normal(scale=0.3, size=len(x)).astype(np.float32) for _ in range(3))
    ctx = G.Context(nx, ny, nz, dx)
    ctx.upload(x, y, z, u, v, w, t)
    oph = phase()
    gph = G.Phase(oph.rho_l, oph.rho_g, oph.alpha_phi, oph.rho_tilde_0)
    if sweeps:
        ctx.set_multigrid(sweeps=sweeps)
    ctx.mark_cells()
    ctx.p2g(gph, 1.0)
    ctx.apply_gravity(1e-3, -9.81)
    ctx.apply_walls()
    st = ctx.project(gph, 1e-3, G.default_solve_cfg(G.STOP_REL2, 1e-10, 20000, pre))
    p = ctx.field(G.FIELD_P)
    return st, [ctx.field(f) for f in range(3)], 4 * (1e-3 / dx) / oph.rho_g * 2.0 ** -24 * np.abs(p).max()


@pytest.mark.parametrize("shape", [(8, 8, 8), (9, 7, 8), (16, 15, 17), (32, 33, 30), (36, 20, 12), (66, 64, 34),
                                   (96, 24, 20), (70, 66, 36)])
def test_cycle_with_the_tail(shape):
    print(f"[tail] {shape}", flush=True)
    mg, f_mg, bound = _solve(shape, G.PRECOND_MULTIGRID)
    ja, f_ja, _ = _solve(shape, G.PRECOND_JACOBI)
    assert mg.converged == 1 and ja.converged == 1 and mg.fallback_used == 0
    assert mg.iterations < ja.iterations
    for a, b in zip(f_mg, f_ja):
        assert np.abs(a - b).max() < bound


@pytest.mark.parametrize("sweeps", [1, 2, 3, 5, 16])
def test_sweep_counts(sweeps):
    print(f"[tail] sweeps {sweeps}", flush=True)
    mg, f_mg, bound = _solve((40, 36, 28), G.PRECOND_MULTIGRID, sweeps)
    ja, f_ja, _ = _solve((40, 36, 28), G.PRECOND_JACOBI)
    assert mg.converged == 1 and mg.fallback_used == 0 and mg.iterations * 2 < ja.iterations
    for a, b in zip(f_mg, f_ja):
        assert np.abs(a - b).max() < bound
