"""The multires operator by cell rows (pf_mr_row.hip) where its layout can go wrong: leaf
cells clipped by a ragged domain, blocks of every level next to every other, a refined box
at a corner, one refined block, no refinement at all; many slots of blocks to a wave; and
leaves that no row can hold.

Bars: both fast solves (Jacobi PCG and multigrid), to a max residual of 1e-11, against the
exact FP64 solution of the oracle's rows: those of the three-level tests, pressure within
1e-6 and faces within 1e-5 norm-wise relative.
"""
import numpy as np
import pytest

import pfflip_amd as G
import pyoracle as O
from _helpers import rel_err
from test_multires3_oracle import _system, exact_solution

pytestmark = pytest.mark.gpu


def _phase():
    ph = O.Phase(1.0, 0.01, 1.0, 1.0)
    ph.rho_tilde_0 = O.calibrate_rho_tilde0(ph, 1.0)
    return ph, G.Phase(ph.rho_l, ph.rho_g, ph.alpha_phi, ph.rho_tilde_0)


def _particles(dims, seed=4):
    """8 jittered particles per cell below 0.6 of the height, a gas ball in them"""
    nx, ny, nz = dims
    k, j, i = np.meshgrid(np.arange(1, nz - 1), np.arange(1, max(2, int(0.6 * ny))), np.arange(1, nx - 1), indexing="ij")
    c = np.repeat(np.stack([i.ravel(), j.ravel(), k.ravel()], 1), 8, axis=0)
    r = np.random.default_rng(seed)
    p = (c + r.uniform(0.01, 0.99, c.shape)).astype(np.float32)
    v = r.normal(scale=0.3, size=p.shape).astype(np.float32)
    t = (((p - np.array([nx / 2, ny * 0.25, nz / 2])) ** 2).sum(1) < (0.15 * nx) ** 2).astype(np.uint8)
    return tuple(np.ascontiguousarray(q) for q in (*p.T, *v.T)) + (t,)


def _to_projection(ctx, gph, dt):
    ctx.mr_mark_cells()
    ctx.mr_p2g(gph, 1.0)
    ctx.apply_gravity(dt, -9.81)
    ctx.apply_walls()


def _against_exact(dims, leaves, modes):
    dt = 0.02
    ph, gph = _phase()
    parts = _particles(dims)
    ctx = G.MRContext(*dims, 1.0)
    ctx.set_layout(leaves)
    ctx.upload(*parts)
    g = O.MRGrid(*dims, 1.0, faithful=False)
    g.set_leaves(leaves)
    ps = O.Particles(*parts[:6], type=parts[6])
    g.mark_cells(ps)
    g.p2g(ps, ph, 1.0)
    g.apply_gravity(dt, -9.81)
    g.apply_walls()
    cells, A, rhs, pin, vol = _system(g, ph, dt)
    g.apply_pressure(ph, dt, exact_solution(A, rhs, vol))
    for mode in modes:
        _to_projection(ctx, gph, dt)
        st = ctx.mr_project(gph, dt, G.mr_solve_cfg(20000, 1e-11, 0.0, mode=mode))
        assert st.converged == 1 and st.true_max_residual < 1e-11 and st.fallback_used == 0
        assert st.fluid_cells == len(cells) and st.pinned_cell == pin
        assert rel_err(ctx.field(G.FIELD_P), g.dense(O.P)) < 1e-6
        for f in range(3):
            assert rel_err(ctx.field(f), g.dense(f)) < 1e-5, f


@pytest.mark.parametrize("dims,level,boxes", [
    ((17, 10, 9), 1, ([4, 3, 2, 13, 9, 8],)), ((24, 20, 28), 1, ([0, 0, 0, 9, 9, 9],)),
    ((21, 19, 30), 1, ([8, 4, 8, 12, 8, 12],)), ((33, 18, 20), 1, ()), ((26, 25, 23), 1, ([0, 9, 0, 26, 20, 23],)),
    ((40, 36, 24), 2, ([0, 14, 0, 40, 24, 24], [16, 0, 8, 24, 12, 16])),
    ((37, 30, 33), 2, ([10, 12, 10, 20, 30, 20],) * 2)])
def test_fast_solves_match_the_exact_solution(dims, level, boxes):
    print(f"[mr rows] {dims} {level} {boxes}", flush=True)
    leaves = G.mr_layout_fine_box(*dims, level=level)
    for b in boxes:
        leaves = G.mr_layout_refine(*dims, leaves, b)
    _against_exact(dims, leaves, (G.MR_SOLVE_FAST, G.MR_SOLVE_MULTIGRID))


def test_level_3_leaves_of_air_alone():
    """level-3 leaves above the water, beside blocks of levels 2, 1 and 0 that hold it"""
    dims = (40, 104, 36)
    leaves = G.mr_layout_fine_box(*dims, level=3)
    for b in ([0, 0, 0, 40, 62, 36], [0, 40, 0, 18, 62, 36], [0, 52, 0, 10, 62, 20]):
        leaves = G.mr_layout_refine(*dims, leaves, b)
    top = [int(lv[2]) * (4 << int(lv[0])) for lv in leaves if lv[0] == 3]
    assert sorted(set(leaves[:, 0])) == [0, 1, 2, 3] and min(top) == 64  # (the water reaches into y = 60..64)
    _against_exact(dims, leaves, (G.MR_SOLVE_FAST,))


def test_fluid_above_level_2_is_refused_and_the_context_stays_usable():
    dims, dt = (64, 64, 64), 0.02
    _, gph = _phase()
    ctx = G.MRContext(*dims, 1.0)
    ctx.set_layout(G.mr_layout_fine_box(*dims, level=3))
    ctx.upload(*_particles(dims))
    for mode in (G.MR_SOLVE_FAST, G.MR_SOLVE_MULTIGRID):
        _to_projection(ctx, gph, dt)
        with pytest.raises(G.PfError):
            ctx.mr_project(gph, dt, G.mr_solve_cfg(2000, 1e-9, 0.0, mode=mode))
    ctx.set_layout(G.mr_layout_fine_box(*dims, level=2))
    _to_projection(ctx, gph, dt)
    st = ctx.mr_project(gph, dt, G.mr_solve_cfg(20000, 1e-9, 0.0))
    assert st.converged == 1 and np.isfinite(ctx.field(G.FIELD_P)).all()


def test_a_refused_solve_leaves_nothing_to_the_next():
    """water everywhere on level 3 (refused once its rows are assembled), then at high x only
    on level 1: its lowest blocks read couplings of blocks that only the first system listed"""
    dims, dt = (64, 64, 64), 0.02
    _, gph = _phase()
    parts = _particles(dims)
    some = tuple(np.ascontiguousarray(q[parts[0] > 33]) for q in parts)
    out = []
    for refused in (True, False):
        ctx = G.MRContext(*dims, 1.0)
        if refused:
            ctx.set_layout(G.mr_layout_fine_box(*dims, level=3))
            ctx.upload(*parts)
            _to_projection(ctx, gph, dt)
            with pytest.raises(G.PfError):
                ctx.mr_project(gph, dt, G.mr_solve_cfg(2000, 1e-9, 0.0))
        ctx.set_layout(G.mr_layout_fine_box(*dims, level=1))
        ctx.upload(*some)
        _to_projection(ctx, gph, dt)
        st = ctx.mr_project(gph, dt, G.mr_solve_cfg(20000, 1e-9, 0.0))
        assert st.converged == 1
        out.append((st.iterations, ctx.field(G.FIELD_P)))
    assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("dims,top,boxes,most", [
    ((68, 72, 62), 54, ([16, 16, 16, 48, 40, 32], [24, 24, 16, 40, 40, 32]), 4096),
    ((212, 232, 206), 214, ([48, 48, 48, 112, 96, 80], [64, 64, 48, 80, 80, 64]), 1 << 20)])
def test_leaf_cells_balance(dims, top, boxes, most):
    """What flows out of each leaf cell of three levels, summed from the faces, is zero to their
    rounding (up to 96 faces, half an ulp each) and its volume times the residual, and the two fast solves
    agree.  The second grid lists 135,000 blocks: waves take up to nine slots of four blocks
    in the iterations and two in the cycle, the last ones ragged."""
    dt, tol = 0.02, 1e-9
    nx, ny, nz = dims
    _, gph = _phase()
    leaves = G.mr_layout_fine_box(*dims, level=2)
    for b in boxes:
        leaves = G.mr_layout_refine(*dims, leaves, b)
    assert sorted(set(leaves[:, 0])) == [0, 1, 2]
    level = np.zeros(dims[::-1], np.int8)
    for L, bx, by, bz in leaves.tolist():
        s = 4 << L
        level[bz * s:(bz + 1) * s, by * s:(by + 1) * s, bx * s:(bx + 1) * s] = L
    # a particle in every cell of 2^3 below the top, and in every fine cell of the finest box
    f = boxes[1]
    grids = [np.meshgrid(np.arange(1, nz - 1, 2), np.arange(1, top, 2), np.arange(1, nx - 1, 2), indexing="ij"),
             np.meshgrid(*(np.arange(f[a], f[a + 3]) for a in (2, 1, 0)), indexing="ij")]
    p = np.concatenate([np.stack([g[2].ravel(), g[1].ravel(), g[0].ravel()], 1) for g in grids]) + 0.5
    r = np.random.default_rng(6)
    v = r.normal(scale=0.3, size=p.shape)
    t = (r.random(len(p)) < 0.2).astype(np.uint8)
    ctx = G.MRContext(*dims, 1.0)
    ctx.set_layout(leaves)
    ctx.upload(*(np.ascontiguousarray(q, np.float32) for q in (*p.T, *v.T)), t)
    got = []
    for mode in (G.MR_SOLVE_FAST, G.MR_SOLVE_MULTIGRID):
        _to_projection(ctx, gph, dt)
        st = ctx.mr_project(gph, dt, G.mr_solve_cfg(20000, tol, 0.0, mode=mode))
        assert st.converged == 1 and st.true_max_residual < tol and st.fallback_used == 0
        faces = [np.asarray(ctx.field(f), np.float64).reshape(ctx.dims(f)[::-1]) for f in range(3)]
        got.append((np.asarray(ctx.field(G.FIELD_P)), *faces))
        fluid = np.asarray(ctx.field(G.FIELD_MARKER)).reshape(nz, ny, nx) == 1  # FLUID
        listed = fluid[::4, ::4, ::4].sum()  # (a block's first cell is FLUID if one is)
        assert listed > 131072 if most > 131072 else listed < most
        out = sum(np.diff(a, axis=2 - f) for f, a in enumerate(faces))
        ulp = 2.0 ** -24 * max(np.abs(a).max() for a in faces)
        for L in range(3):
            s = 1 << L
            # (away from the walls, whose faces the rows leave out)
            z, y, x = (slice(8, (n - 12) // 4 * 4) for n in dims[::-1])
            a = out[z, y, x]
            a = a.reshape(a.shape[0] // s, s, a.shape[1] // s, s, a.shape[2] // s, s).sum(axis=(1, 3, 5))
            here = (level[z, y, x] == L)[::s, ::s, ::s] & fluid[z, y, x][::s, ::s, ::s]
            assert here.sum() > 1000 and np.abs(a[here]).max() < 6 * 4 ** L * ulp + 8 ** L * tol, L
    assert rel_err(got[0][0], got[1][0]) < 1e-6
    for f in range(1, 4):
        assert rel_err(got[0][f], got[1][f]) < 1e-5, f
