"""The work that a program built on this framework has it do, as measurable cases.

A case names one path through the public entry points (include/pf_gpu.h and its Python
binding), with sizes and options:

  cfl        pf_timestep_noalloc on the caller's own device arrays
  splat      pf_mark_cells and pf_p2g: markers, face velocities and face masses
  project    the grid half of a step called stage by stage (mark, P2G, save, gravity,
             walls, projection): pressure and projected face velocities
  transport  the particle half called stage by stage (binning, G2P, advection) over
             some substeps in a given velocity field: the moved particles
  frame      whole time steps with the particles resident on the GPU, then the
             particle state taken to page-locked memory, as a program that writes
             every n-th step does; two-phase, single-phase, both multires solvers
  learned    one training gradient of the learned preconditioner

Scenes and options are those of the tests and the benchmark: 8 jittered particles per
cell, density ratios up to 1000:1, FLIP ratio 0.95, gravity -9.81.  Grids are ragged
and not powers of two as often as they are the benchmark's cubes.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "adaptive-pf-flip_amd"))

import pfflip_amd as G  # noqa: E402

DEVICE = "cuda"
GRAVITY = -9.81
AIR, FLUID, SOLID = 0, 1, 2
# network work per aggregate: three 3^3 convolutions of widths 4-16-32-16 and the head
LEARNED_FLOPS = 2 * (27 * (4 * 16 + 16 * 32 + 32 * 16) + 16)


def listed():
    return [
        # the smallest call: the CFL limit of a caller that keeps its own velocities
        {"name": "cfl_100k", "kind": "cfl", "n": 100003},
        # the splat alone on a ragged grid whose spacing is no power of two
        {"name": "splat_ragged", "kind": "splat", "scene": "rt", "nx": 144, "ny": 101, "nz": 131, "ratio": 1000.0},
        # the reference's Jacobi PCG on a small open tank, to a tight residual
        {"name": "project_jacobi_48", "kind": "project", "scene": "tank", "nx": 48, "ny": 45, "nz": 50,
         "ratio": 100.0, "solver": "jacobi"},
        # the multigrid projection at an ordinary size, closed box (pinned cell)
        {"name": "project_multigrid_160", "kind": "project", "scene": "rt", "nx": 161, "ny": 120, "nz": 143,
         "ratio": 1000.0, "solver": "multigrid"},
        # binning, G2P and RK2 advection alone
        {"name": "transport_128", "kind": "transport", "scene": "rt", "nx": 128, "ny": 128, "nz": 128,
         "substeps": 6},
        # the 64^3 Rayleigh-Taylor step as the reference solves it: Jacobi, |r|_inf < 1e-7
        {"name": "frame_rt64_reference", "kind": "frame", "model": "two_phase", "scene": "rt", "nx": 64, "ny": 64,
         "nz": 64, "solver": "reference", "steps": 2, "surface": False},
        # the 128^3 bubble tank with surface tension and the interface diagnostics
        {"name": "frame_bubble128", "kind": "frame", "model": "two_phase", "scene": "tank", "nx": 128, "ny": 128,
         "nz": 128, "solver": "multigrid", "steps": 4, "surface": True},
        # a single-phase dam break on a ragged grid
        {"name": "frame_dambreak_single", "kind": "frame", "model": "single_phase", "scene": "dam", "nx": 150,
         "ny": 90, "nz": 110, "solver": "reference", "steps": 4, "surface": False},
        # the headline: 256^3 Rayleigh-Taylor, multigrid to 1e-6 in FP64
        {"name": "frame_rt256", "kind": "frame", "model": "two_phase", "scene": "rt", "nx": 256, "ny": 256,
         "nz": 256, "solver": "multigrid", "steps": 8, "surface": False},
        # the two-level multires tank that refines around its bubble as it moves
        {"name": "frame_multires_refine", "kind": "frame", "model": "multires", "scene": "band", "nx": 80, "ny": 72,
         "nz": 80, "solver": "fast", "steps": 4, "surface": False},
        # the three-level multires tank of 16 bubbles with its multigrid
        {"name": "frame_multires_bubbles", "kind": "frame", "model": "multires", "scene": "bubbles", "nx": 256,
         "ny": 256, "nz": 256, "solver": "multigrid", "steps": 2, "surface": False},
        # one training gradient through the multigrid cycle
        {"name": "learned_gradient", "kind": "learned", "nx": 96, "ny": 96, "nz": 96, "ratio": 300.0},
    ]


def _between(rng, lo, hi):
    """an integer spread over the logarithm of its range"""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["cfl", "splat", "project", "project", "transport", "frame", "frame", "frame", "learned"])
    if kind == "cfl":
        return {"kind": kind, "n": _between(rng, 1000, 30000000)}

    def dims(lo, hi):
        n = _between(rng, lo, hi)
        if rng.random() < 0.25:  # a cube whose spacing is a power of two
            n = 1 << int(math.log2(n))
            return {"nx": n, "ny": n, "nz": n}
        return {"nx": n, "ny": max(12, int(n * rng.uniform(0.6, 1.2))), "nz": max(12, int(n * rng.uniform(0.6, 1.2)))}

    ratio = round(math.exp(rng.uniform(math.log(10.0), math.log(1000.0))), 1)
    if kind == "splat":
        return {"kind": kind, "scene": rng.choice(["rt", "tank"]), **dims(16, 170), "ratio": ratio}
    if kind == "transport":
        return {"kind": kind, "scene": rng.choice(["rt", "tank"]), **dims(16, 170), "substeps": rng.randint(2, 6)}
    if kind == "project":
        solver = rng.choice(["jacobi", "multigrid", "multigrid"])
        return {"kind": kind, "scene": rng.choice(["rt", "tank"]), **dims(16, 64 if solver == "jacobi" else 170),
                "ratio": ratio, "solver": solver}
    if kind == "learned":
        return {"kind": kind, **dims(24, 128), "ratio": ratio}
    model = rng.choice(["two_phase", "two_phase", "single_phase", "multires"])
    case = {"kind": kind, "model": model}
    if model == "two_phase":
        solver = rng.choice(["multigrid", "multigrid", "reference"])
        case.update(scene=rng.choice(["rt", "tank"]), solver=solver, steps=rng.randint(1, 4),
                    surface=rng.random() < 0.4, **dims(24, 72 if solver == "reference" else 200))
    elif model == "single_phase":
        case.update(scene="dam", solver="reference", steps=rng.randint(1, 4), surface=False, **dims(24, 160))
    elif rng.random() < 0.5:
        case.update(scene="band", solver="fast", steps=rng.randint(1, 4), surface=False, **dims(24, 88))
    else:
        n = 16 * _between(rng, 4, 14)
        case.update(scene="bubbles", solver="multigrid", steps=rng.randint(1, 2), surface=False, nx=n, ny=n, nz=n)
    return case


# ------------------------------------------------------------------ inputs

def _spacing(case):
    """the longest side has length 1; the multires tank keeps the reference's unit cells"""
    return 1.0 if case.get("scene") == "band" else 1.0 / max(case["nx"], case["ny"], case["nz"])


def _phase(ratio):
    ph = G.Phase(1000.0, 1000.0 / ratio, 1.0, 1.0)
    ph.rho_tilde_0 = G.calibrate_rho_tilde0(ph, 1.0)
    return ph


def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _motion(case, seed):
    """a smooth swirl with some phases of the seed's: f(axis, x, y, z) in units of the box"""
    r = np.random.default_rng(seed)
    amp, ph = r.uniform(0.4, 0.9, 3), r.uniform(0.0, 2.0 * math.pi, (3, 2))

    def at(axis, x, y, z):
        q = [x, y, z]
        a, b = q[(axis + 1) % 3], q[(axis + 2) % 3]
        return amp[axis] * torch.sin(math.pi * q[axis]) * torch.cos(2 * math.pi * a + ph[axis, 0]) \
            * torch.cos(2 * math.pi * b + ph[axis, 1])
    return at


def _particles(case, seed):
    """8 jittered particles per filled interior cell: FP32 positions and velocities and
    the phase, on the GPU.  rt: a full box, heavy above a wavy interface; tank: filled
    to 0.6 of the height with a bubble; band: the multires tank, filled to half."""
    nx, ny, nz, dx = case["nx"], case["ny"], case["nz"], _spacing(case)
    scene = case["scene"]
    top = {"rt": ny - 1, "tank": max(2, min(ny - 1, int(0.6 * ny))), "band": ny // 2}[scene]
    ax = [torch.arange(1, m, device=DEVICE, dtype=torch.float64) for m in (nx - 1, top, nz - 1)]
    k, j, i = torch.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    cell = torch.stack([i.reshape(-1), j.reshape(-1), k.reshape(-1)]).repeat_interleave(8, dim=1)
    del i, j, k
    gen = _generator(seed)
    # the jitter keeps a particle in its cell when its position is rounded to FP32
    jitter = torch.rand(cell.shape, generator=gen, device=DEVICE, dtype=torch.float64) * 0.999 + 0.0005
    pos = ((cell + jitter) * dx).float()
    del cell, jitter
    x, y, z = pos[0], pos[1], pos[2]
    L = [nx * dx, ny * dx, nz * dx]
    if scene == "rt":
        level = 0.5 * L[1] + 0.05 * L[0] * torch.cos(2 * math.pi * x / L[0]) * torch.cos(2 * math.pi * z / L[2])
        kind = (y <= level).to(torch.uint8)
    else:
        cy, r = (0.25 * L[1], 0.12 * L[0]) if scene == "tank" else (0.1875 * L[1], 0.1875 * min(L[0], L[2]))
        kind = ((x - 0.5 * L[0]) ** 2 + (y - cy) ** 2 + (z - 0.5 * L[2]) ** 2 < r * r).to(torch.uint8)
    at, scale = _motion(case, seed), max(L)
    vel = torch.stack([at(a, x / scale, y / scale, z / scale) for a in range(3)])
    vel = vel + 0.05 * torch.randn(vel.shape, generator=gen, device=DEVICE)
    return pos, vel.float() * scale, kind


def _upload(ctx, pos, vel, kind):
    p, v = pos.cpu().numpy(), vel.cpu().numpy()
    ctx.upload(p[0], p[1], p[2], v[0], v[1], v[2], type=kind.cpu().numpy())


FACES = (G.FIELD_U, G.FIELD_V, G.FIELD_W)
MASSES = (G.FIELD_MU, G.FIELD_MV, G.FIELD_MW)
SAVED = (G.FIELD_SAVED_U, G.FIELD_SAVED_V, G.FIELD_SAVED_W)


def _face_dims(case, axis):
    """(nz, ny, nx) of a face field; axis 3 is a cell field"""
    d = [case["nx"], case["ny"], case["nz"]]
    if axis < 3:
        d[axis] += 1
    return d[2], d[1], d[0]


def _given_field(case, seed):
    """prescribed face velocities, now and before the projection, per axis on the GPU"""
    dx, at = _spacing(case), _motion(case, seed + 1)
    scale = dx * max(case["nx"], case["ny"], case["nz"])
    now, before = [], []
    gen = _generator(seed + 2)
    for axis in range(3):
        dz, dy, dxs = _face_dims(case, axis)
        g = [torch.arange(m, device=DEVICE, dtype=torch.float64) + (0.0 if a == axis else 0.5)
             for a, m in enumerate((dxs, dy, dz))]
        z, y, x = torch.meshgrid(g[2] * dx / scale, g[1] * dx / scale, g[0] * dx / scale, indexing="ij")
        f = at(axis, x, y, z) * scale
        now.append(f.float())
        before.append((0.98 * f + 0.02 * scale * torch.rand(f.shape, generator=gen, device=DEVICE)).float())
    return now, before


# ------------------------------------------------------------------ outputs

class _Held:
    """A program's page-locked output buffers, filled by the library's downloads."""

    def __init__(self, ctx, fields=(), particles=False):
        self.ctx, self.fields = ctx, {}
        for f in fields:
            nx, ny, nz = ctx.dims(f)
            self.fields[f] = torch.empty((nz, ny, nx), dtype=torch.float32, pin_memory=True)
        n = ctx.count()
        self.particles = [torch.empty(n, dtype=torch.float32, pin_memory=True) for _ in range(6)] if particles else []

    def take(self):
        out, lib, h = {}, G.lib(), self.ctx.h
        for f, t in self.fields.items():
            self.ctx._check(lib.pf_field_download(h, f, ctypes.c_void_p(t.data_ptr())), "pf_field_download")
            out["field%02d" % f] = t
        if self.particles:
            self.ctx._check(lib.pf_particles_download(h, *[ctypes.c_void_p(t.data_ptr()) for t in self.particles]),
                            "pf_particles_download")
            out.update(zip(("px", "py", "pz", "pu", "pv", "pw"), self.particles))
        return out


# ------------------------------------------------------------------ cases

DT_PROJECT = 1e-3
BUBBLES_SEED = 20250601
FLIP = 0.95


def _solve_cfg(solver):
    if solver == "jacobi":  # tight: the exact pressure is what is compared
        return G.SolveCfg(max_iters=50000, stop_rule=G.STOP_REL2, tol=1e-10, inner_rel_tol=0.1, max_outer=10000,
                          warm_start=0, check_every=16, precond=G.PRECOND_JACOBI)
    return G.SolveCfg(max_iters=50000, stop_rule=G.STOP_REL2, tol=1e-10, inner_rel_tol=1e-2, max_outer=10000,
                      warm_start=0, check_every=4, precond=G.PRECOND_MULTIGRID)


def _transport_dt(case):
    return 0.3 * _spacing(case)  # about a third of a cell per substep at unit speed


def _frame_sim(case, seed):
    n, dx = (case["nx"], case["ny"], case["nz"]), _spacing(case)
    if case["model"] == "single_phase":
        sim = G.SparseSim3D(*n, dx)
        sim.ctx.scene(G.SCENE_DAMBREAK, seed)
        sim.dt = 2e-3
        sim.cg_iters, sim.cg_tol = 3000, 1e-6
        sim.adaptive_timestep, sim.adaptive_cfl = True, 1.0
        return sim
    if case["model"] == "multires":
        sim = G.MRSim3DTP(*n, dx)
        sim.cg_iters, sim.cg_tol = 20000, 0.0
        if case["scene"] == "band":
            sim.phase = G.Phase(1.0, 0.01, 1.0, 1.0)
            sim.dt = 0.02
            pos, vel, kind = _particles(case, seed)
            sim.set_layout(G.mr_layout_fine_box(*n))
            _upload(sim.ctx, pos, 0.0 * vel, kind)
        else:
            sim.dt, sim.dynamic_refinement = 5e-4, False
            # the same bubbles and layout for every seed, which moves their particles
            sim.ctx.scene_bubbles(BUBBLES_SEED, 16, 6)
            x, y, z = (torch.as_tensor(q).to(DEVICE) for q in sim.ctx.download()[:3])
            kind = torch.as_tensor(sim.ctx.download_ext()[0])
            at, gen = _motion(case, seed), _generator(seed)
            vel = torch.stack([at(a, x, y, z) for a in range(3)])
            vel = vel + 0.05 * torch.randn(vel.shape, generator=gen, device=DEVICE)
            _upload(sim.ctx, torch.stack([x, y, z]), vel.float(), kind)
            sim.phase = G.Phase(1000.0, 1.0, 1.0, 1.0)
            sim.solve_options = {"mode": G.MR_SOLVE_MULTIGRID}
    else:
        sim = G.SparseSim3DTP(*n, dx)
        sim.ctx.scene(G.SCENE_RT if case["scene"] == "rt" else G.SCENE_BUBBLE, seed)
        sim.phase = G.Phase(1000.0, 1.0, 1.0, 1.0)
        sim.dt = 1e-3 if case["scene"] == "rt" else 5e-4
        sim.cg_iters = 2000
        if case["solver"] == "multigrid":
            sim.precond, sim.stop_rule, sim.cg_tol, sim.cg_iters = G.PRECOND_MULTIGRID, G.STOP_REL2, 1e-6, 50000
            sim.inner_rel_tol, sim.check_every = 1e-4, 4
        sim.surface_tension = case["surface"]
        sim.interface_diagnostics = case["surface"]
    sim.phase.rho_tilde_0 = G.calibrate_rho_tilde0(sim.phase, 1.0)
    sim.adaptive_timestep, sim.adaptive_cfl = True, 0.5
    return sim


def prepare(case, seed):
    kind = case["kind"]
    if kind == "cfl":
        gen = _generator(seed)
        return {"case": case, "v": [torch.randn(case["n"], generator=gen, device=DEVICE) for _ in range(3)],
                "out": [ctypes.c_double(), ctypes.c_double(), ctypes.c_double(), ctypes.c_int32()]}
    if kind == "frame":
        sim = _frame_sim(case, seed)
        return {"case": case, "sim": sim, "held": _Held(sim.ctx, particles=True)}
    if kind == "learned":
        ctx = G.Context(case["nx"], case["ny"], case["nz"], _spacing(case))
        ctx.scene(G.SCENE_RT, seed)
        ph = _phase(case["ratio"])
        net = G.LearnedPreconditioner(seed)
        # weights away from the zero head, so that the gradient reaches every layer
        r = np.random.default_rng(seed)
        w = net.weights()
        w[-16:] = r.normal(0.0, 0.2, 16)
        net.set_weights(w)
        net.attach(ctx)
        G.lpc_record(ctx, 2, 1)
        _grid_half(ctx, ph, G.SolveCfg(max_iters=200, stop_rule=G.STOP_REL2, tol=1e-6, inner_rel_tol=0.01,
                                       max_outer=10000, warm_start=0, check_every=4, precond=G.PRECOND_MULTIGRID))
        return {"case": case, "ctx": ctx, "net": net}
    pos, vel, what = _particles({**case}, seed)
    ctx = G.Context(case["nx"], case["ny"], case["nz"], _spacing(case))
    _upload(ctx, pos, vel, what)
    state = {"case": case, "ctx": ctx}
    if kind == "splat":
        state.update(phase=_phase(case["ratio"]), held=_Held(ctx, (G.FIELD_MARKER,) + FACES + MASSES))
    elif kind == "project":
        state.update(phase=_phase(case["ratio"]), held=_Held(ctx, (G.FIELD_P,) + FACES))
    else:
        now, before = _given_field(case, seed)
        for axis in range(3):
            ctx.set_field(FACES[axis], now[axis].cpu().numpy())
            ctx.set_field(SAVED[axis], before[axis].cpu().numpy())
        state.update(held=_Held(ctx, particles=True))
    return state


def _grid_half(ctx, phase, solve):
    ctx.mark_cells()
    ctx.p2g(phase, 1.0)
    ctx.save_velocity()
    ctx.apply_gravity(DT_PROJECT, GRAVITY)
    ctx.apply_walls()
    return ctx.project(phase, DT_PROJECT, solve)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "cfl":
        u, v, w = state["v"]
        eff, vmax, cfl, lim = state["out"]
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        status = _noalloc()(u.data_ptr(), v.data_ptr(), w.data_ptr(), u.numel(), 1.0 / 64, 1e-2, 1, 0.5, 1e-6,
                            stream, ctypes.byref(eff), ctypes.byref(vmax), ctypes.byref(cfl), ctypes.byref(lim))
        if status != 0:
            raise RuntimeError("pf_timestep_noalloc: status %d" % status)
        return {"dt": eff.value, "speed": vmax.value, "cfl_dt": cfl.value, "limited": lim.value}
    if kind == "frame":
        for _ in range(case["steps"]):
            state["sim"].step()
        return state["held"].take()
    if kind == "learned":
        grad, loss = state["net"].grad(state["ctx"], 0)
        return {"grad": grad, "loss": loss}
    ctx = state["ctx"]
    if kind == "splat":
        ctx.mark_cells()
        ctx.p2g(state["phase"], 1.0)
    elif kind == "project":
        _grid_half(ctx, state["phase"], _solve_cfg(case["solver"]))
    else:
        for _ in range(case["substeps"]):
            ctx.mark_cells()
            ctx.g2p(FLIP, 0.9)
            ctx.advect(_transport_dt(case), 2)
    return state["held"].take()


_NOALLOC = None


def _noalloc():
    """pf_timestep_noalloc of the C ABI, with its argument types"""
    global _NOALLOC
    if _NOALLOC is None:
        f = G.lib().pf_timestep_noalloc
        p, d, i = ctypes.c_void_p, ctypes.c_double, ctypes.c_int32
        f.restype = ctypes.c_int
        f.argtypes = [p, p, p, ctypes.c_int64, d, d, i, d, d, p, ctypes.POINTER(d), ctypes.POINTER(d),
                      ctypes.POINTER(d), ctypes.POINTER(i)]
        _NOALLOC = f
    return _NOALLOC


# ------------------------------------------------------------------ work

def _counts(case):
    """(particles, cells, fluid cells) of a case, from its scene"""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    inner = (nx - 2) * (nz - 2)
    fluid = {"rt": inner * (ny - 2), "tank": inner * int(0.6 * ny), "band": inner * (ny // 2),
             "dam": int(0.4 * nx) * int(0.6 * ny) * (nz - 2), "bubbles": inner * (ny // 2)}[case.get("scene", "rt")]
    if case.get("scene") == "bubbles":
        # fine cells near the surface and the bubbles, 4^3 fine cells to a cell elsewhere
        fluid = fluid // 8
    return 8 * fluid, nx * ny * nz, fluid


def work(case):
    kind = case["kind"]
    if kind == "cfl":
        return {"bytes": 12 * case["n"], "flops": 6 * case["n"]}
    parts, cells, fluid = _counts(case)
    splat_flops = 3 * 36 * 10 * parts  # 36 nodes an axis, about 10 operations a node
    if kind == "splat":
        return {"bytes": 25 * parts + 28 * cells, "flops": splat_flops}
    if kind == "project":
        # particles in, face masses in and velocities and pressure out; one operator pass
        return {"bytes": 25 * parts + 28 * cells + 32 * fluid, "flops": splat_flops}
    if kind == "transport":
        # a substep reads and writes the particles and reads the velocity fields
        n = case["substeps"]
        return {"bytes": n * (49 * parts + 24 * cells) + 24 * parts, "flops": n * 300 * parts}
    if kind == "learned":
        return {"bytes": 40 * cells, "flops": 3 * LEARNED_FLOPS * (cells // 8)}
    # a step reads and writes every particle and the faces' velocities and masses; the
    # frame then reads the particles once more
    return {"bytes": case["steps"] * (53 * parts + 40 * fluid) + 24 * parts,
            "flops": case["steps"] * (splat_flops + 300 * parts)}


def tolerance(case):
    """About four times what was measured between two correct forms of the path.  Splat
    and transport: against FP64.  Projection and frames: the Jacobi PCG against the
    multigrid, and a fifth of the solver's tolerance against the tolerance itself; the
    velocity components that stay small, and curvatures at the bubble, show it most
    (8e-4 over the 2-norm with surface tension, 5e-6 without)."""
    kind = case["kind"]
    if kind == "cfl":
        return {"rel": 2e-7, "max": 2e-7}
    if kind == "splat":
        return {"rel": 1e-6, "max": 1e-3}
    if kind == "project":
        return {"rel": 1e-5, "max": 1e-3}
    if kind == "transport":
        return {"rel": 4e-6, "max": 1e-3}
    if kind == "learned":  # products of bf16 weights and activations
        return {"rel": 2e-2}
    if case["model"] == "multires":
        return {"rel": 1e-5, "max": 1e-3}
    if case["model"] == "single_phase":
        return {"rel": 2e-4, "max": 5e-3}
    return {"rel": 3e-3, "max": 0.9} if case["scene"] == "tank" or case["surface"] else {"rel": 5e-5, "max": 2e-3}


# ------------------------------------------------------------------ the same in 64 bits

def _axes(case, axis):
    """offset of a face field's nodes from the cell corners, per coordinate"""
    return [0.0 if a == axis else 0.5 for a in range(3)]


def _splat64(case, pos, vel, kind, phase):
    """normalised face velocities and face masses, (nz, ny, nx) each, in FP64: weights
    (1 - d^2 / 2.25)^3 within 1.5 cells, normalised over the nodes inside the grid"""
    dx = _spacing(case)
    mass = torch.where(kind == 0, phase.rho_l, phase.rho_g).double()
    faces, masses = [], []
    for axis in range(3):
        dims = _face_dims(case, axis)
        off = _axes(case, axis)
        flow = torch.zeros(dims[0] * dims[1] * dims[2], dtype=torch.float64, device=DEVICE)
        summed = torch.zeros_like(flow)
        for lo in range(0, pos.shape[1], 1 << 22):
            part = slice(lo, lo + (1 << 22))
            g = [pos[a, part].double() / dx - off[a] for a in range(3)]
            base = [q.floor() for q in g]
            total = torch.zeros_like(g[0])
            for deposit in (False, True):
                for n in range(64):
                    node = [base[a] + ((n >> (2 * a)) & 3) - 1 for a in range(3)]
                    d2 = sum((g[a] - node[a]) ** 2 for a in range(3))
                    wgt = (1.0 - d2 / 2.25).clamp_min(0.0) ** 3
                    for a in range(3):
                        wgt = torch.where((node[a] >= 0) & (node[a] < dims[2 - a]), wgt, 0.0)
                    if not deposit:
                        total += wgt
                        continue
                    idx = sum((node[a].clamp(0, dims[2 - a] - 1)).long() * s
                              for a, s in enumerate((1, dims[2], dims[2] * dims[1])))
                    add = mass[part] * wgt / total
                    summed.index_add_(0, idx, add)
                    flow.index_add_(0, idx, add * vel[axis, part].double())
        faces.append(torch.where(summed > 0, flow / summed.clamp_min(1e-300), 0.0).reshape(dims))
        masses.append(summed.reshape(dims))
    return faces, masses


def _markers64(case, pos):
    dx = _spacing(case)
    nz, ny, nx = _face_dims(case, 3)
    cell = (pos.double() / dx).long()
    mark = torch.zeros(nz, ny, nx, dtype=torch.float64, device=DEVICE)
    mark.view(-1)[cell[0] + nx * (cell[1] + ny * cell[2])] = FLUID
    for a in range(3):
        mark.select(a, 0).fill_(SOLID)
        mark.select(a, mark.shape[a] - 1).fill_(SOLID)
    return mark


def _beta64(raw, phase):
    floor = math.log(phase.rho_l / phase.rho_g) * phase.rho_g * phase.rho_tilde_0
    phi = ((raw - floor).clamp_min(0.0) / (phase.alpha_phi * phase.rho_tilde_0 * phase.rho_l)).sqrt().clamp_max(1.0)
    return 1.0 / (phi * phase.rho_l + (1.0 - phi) * phase.rho_g)


def _project64(case, phase, mark, faces, masses):
    """the pressure of the variable-coefficient system solved to rounding, and the
    projected face velocities"""
    dx, dt = _spacing(case), DT_PROJECT
    fluid, solid = mark == FLUID, mark == SOLID
    unknown = fluid.clone()
    air_side = torch.zeros(1, dtype=torch.bool, device=DEVICE)
    flow, coef = [], []
    for axis in range(3):  # interior faces only: the outermost cells are solid
        d = 2 - axis
        n = mark.shape[d]
        left, right = fluid.narrow(d, 0, n - 1), fluid.narrow(d, 1, n - 1)
        closed = solid.narrow(d, 0, n - 1) | solid.narrow(d, 1, n - 1)
        air_side |= ((left != right) & ~closed).any()
        flow.append(torch.where(closed, 0.0, faces[axis].narrow(d, 1, n - 1)))
        coef.append(torch.where((left | right) & ~closed, _beta64(masses[axis].narrow(d, 1, n - 1), phase), 0.0))
    if not bool(air_side):  # no free surface: the first fluid cell is pinned at zero
        unknown.view(-1)[torch.nonzero(fluid.view(-1))[0]] = False

    def apply(p):
        out = torch.zeros_like(p)
        for axis in range(3):
            d, n = 2 - axis, p.shape[2 - axis]
            g = coef[axis] * (p.narrow(d, 1, n - 1) - p.narrow(d, 0, n - 1))
            out.narrow(d, 0, n - 1).sub_(g)
            out.narrow(d, 1, n - 1).add_(g)
        return torch.where(unknown, out * (dt / dx ** 2), 0.0)

    rhs, diag = torch.zeros_like(mark), torch.zeros_like(mark)
    for axis in range(3):
        d, n = 2 - axis, mark.shape[2 - axis]
        rhs.narrow(d, 0, n - 1).sub_(flow[axis] / dx)
        rhs.narrow(d, 1, n - 1).add_(flow[axis] / dx)
        diag.narrow(d, 0, n - 1).add_(coef[axis] * (dt / dx ** 2))
        diag.narrow(d, 1, n - 1).add_(coef[axis] * (dt / dx ** 2))
    rhs = torch.where(unknown, rhs, 0.0)
    inv = torch.where(unknown & (diag > 0), 1.0 / diag.clamp_min(1e-300), 0.0)
    p, r = torch.zeros_like(rhs), rhs.clone()
    z = r * inv
    q, rz, bound = z.clone(), (r * z).sum(), 1e-13 * float(rhs.norm())
    for it in range(20000):
        aq = apply(q)
        alpha = rz / (q * aq).sum()
        p += alpha * q
        r -= alpha * aq
        if it % 64 == 0 and float(r.norm()) <= bound:
            break
        z = r * inv
        new = (r * z).sum()
        q = z + (new / rz) * q
        rz = new
    out = []
    for axis in range(3):
        d, n = 2 - axis, mark.shape[2 - axis]
        near = fluid.narrow(d, 0, n - 1) | fluid.narrow(d, 1, n - 1)
        closed = solid.narrow(d, 0, n - 1) | solid.narrow(d, 1, n - 1)
        f = faces[axis].clone()
        inner = f.narrow(d, 1, n - 1)
        step = (dt / dx) * coef[axis] * (p.narrow(d, 1, n - 1) - p.narrow(d, 0, n - 1))
        inner.copy_(torch.where(near, torch.where(closed, 0.0, inner - step), inner))
        out.append(f)
    return p, out


def _walls64(faces):
    for axis in range(3):
        f, d = faces[axis], 2 - axis
        for at in (0, 1, f.shape[d] - 2, f.shape[d] - 1):
            f.select(d, at).zero_()


def _sample64(case, faces, pos):
    dx, out = _spacing(case), []
    for axis in range(3):
        f = faces[axis].double()
        dims = f.shape
        off = _axes(case, axis)
        g = [pos[a] / dx - off[a] for a in range(3)]
        base = [q.floor() for q in g]
        total = torch.zeros_like(g[0])
        for n in range(8):
            bit = [(n >> a) & 1 for a in range(3)]
            wgt = torch.ones_like(total)
            idx = torch.zeros(total.shape, dtype=torch.long, device=DEVICE)
            for a, s in enumerate((1, dims[2], dims[2] * dims[1])):
                fr = g[a] - base[a]
                wgt = wgt * (fr if bit[a] else 1.0 - fr)
                idx += (base[a] + bit[a]).clamp(0, dims[2 - a] - 1).long() * s
            total += wgt * f.reshape(-1)[idx]
        out.append(total)
    return torch.stack(out)


def exact(case, seed):
    """run()'s outputs in 64 bits where the path has such a value.  Frames have none:
    their pressure is solved to the program's own tolerance in every step; nor has the
    gradient of a network that computes in bf16."""
    kind = case["kind"]
    if kind == "cfl":
        gen = _generator(seed)
        v = [torch.randn(case["n"], generator=gen, device=DEVICE).double() for _ in range(3)]
        speed = float((v[0] ** 2 + v[1] ** 2 + v[2] ** 2).max().sqrt())
        cfl = 0.5 * (1.0 / 64) / speed
        return {"dt": np.float64(min(1e-2, max(1e-6, cfl))), "speed": np.float64(speed), "cfl_dt": np.float64(cfl),
                "limited": None}
    if kind in ("frame", "learned"):
        return None
    pos, vel, what = _particles(case, seed)
    if kind == "transport":
        now, before = _given_field(case, seed)
        p, v = pos.double(), vel.double()
        alpha = torch.where(what == 0, FLIP, 0.9).double()
        dt, dx = _transport_dt(case), _spacing(case)
        for _ in range(case["substeps"]):
            here = _sample64(case, now, p)
            v = (v + here - _sample64(case, before, p)) * alpha + here * (1.0 - alpha)
            p = p + dt * _sample64(case, now, p + 0.5 * dt * here)
            for a, n in enumerate((case["nx"], case["ny"], case["nz"])):
                p[a].clamp_(0.5 * dx, (n - 0.5) * dx)
        return {"px": p[0], "py": p[1], "pz": p[2], "pu": v[0], "pv": v[1], "pw": v[2]}
    phase = _phase(case["ratio"])
    faces, masses = _splat64(case, pos, vel, what, phase)
    mark = _markers64(case, pos)
    if kind == "splat":
        return {"field%02d" % f: t for f, t in zip((G.FIELD_MARKER,) + FACES + MASSES, [mark] + faces + masses)}
    faces[1] = torch.where(masses[1] > 0, faces[1] + DT_PROJECT * GRAVITY, faces[1])
    _walls64(faces)
    p, faces = _project64(case, phase, mark, faces, masses)
    return {"field%02d" % f: t for f, t in zip((G.FIELD_P,) + FACES, [p] + faces)}
