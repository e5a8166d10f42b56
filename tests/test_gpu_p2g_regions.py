"""P2G with the blocks' node sums gathered from memory (grids of up to 262144 blocks)
against the launches by colour (larger grids): the same particles in 260 x 260 x 248 and in
260^3 cells, which share every wall that the particles reach, give the same momentum, mass
and active blocks bit for bit, since both add a node's sums in colour order.  The three
splats (multires: levels 0 to 2), FP32 and FP64 cell coordinates; particles by the walls and on cell edges, a crowded
cell, lone particles far apart; then fewer particles in the same contexts, whose other
blocks have to come out empty.
"""
import numpy as np
import pytest

import pfflip_amd as G

pytestmark = pytest.mark.gpu

NX, SHORT, TALL = 260, 248, 260
FIELDS = (G.FIELD_U, G.FIELD_V, G.FIELD_W, G.FIELD_MU, G.FIELD_MV, G.FIELD_MW)


def _particles(rng):
    full = rng.uniform([0, 0, 0], [13, 10, 11], (8 * 13 * 10 * 11, 3))          # a low corner
    high = np.array([NX, NX, 238]) - rng.uniform(0, 1, (3000, 3)) * [9, 6, 7]   # by the high walls
    lone = rng.uniform([0, 0, 0], [NX, NX, 238], (400, 3))
    crowd = np.array([50, 60, 70]) + rng.uniform(0, 1, (150, 3))
    edge = rng.integers(1, 130, (300, 3)).astype(np.float64)
    p = np.concatenate([full, high, lone, crowd, edge])
    return p[rng.permutation(len(p))]


@pytest.mark.parametrize("dx", [0.25, 0.3])
@pytest.mark.parametrize("kind", ["two_phase", "single", "multires"])
def test_regions_equal_colour_launches(dx, kind):
    rng = np.random.default_rng(5)
    p = _particles(rng)
    vel = rng.normal(size=p.shape).astype(np.float32)
    ty = (rng.random(len(p)) < 0.4).astype(np.uint8)
    x = np.clip((p * dx).astype(np.float32), 0, np.nextafter(np.float32(NX * dx), np.float32(0)))
    ph = G.Phase(1000.0, 1.0, 0.0, 1.0)
    ctxs = [(G.MRContext if kind == "multires" else G.Context)(NX, NX, nz, dx) for nz in (SHORT, TALL)]
    if kind == "multires":
        for ctx, nz in zip(ctxs, (SHORT, TALL)):
            leaves = G.mr_layout_fine_box(NX, NX, nz, level=2)
            for box in ([0, 0, 0, 90, 40, 40], [0, 0, 0, 30, 10, 16], [230, 240, 200, 260, 260, 232]):
                leaves = G.mr_layout_refine(NX, NX, nz, leaves, box)
            ctx.set_layout(leaves)
    assert (NX // 4) ** 2 * ((SHORT + 3) // 4) <= 262144 < (NX // 4) ** 2 * (TALL // 4)
    for keep in (len(p), len(p) // 7):
        got = []
        for ctx in ctxs:
            ctx.upload(*x[:keep].T.copy(), *vel[:keep].T.copy(), ty[:keep])
            ctx.p2g_single() if kind == "single" else (ctx.mr_p2g if kind == "multires" else ctx.p2g)(ph, 1.0)
            nz = ctx.dims(G.FIELD_U)[2]
            f = []
            for k in FIELDS:
                d = ctx.dims(k)
                a = np.asarray(ctx.field(k)).reshape(d[2], d[1], d[0])
                assert nz == SHORT or not a[SHORT:].any()
                f.append(a[:SHORT])
            got.append((f, [ctx.active_blocks(k) for k in FIELDS]))
        for a, b in zip(got[0][0], got[1][0]):
            assert a.any() and np.array_equal(a, b)
        for a, b in zip(got[0][1], got[1][1]):
            assert len(a) and np.array_equal(np.sort(a), np.sort(b))
