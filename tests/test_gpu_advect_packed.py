"""Advection alone with the velocity packed in pairs (many particles) against the plain gathers
(few): the same particles advected in one context that holds only them and in one filled up
with others give the same bits, both orders, near every wall and past it (clamped), on
ragged grids.
"""
import numpy as np
import pytest
import torch

import pfflip_amd as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [2, 3])
@pytest.mark.parametrize("dims", [(3, 3, 3), (5, 9, 6), (17, 16, 12), (31, 8, 22)])
def test_pairs_equal_plain_gathers(dims, order):
    nx, ny, nz = dims
    dx = 1.0 / nx
    r = np.random.default_rng(7)
    cells, few = nx * ny * nz, nx * ny * nz // 2
    n = 700000 + cells
    lim = np.array(dims) * dx
    p = (r.uniform(0.0, 1.0, (n, 3)) * lim).astype(np.float32)
    p = np.minimum(p, np.nextafter(lim.astype(np.float32), np.float32(0)))
    p[: few // 2, 0] = np.where(r.random(few // 2) < 0.5, 1e-4 * dx, lim[0] * 0.9999)  # the first and last x cells
    fields = {}
    for f, d in ((G.FIELD_U, (nz, ny, nx + 1)), (G.FIELD_V, (nz, ny + 1, nx)), (G.FIELD_W, (nz + 1, ny, nx))):
        fields[f] = r.normal(scale=0.6, size=d).astype(np.float32)
    out = []
    for m in (few, n):
        least = 600000 + cells // 5 * 2 if order == 3 else 700000 + cells // 3 * 2
        assert (m >= max(cells, least)) == (m == n)
        ctx = G.Context(nx, ny, nz, dx)
        ctx.upload(p[:m, 0], p[:m, 1], p[:m, 2])
        for f, a in fields.items():
            ctx.set_field(f, a)
        es = ctx.advect(2.0 * dx, order)
        assert es.clamped_liquid > 0
        out.append([q[:few] for q in ctx.download()[:3]])
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_pairs_take_their_own_size():
    """advection alone holds 8 bytes a face, not the G2P's 16; a G2P after it the quads alone,
    and advection then goes on in them"""
    n = 128
    ctx = G.Context(n, n, n, 1.0 / n)
    r = np.random.default_rng(3)
    p = r.uniform(0.05, 0.95, (n ** 3, 3)).astype(np.float32)
    ctx.upload(*(np.ascontiguousarray(p[:, a]) for a in range(3)))
    ctx.set_field(G.FIELD_U, r.normal(size=(n, n, n + 1)).astype(np.float32))
    first = torch.cuda.mem_get_info()[0]
    ctx.advect(0.1 / n, 2)
    pairs = first - torch.cuda.mem_get_info()[0]
    moved = ctx.download()[0]
    faces = 3 * n * n * (n + 4)
    assert pairs < 10 * faces
    ctx.upload(*(np.ascontiguousarray(p[:, a]) for a in range(3)))
    ctx.g2p(0.95, 0.9)
    assert first - torch.cuda.mem_get_info()[0] < 18 * faces
    ctx.advect(0.1 / n, 2)
    assert first - torch.cuda.mem_get_info()[0] < 18 * faces
    assert np.array_equal(moved, ctx.download()[0])
