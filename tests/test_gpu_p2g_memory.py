"""The splat's regions under memory pressure: an allocation that does not fit gives them
back before it fails, and the next splat, which takes them again, gives the same bits.
"""
import numpy as np
import pytest
import torch

import pfflip_amd as G

pytestmark = pytest.mark.gpu


def test_regions_are_given_back_before_an_allocation_fails():
    n = 128
    ctx = G.Context(n, n, n, 1.0 / n)
    ctx.scene(G.SCENE_RT, 3)
    ph = G.Phase(1000.0, 1.0, 0.0, 1.0)
    ctx.p2g(ph, 1.0)
    before = [ctx.field(f) for f in (G.FIELD_U, G.FIELD_MV)]
    free, total = torch.cuda.mem_get_info()
    regions = 3 * 256 * 8 * (n // 4) ** 3
    with pytest.raises(G.PfError, match="out of memory"):
        G.lpc_record(ctx, 2 * total // (4 * n ** 3))  # snapshots of twice the card's memory
    assert torch.cuda.mem_get_info()[0] >= free + regions - (16 << 20)  # (the runtime takes a little itself)
    ctx.p2g(ph, 1.0)
    for a, f in zip(before, (G.FIELD_U, G.FIELD_MV)):
        assert np.array_equal(a, ctx.field(f))
    assert torch.cuda.mem_get_info()[0] <= free + (16 << 20)
