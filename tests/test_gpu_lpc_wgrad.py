"""Weight gradients on the matrix cores, their partial sums and the four-row convolution,
against the oracle with the same BF16 rounding points.

Weights, inputs and output gradients are small integers, so every product is a whole
number and every FP32 partial sum is exact in any order while it stays under 2^24 (the
test checks the sum of magnitudes): the forward pass and all four layers' gradients have to
equal the oracle's exactly.  Tile counts: one tile (8 partials a layer, fewer than the 16
threads that sum an output), 3, and 37 (296 units for at most 256 partials: some
workgroups take two).
"""
import numpy as np
import pytest
import torch

import lpc_oracle as LO
import pfflip_amd as G

pytestmark = pytest.mark.gpu


def _case(nt, seed):
    rng = np.random.default_rng(seed)
    w = np.where(rng.random(sum(LO.SIZES)) < 0.04, rng.choice([-1.0, 1.0], sum(LO.SIZES)), 0.0)
    w[-LO.SIZES[3]:] = rng.choice([-2.0, -1.0, 1.0, 2.0], LO.SIZES[3])
    X = np.where(rng.random((nt, 18, 18, 18, 4)) < 0.5, rng.integers(-3, 4, (nt, 18, 18, 18, 4)), 0)
    gO = np.where(rng.random((nt, 16, 16, 16)) < 0.25, rng.choice([-1.0, 1.0], (nt, 16, 16, 16)), 0.0)
    return w.astype(np.float32), X.astype(np.float32), gO.astype(np.float32)


@pytest.mark.parametrize("nt", [1, 3, 37])
def test_integer_gradients_are_exact(nt):
    w, X, gO = _case(nt, 11 + nt)
    net = G.LearnedPreconditioner(seed=1)
    net.set_weights(w)
    out, cache = LO.forward(X, w.astype(np.float64), bf16=True)
    ref = LO.backward(cache, gO, w.astype(np.float64), bf16=True)
    bound = LO.backward(cache, np.abs(gO), np.abs(w).astype(np.float64), bf16=True)
    assert np.abs(bound).max() < 2 ** 24
    assert np.abs(ref).max() > 0 and all(
        np.abs(ref[o:o + n]).max() > 0 for o, n in zip(np.cumsum([0, *LO.SIZES[:3]]), LO.SIZES))
    assert np.array_equal(net.forward_tiles(X), out.astype(np.float32))
    assert np.array_equal(net.grad_tiles(X, gO), ref.astype(np.float32))


def test_one_tile_takes_one_tile_of_memory():
    """activations and gradients of a tile take about 1.2 MB, its 8 partials a layer 2 MB"""
    _, X, gO = _case(1, 3)
    G.LearnedPreconditioner(seed=1).grad_tiles(X, gO)  # (what the kernels' first launch takes)
    net = G.LearnedPreconditioner(seed=1)
    free = torch.cuda.mem_get_info()[0]
    net.grad_tiles(X, gO)
    assert free - torch.cuda.mem_get_info()[0] < 24 << 20


@pytest.mark.parametrize("e", [112, 117, 123])
def test_gradients_past_the_range_of_float32_are_infinite(e):
    """output gradients of 2^e: sums past FP32's range in the last sum alone (some stay below,
    exact), in a workgroup's, in a chain; nothing is negative, so they come out as Inf and
    not as NaN.  (The last layer's: further down 0 times Inf is NaN in the gradient itself.)"""
    w, X, gO = _case(3, 5)
    w, gO = np.abs(w), np.abs(gO)
    net = G.LearnedPreconditioner(seed=1)
    net.set_weights(w)
    _, cache = LO.forward(X, w.astype(np.float64), bf16=True)
    layer = slice(sum(LO.SIZES[:2]), sum(LO.SIZES[:3]))
    ref = LO.backward(cache, gO, w.astype(np.float64), bf16=True)[layer]
    assert ref.max() < 2 ** 24 and (ref >= 2 ** 16).any() and (ref < 2 ** 16).any()
    with np.errstate(over="ignore"):
        want = (ref * 2.0 ** e).astype(np.float32)
    assert np.array_equal(net.grad_tiles(X, gO * np.float32(2.0 ** e))[layer], want)
