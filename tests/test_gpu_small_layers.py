"""Layers over images of at most four channels: the sizes at which the windowed kernels can go
wrong.  Rows that end inside a wave's 32 pixels, grids with fewer rows than a workgroup has
waves, more batch elements than a window space holds, kernel sizes on both sides of a lane
half's sample group, output channels on both sides of a 32-row block, maps that fit no window,
point weights, and values that must not be touched under a zero weight.

Tolerances: forward sums at most 4 * 25 products (1e-5); gradients add over batch and pixels in an
order of their own (1e-4), as for the other float32 convolution kernels.
"""
import numpy as np
import pytest
import torch

import workloads
from conftest import relerr

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from _spherical_distortion_ext import _ops
    return _ops


def _t(a):
    return None if a is None else torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def _check(ops, oracle, B, Cin, Cout, m, wts, H, W, interp, seed):
    rng = np.random.default_rng(seed)
    K = m.shape[2]
    x = rng.standard_normal((B, Cin, H, W)).astype(np.float32)
    w = (rng.standard_normal((Cout, Cin, K)) / np.sqrt(Cin * K)).astype(np.float32)
    b = rng.standard_normal(Cout).astype(np.float32)
    g = rng.standard_normal((B, Cout) + m.shape[:2]).astype(np.float32)
    y = ops.mapped_conv_forward(_t(x), _t(m), _t(wts), _t(w), _t(b), K, interp)
    assert relerr(y.cpu().numpy(),
                  oracle.mapped_conv_forward(x, m, w, b, K, interp, wts)) <= 1e-5
    grads = ops.mapped_conv_backward(_t(g), _t(m), _t(wts), _t(x), _t(w), _t(b), K, interp)
    for got, want in zip(grads, oracle.mapped_conv_backward(g, m, x, w, b, K, interp, wts)):
        assert relerr(got.cpu().numpy(), want) <= 1e-4


def _near(rng, OH, OW, K, spread, wild, stride=1):
    """Samples within `spread` of their pixel, a share `wild` of them anywhere, some outside."""
    ys, xs = np.meshgrid(np.arange(OH) * stride, np.arange(OW) * stride, indexing="ij")
    c = np.stack([xs, ys], -1)[:, :, None, :] + rng.uniform(-spread, spread, (OH, OW, K, 2))
    far = rng.uniform(-3, 1.1 * stride * max(OH, OW), (OH, OW, K, 2))
    return np.where(rng.random((OH, OW, K, 1)) < wild, far, c).astype(np.float32)


@pytest.mark.parametrize("interp", [0, 1, 2])
@pytest.mark.parametrize("B,Cin,Cout,OH,OW,K", [
    (1, 1, 8, 3, 31, 9),      # three rows, no full piece, one pixel row block
    (2, 3, 17, 5, 33, 10),    # one pixel in a second piece; the largest single sample group
    (9, 3, 32, 40, 64, 9),    # full pieces; nine batch elements through the weight gradient
    (3, 4, 33, 37, 70, 11),   # a second 32-row block; the smallest of three sample groups
    (1, 2, 65, 1, 130, 1),    # one row, one sample, a second channel chunk
    (2, 4, 128, 9, 40, 25),
])
def test_edges_of_pieces_groups_and_blocks(ops, oracle, B, Cin, Cout, OH, OW, K, interp):
    rng = np.random.default_rng(OH * OW + K)
    m = _near(rng, OH, OW, K, 1.6, 0.0)
    _check(ops, oracle, B, Cin, Cout, m, None, OH, OW, interp, 3)


def _tiling(B, OH, OW):
    """(waves of a workgroup, stacked?, tiles, batch elements of a forward's and of a weight gradient's
    workgroup, workgroups of the latter that walk tiles), as small_tiling and its callers choose."""
    pieces = -(-OW // 32)
    waves = 4 if pieces * OH * B >= 1024 else 1
    stacked = OH >= waves
    tiles = pieces * -(-OH // waves) if stacked else -(-OW // (32 * waves)) * OH
    want = min(768, max(64, int(8 * (tiles * B) ** 0.5)))
    walkers = min(tiles, want)
    return (waves, stacked, tiles, -(-B // min(B, -(-2048 // tiles))),
            -(-B // min(B, max(1, want // walkers))), walkers)


@pytest.mark.parametrize("Cin,Cout,K,B,OH,OW,stride", [
    (3, 17, 7, 1, 1, 33001, 1),     # a vertex list: four waves side by side
    (3, 17, 9, 1, 3, 12001, 1),     # fewer rows than a workgroup's waves
    (3, 20, 9, 4, 101, 70, 1),      # four waves, the last tiles cut below and on the right
    (3, 17, 9, 6, 245, 515, 1),     # several batch elements in the windows at once, more to come
    (4, 33, 9, 4, 245, 515, 2),     # windows so large that each batch element has its own turn
])
def test_workgroups_of_four_waves(ops, oracle, Cin, Cout, K, B, OH, OW, stride):
    waves, stacked, tiles, forward, weights, walkers = _tiling(B, OH, OW)
    assert waves == 4 and stacked == (OH >= 4)
    if OH == 245:    # the batch loops and the walk over several tiles
        assert forward > 1 and weights == B and walkers < tiles
    else:
        assert OW % 32 and OH % 4
    rng = np.random.default_rng(OW)
    m = _near(rng, OH, OW, K, 1.6 if OH > 3 else 0.9, 0.0, stride)
    _check(ops, oracle, B, Cin, Cout, m, None, OH * stride, OW * stride, 1, OH)


@pytest.mark.parametrize("interp", [0, 1, 2])
def test_tiles_that_fit_no_window(ops, oracle, interp):
    rng = np.random.default_rng(5)
    m = _near(rng, 48, 96, 9, 1.6, 0.3)
    # (coordinates that no integer holds are left out: converting them is undefined in C++, and
    # the oracle's result for them with it)
    m[1, 2, 3] = [1e6, -1e6]
    _check(ops, oracle, 4, 3, 24, m, None, 48, 96, 1 if interp == 2 else interp, 4)
    # a spherical kernel: the rows next to the poles span the image, tiles cross the wrap seam
    m = workloads.gnomonic_kernel_map(64, 128)
    _check(ops, oracle, 4, 3, 24, m, None, 64, 128, interp, 5)
    m = workloads.gnomonic_kernel_map(65, 130, stride=2)
    _check(ops, oracle, 2, 4, 40, m, None, 65, 130, interp, 6)


def test_point_weights(ops, oracle):
    m, wts = workloads.four_nearest_weighted(workloads.gnomonic_kernel_map(40, 80), 40, 80)
    _check(ops, oracle, 3, 3, 20, m, wts, 40, 80, 2, 7)


def test_zero_weight_taps_are_not_read(ops):
    """Integer coordinates put weight on one tap; infinite and missing values all round it must
    not reach the sums."""
    H, W, K, Cout = 32, 64, 9, 24
    ys, xs = np.meshgrid(np.arange(H) // 2 * 2, np.arange(W) // 2 * 2, indexing="ij")
    m = np.broadcast_to(np.stack([xs, ys], -1)[:, :, None, :], (H, W, K, 2)).astype(np.float32)
    x = np.full((4, 3, H, W), np.inf, np.float32)
    x[:, :, 1::2] = np.nan
    x[:, :, ::2, ::2] = 1.0
    w = np.ones((Cout, 3, K), np.float32)
    g = np.ones((4, Cout, H, W), np.float32)
    b = np.zeros(Cout, np.float32)
    y = ops.mapped_conv_forward(_t(x), _t(m), None, _t(w), _t(b), K, 1)
    assert torch.equal(y, torch.full_like(y, 3.0 * K))
    _, gw, _ = ops.mapped_conv_backward(_t(g), _t(m), None, _t(x), _t(w), _t(b), K, 1)
    assert torch.equal(gw, torch.full_like(gw, 4.0 * H * W))


@pytest.mark.parametrize("OH,OW", [(2048, 2048), (2049, 2048)])
def test_both_sides_of_the_stores_of_a_descriptor(ops, OH, OW):
    """4194304 output pixels are the most the matrix kernel's stores reach; a picture of more takes
    the flat forward, and its backward the same kernels as every first layer's."""
    gen = torch.Generator(device=DEV).manual_seed(OH)
    H, W, Cin, Cout = 32, 64, 3, 17
    at = torch.randint(0, H * W, (OH, OW, 1), generator=gen, device=DEV)
    m = torch.stack([at % W, at // W], -1).float()
    x, w, b, g = (torch.randn(s, generator=gen, device=DEV) for s in (
        (1, Cin, H, W), (Cout, Cin, 1), (Cout,), (1, Cout, OH, OW)))
    y = ops.mapped_conv_forward(x, m, None, w, b, 1, 0)
    gi, gw, gb = ops.mapped_conv_backward(g, m, None, x, w, b, 1, 0)
    cols, wide = x.double().reshape(Cin, -1)[:, at.reshape(-1)], g.double().reshape(Cout, -1)
    want = (w[..., 0].double() @ cols + b[:, None].double()).reshape(y.shape)
    assert float((y - want).abs().max() / want.abs().max()) <= 1e-6    # sums of four terms
    grad = torch.zeros(Cin, H * W, dtype=torch.float64, device=DEV)
    grad.index_add_(1, at.reshape(-1), w[..., 0].double().T @ wide)
    for got, ref in ((gi.reshape(Cin, -1), grad), (gw[..., 0], wide @ cols.T), (gb, wide.sum(1))):
        assert float((got - ref).abs().max() / ref.abs().max()) <= 1e-4


@pytest.mark.parametrize("wild", [0.0, 0.4])
@pytest.mark.parametrize("Cin,Cout,K", [(3, 17, 9), (3, 17, 11), (2, 17, 9), (2, 17, 11), (2, 8, 9),
                                        (2, 8, 11), (3, 8, 11)])
def test_infinities_stay_in_their_channel(ops, oracle, Cin, Cout, K, wild):
    """Window elements and weights are padded to three or four channels: an infinity of the image
    gives infinities, no NaN from the padding's zero weights."""
    rng = np.random.default_rng(Cin + K)
    OH, OW = 37, 70
    m = _near(rng, OH, OW, K, 1.6, wild)
    x = rng.standard_normal((2, Cin, OH, OW)).astype(np.float32)
    x[0, 0, 5, 7], x[1, Cin - 1, 20, 30] = np.inf, np.inf
    w = rng.uniform(0.1, 1, (Cout, Cin, K)).astype(np.float32)
    b = rng.standard_normal(Cout).astype(np.float32)
    y = ops.mapped_conv_forward(_t(x), _t(m), None, _t(w), _t(b), K, 0).cpu().numpy()
    want = oracle.mapped_conv_forward(x, m, w, b, K, 0, None)
    assert np.isinf(want).any() and not np.isnan(want).any()
    assert np.array_equal(np.isinf(y), np.isinf(want)) and not np.isnan(y).any()
    on = np.isfinite(want)
    assert relerr(y[on], want[on]) <= 1e-5


def test_bias_gradient_keeps_the_bits_of_its_sum(ops):
    """Half a million pixels: an atomic per wave, one after the other on the channel, left the sums
    8.8e-7 from float64 in the norm, 4.2e-7 before that."""
    m = _t(workloads.gnomonic_kernel_map(256, 512).astype(np.float32))
    off = []
    for seed in range(12):     # (the atomics' order varies, and the error with it)
        gen = torch.Generator(device=DEV).manual_seed(seed)
        x, w, b, g = (torch.randn(s, generator=gen, device=DEV) for s in (
            (4, 3, 256, 512), (32, 3, 9), (32,), (4, 32, 256, 512)))
        gb = ops.mapped_conv_backward(g, m, None, x, w, b, 9, 1)[2].double()
        want = g.double().sum((0, 2, 3))
        off.append(float((gb - want).norm() / want.norm()))
    assert np.mean(off) <= 6.5e-7
