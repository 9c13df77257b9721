"""The LDS-window convolution kernels (csrc/conv_window_*.hip) on values
whose every product and sum is a float32 number, rounded to bf16 or not: integers of at most four
bits and sample positions at halves, so blended values are multiples of 1/4 below 2^6 and sums stay
below 2^24 quarters.  Every arithmetic then has one right answer, the oracle's, to the bit."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# (batch, Cin, Cout, H, W, OH, OW, K, interp, points): channels around a chunk of 32, rows around the
# 32, 64 and 128 a workgroup multiplies, widths no multiple of 4 or of a tile's 16 pixels, every way
# the samples are shared among the waves (K % 4, K = 10 in eight waves), single-row plans, more than
# four rows a sample, tiles inside their window and (strided, scattered samples) big ones
SIZES = [
    (1, 5, 65, 9, 20, 9, 20, 9, 1, 0),
    (2, 32, 128, 17, 33, 17, 33, 9, 1, 0),
    (1, 33, 130, 16, 32, 16, 32, 10, 2, 0),
    (1, 70, 96, 10, 19, 10, 19, 7, 0, 0),
    (2, 40, 72, 48, 96, 24, 48, 9, 1, 0),
    (1, 64, 100, 40, 80, 20, 40, 4, 2, 0),
    (1, 37, 66, 12, 24, 12, 24, 1, 1, 0),
    (1, 34, 68, 8, 11, 8, 11, 2, 1, 0),
    (1, 8, 80, 9, 16, 9, 16, 3, 0, 2),
    (2, 31, 33, 14, 18, 14, 18, 5, 1, 0),
    (1, 36, 127, 16, 40, 16, 40, 6, 2, 0),
    (1, 64, 66, 24, 40, 12, 20, 8, 0, 2),
    (3, 20, 129, 32, 64, 32, 64, 9, 0, 2),
    # big tiles whose samples do not halve among the two groups of waves
    (1, 34, 100, 48, 96, 12, 24, 1, 1, 0),
    (1, 34, 70, 48, 96, 12, 24, 3, 2, 0),
    (2, 40, 40, 48, 96, 12, 24, 5, 0, 0),
    # at most 64 rows: two row blocks, each with half of the pixels in two waves
    (1, 33, 1, 9, 20, 9, 20, 3, 1, 0),
    (2, 5, 32, 17, 33, 17, 33, 4, 2, 0),
    (1, 40, 33, 48, 96, 24, 48, 9, 1, 0),
    (2, 70, 64, 48, 96, 24, 48, 10, 2, 0),
    (1, 32, 64, 40, 80, 20, 40, 7, 0, 0),
    (1, 64, 63, 24, 40, 12, 20, 6, 0, 2),
    (1, 20, 40, 12, 9, 12, 9, 2, 0, 0),
]


def _arrays(tc):
    B, Cin, Cout, H, W, OH, OW, K, interp, P = tc
    rng = np.random.default_rng(sum(tc))
    side = int(np.ceil(np.sqrt(K)))
    k = np.arange(K)
    ys = np.arange(OH)[:, None, None] * (H / OH) + (k // side - 1) * 1.5
    xs = np.arange(OW)[None, :, None] * (W / OW) + (k % side - 1) * 1.5
    ys, xs = (np.broadcast_to(a, (OH, OW, K)) + rng.integers(-1, 2, (OH, OW, K)) * 0.5
              for a in (ys, xs))
    ys = np.round(ys * 2) / 2
    xs = np.round(xs * 2) / 2 % W
    iw = None
    if P:
        ys, xs = (np.stack([a + p for p in range(P)], -1) for a in (np.floor(ys), np.floor(xs)))
        iw = np.broadcast_to(np.array([0.5, 0.25, 0.25, 0.5][:P]), ys.shape).astype(np.float32).copy()
    m = np.stack([xs, ys], -1).astype(np.float32)
    f = lambda *s: rng.integers(-4, 5, s).astype(np.float32)  # noqa: E731
    return m, iw, f(B, Cin, H, W), f(Cout, Cin, K), f(Cout), f(B, Cout, OH, OW)


@pytest.mark.parametrize("mode", ["native", "split", "bf16"])
@pytest.mark.parametrize("tc", SIZES, ids=lambda t: "x".join(map(str, t)))
def test_exact_values(oracle, tile_kernels, tc, mode):
    import _spherical_distortion_ext._ops as ops
    K, interp = tc[7], tc[8]
    m, iw, x, w, b, g = _arrays(tc)
    t = lambda a: None if a is None else torch.from_numpy(a).to(DEV)  # noqa: E731
    tx, tm, tiw, tw, tb, tg = map(t, (x, m, iw, w, b, g))
    with ops.conv_compute(mode):
        y = ops.ops.mapped_conv_forward(tx, tm, tiw, tw, tb, K, interp)
        gi, gw, gb = ops.ops.mapped_conv_backward(tg, tm, tiw, tx, tw, tb, K, interp)
    assert np.array_equal(y.cpu().numpy(), oracle.mapped_conv_forward(x, m, w, b, K, interp, iw))
    wi, ww, wb = oracle.mapped_conv_backward(g, m, x, w, b, K, interp, iw)
    for have, want in ((gi, wi), (gw, ww), (gb, wb)):
        assert np.array_equal(have.cpu().numpy(), want)


# Batches so large that a workgroup of the weight gradient takes two or three tiles of the list after one
# another (one of eight groups a batch element; 20, 15 and 9 tiles, the last ones of fewer pixels and with
# windows of another size): four waves and two, eight waves (ten samples, big tiles), every remainder of
# K by 4, one row a sample and four
TURNS = [
    (64, 5, 40, 40, 60, 40, 60, 9, 1, 0), (64, 5, 40, 40, 60, 40, 60, 7, 0, 0),
    (64, 6, 66, 24, 72, 24, 72, 9, 1, 0), (64, 5, 66, 40, 60, 40, 60, 7, 0, 0),
    (64, 5, 66, 24, 72, 24, 72, 6, 2, 0), (64, 5, 33, 24, 72, 24, 72, 8, 1, 0),
    (64, 5, 70, 40, 60, 40, 60, 10, 0, 0), (64, 5, 66, 24, 72, 24, 72, 10, 1, 0),
    (64, 5, 33, 40, 60, 40, 60, 10, 1, 0), (64, 5, 66, 96, 192, 24, 48, 9, 1, 0),
    (64, 5, 40, 96, 192, 24, 48, 7, 0, 0), (64, 5, 66, 96, 192, 24, 48, 10, 0, 0),
    (64, 5, 40, 96, 192, 24, 48, 10, 1, 0),
]


@pytest.mark.parametrize("tc", TURNS, ids=lambda t: "x".join(map(str, t)))
def test_weight_gradient_over_several_tiles(oracle, tile_kernels, tc):
    import _spherical_distortion_ext._ops as ops
    K, interp = tc[7], tc[8]
    m, _, x, w, b, g = _arrays(tc)
    t = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    want = oracle.mapped_conv_backward(g, m, x, w, b, K, interp, None)[1]
    for mode in ("native", "split", "bf16"):
        with ops.conv_compute(mode):
            gw = ops.ops.mapped_conv_backward_select(t(g), t(m), None, t(x), t(w), K, interp, False,
                                                     False, True)[1]
        assert np.array_equal(gw.cpu().numpy(), want), mode


# several batch elements and channel tiles over lists that are shorter than their launch and no multiple
# of 8: windows of every form (contraction with wide, 64 and 32 rows, product form in the strided ones)
SHARES = [
    (3, 20, 257, 40, 72, 40, 72, 9, 1, 0),
    (5, 257, 33, 17, 33, 17, 33, 9, 1, 0),
    (3, 130, 64, 48, 96, 24, 48, 9, 1, 0),
    (7, 9, 130, 9, 16, 9, 16, 4, 0, 0),
]


@pytest.mark.parametrize("mode", ["native", "split", "bf16"])
@pytest.mark.parametrize("tc", SHARES, ids=lambda t: "x".join(map(str, t)))
def test_every_tile_of_every_batch_element_is_written_once(oracle, tile_kernels, tc, mode):
    import _spherical_distortion_ext._ops as ops
    K, interp = tc[7], tc[8]
    m, _, x, w, b, g = _arrays(tc)
    tx, tm, tw, tb, tg = (torch.from_numpy(a).to(DEV) for a in (x, m, w, b, g))
    with ops.conv_compute(mode):
        y = ops.ops.mapped_conv_forward(tx, tm, None, tw, tb, K, interp)
        gi = ops.ops.mapped_conv_backward(tg, tm, None, tx, tw, tb, K, interp)[0]
    np.testing.assert_array_equal(y.cpu().numpy(), oracle.mapped_conv_forward(x, m, w, b, K, interp))
    np.testing.assert_array_equal(gi.cpu().numpy(), oracle.mapped_conv_backward(g, m, x, w, b, K, interp)[0])


@pytest.mark.parametrize("mode", ["native", "split", "bf16"])
def test_values_that_are_not_finite_stay_where_they_are(tile_kernels, mode):
    """An infinite pixel reaches the outputs and weights that read it and no others (padding of
    plans, channels and rows multiplies zeros by zeros)."""
    import _spherical_distortion_ext._ops as ops
    tc = (1, 33, 70, 16, 36, 16, 36, 9, 1, 0)
    m, _, x, w, b, g = _arrays(tc)
    w[w == 0], g[g == 0] = 1, 1
    x[0, 32, 5, 7] = np.inf
    m[..., 0] = np.minimum(np.abs(m[..., 0]), 34)
    t = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    with ops.conv_compute(mode):
        y = ops.ops.mapped_conv_forward(t(x), t(m), None, t(w), t(b), 9, 1).cpu().numpy()
        gw = ops.ops.mapped_conv_backward(t(g), t(m), None, t(x), t(w), t(b), 9, 1)[1].cpu().numpy()
    reads = ((np.abs(m[..., 0] - 7) < 1) & (np.abs(m[..., 1] - 5) < 1)).any(-1)
    assert np.array_equal(~np.isfinite(y[0]).all(0), reads)
    assert np.isfinite(gw[:, :32]).all() and not np.isfinite(gw[:, 32]).all()


@pytest.mark.parametrize("mode", ["native", "split"])
def test_more_than_two_gigabytes_of_weights(tile_kernels, mode):
    """The last output channel's row of a weight tensor past 2^31 bytes, integers as above."""
    import _spherical_distortion_ext._ops as ops
    C, K, H, W = 7744, 9, 8, 16
    rng = np.random.default_rng(7)
    x = torch.from_numpy(rng.integers(-4, 5, (1, C, H, W)).astype(np.float32)).to(DEV)
    row = torch.from_numpy(rng.integers(-4, 5, (C, K)).astype(np.float32)).to(DEV)
    at = torch.from_numpy(rng.integers(0, H * W, (H, W, K))).to(DEV)
    w = torch.zeros(C, C, K, device=DEV)
    assert w.numel() * 4 > 2 ** 31
    w[-1] = row
    m = torch.stack([at % W, at // W], -1).float().contiguous()
    with ops.conv_compute(mode):
        y = ops.ops.mapped_conv_forward(x, m, None, w, torch.zeros(C, device=DEV), K, 0)
    want = (x.flatten(2)[0][:, at].double() * row.double()[:, None, None, :]).sum((0, 3))
    assert torch.equal(y[0, -1].double(), want)
    assert not y[0, :-1].any()


@pytest.mark.parametrize("mode", ["native", "split", "bf16"])
@pytest.mark.parametrize("tc", [(66, 4096, 4104, 2, 1), (66, 4097, 4099, 1, 0), (40, 4096, 4104, 3, 0)],
                         ids=lambda t: "x".join(map(str, t)))
def test_weight_gradient_of_more_than_2_24_pixels(oracle, tile_kernels, tc, mode):
    """Planes of which 32 are more than 2^31 bytes; 16-byte reads and, on an odd width, single ones;
    the window kernels take such a layer (they leave their sums in a workspace with room for them)."""
    import _spherical_distortion_ext._ops as ops
    from _spherical_distortion_ext import _capi
    Cout, OH, OW, K, interp = tc
    Cin, H, W = 8, 64, 96
    assert OH * OW > 2 ** 24
    rng = np.random.default_rng(sum(tc))
    k = np.arange(K)
    y, x = torch.arange(OH, device=DEV) * H // OH, torch.arange(OW, device=DEV) * W // OW
    m = torch.stack([x.expand(OH, OW)[..., None] + torch.from_numpy(k % 2 * 0.5).to(DEV),
                     y[:, None].expand(OH, OW)[..., None] - torch.from_numpy(k // 2 * 0.5).to(DEV)], -1)
    m = m.float().contiguous()
    # gradients at some pixels, the corners among them: few enough for the oracle, and the sums exact
    at = np.unique(np.concatenate([rng.integers(0, OH * OW, 4000),
                                   [0, OW - 1, (OH - 1) * OW, OH * OW - 1, 2 ** 24 - 1, 2 ** 24]]))
    values = rng.integers(-4, 5, (1, Cout, at.size)).astype(np.float32)
    g = torch.zeros(1, Cout, OH, OW, device=DEV)
    tat = torch.from_numpy(at).to(DEV)
    g.view(1, Cout, -1)[..., tat] = torch.from_numpy(values).to(DEV)
    img = rng.integers(-4, 5, (1, Cin, H, W)).astype(np.float32)
    w = np.zeros((Cout, Cin, K), np.float32)
    t = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    with ops.conv_compute(mode):
        _, gw, gb = ops.ops.mapped_conv_backward_select(g, m, None, t(img), t(w), K, interp, False,
                                                        False, True)
    few = m.view(1, -1, K, 2)[:, tat].cpu().numpy()
    _, want, wb = oracle.mapped_conv_backward(values[:, :, None], few, img, w,
                                              np.zeros(Cout, np.float32), K, interp, None)
    assert np.array_equal(gw.cpu().numpy(), want)
    assert np.array_equal(gb.cpu().numpy(), wb)
