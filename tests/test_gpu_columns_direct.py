"""Small calls whose columns are blended on the way to LDS (csrc/conv_columns_direct.hip), against the
oracle."""
import numpy as np
import pytest
import torch

import test_gpu_columns as columns
from conftest import runs_by_columns

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    import _spherical_distortion_ext._ops as o
    return o


@pytest.fixture(scope="module")
def oracle():
    from oracle import oracle as o
    return o


# (batch, Cin, Cout, H, W, OH, OW, K, P, interp), as in test_gpu_columns: every number of channel
# blocks a tile may have and one over (32 .. 161 channels), tiles of one pixel and one over 32
# pixels, one and several groups and splits of the reduction (K * Cin of 32 steps and more on few
# tiles), runs of samples that share no table of taps (25 samples, weighted samples of up to 16
# taps, channel counts whose steps and tiles of 32 straddle samples), calls with more tiles than XCDs'
# shares, and one with more strips of pixels than a wave of the weight gradient's sums adds up
SIZES = [
    (1, 8, 32, 6, 9, 3, 11, 9, 0, 1),
    (1, 40, 33, 6, 9, 3, 11, 9, 0, 2),
    (2, 24, 96, 9, 14, 7, 13, 9, 0, 1),
    (1, 33, 97, 9, 14, 8, 8, 9, 0, 0),
    (1, 16, 160, 9, 14, 8, 9, 4, 0, 1),
    (1, 16, 161, 9, 14, 8, 9, 4, 0, 0),
    (1, 72, 64, 9, 14, 4, 8, 25, 0, 1),
    (2, 130, 40, 9, 14, 5, 7, 25, 0, 2),
    (1, 64, 128, 9, 14, 5, 7, 25, 0, 0),
    (1, 8, 16, 9, 14, 5, 7, 25, 4, 1),
    (2, 40, 24, 9, 14, 5, 7, 9, 4, 2),
    (1, 21, 24, 9, 14, 5, 7, 25, 3, 0),
    (1, 96, 48, 9, 14, 5, 7, 25, 2, 1),
    (3, 12, 20, 40, 80, 40, 80, 9, 0, 1),
    (1, 16, 64, 64, 128, 64, 128, 9, 4, 1),
    (4100, 8, 8, 4, 4, 2, 2, 1, 0, 1),
    (5, 24, 70, 20, 31, 17, 31, 9, 2, 2),
    # ... six to eleven blocks, nine with few columns and with many; five of fewer steps than 24 and of as many
    (1, 16, 192, 9, 14, 8, 9, 9, 0, 1),
    (2, 16, 200, 9, 14, 8, 9, 9, 0, 2),
    (1, 24, 288, 9, 14, 8, 9, 9, 0, 1),
    (1, 96, 257, 9, 14, 8, 9, 25, 0, 1),
    (1, 24, 290, 9, 14, 8, 9, 9, 4, 1),
    (1, 24, 330, 9, 14, 8, 9, 9, 0, 0),
    (1, 88, 160, 9, 14, 8, 9, 9, 0, 2),
    (1, 80, 131, 9, 14, 8, 9, 9, 0, 1),
]


@pytest.mark.parametrize("mode", ["native", "split", "bf16"])
@pytest.mark.parametrize("tc", SIZES, ids=lambda t: "x".join(map(str, t)))
def test_contractions_match_the_oracle(ops, oracle, tc, mode):
    from _spherical_distortion_ext import _capi
    B, Cin, Cout, H, W, OH, OW, K, P, interp = tc
    assert _capi.load().sdk_mapped_conv_by_columns(B, Cin, Cout, H, W, OH, OW, K, P, interp,
                                                   _capi.SDK_F32, 0, 0) == 1
    m, iw, x, w, b, g, _ = columns._arrays(tc)
    t = lambda a: None if a is None else torch.from_numpy(a).to(DEV)  # noqa: E731
    odd = torch.empty(m.size + 1, device=DEV)[1:].view(m.shape).copy_(t(m))   # 4 bytes off a pair's place
    want = oracle.mapped_conv_forward(x, m, w, b, K, interp, iw)
    # float32: sums of at most K * Cin terms of random signs, eps * sqrt(n) < 5e-6; bf16 operands: 2^-9 each
    tol = 4e-3 if mode == "bf16" else 5e-6
    with ops.conv_compute(mode):
        y = ops.ops.mapped_conv_forward(t(x), t(m), t(iw), t(w), t(b), K, interp)
        again = ops.ops.mapped_conv_forward(t(x), odd, t(iw), t(w), t(b), K, interp)
        grads = ops.ops.mapped_conv_backward(t(g), t(m), t(iw), t(x), t(w), t(b), K, interp)
        weights_alone = ops.ops.mapped_conv_backward_select(t(g), t(m), t(iw), t(x), t(w), K, interp,
                                                            False, False, True)
    assert columns._rel(y.cpu().numpy(), want) <= tol
    assert torch.equal(y, again)
    for have, want in zip(grads, oracle.mapped_conv_backward(g, m, x, w, b, K, interp, iw)):
        assert columns._rel(have.cpu().numpy(), want) <= tol
    assert torch.equal(weights_alone[1], grads[1])
    # (a bias gradient of many strips is added up by atomics, in any order)
    assert columns._rel(weights_alone[2].cpu().numpy(), grads[2].cpu().numpy()) <= 5e-6


@pytest.mark.parametrize("height", [64, 128])
def test_bias_gradient_keeps_the_bits_of_its_sums(ops, height):
    """8 x 512 strips of 64 pixels a channel, the most that are added up here: in a float32 chain they were 1.8e-7
    from float64 in the norm, the sums of before 1.4e-7.  A strip is a tree of six float32 additions and the result is
    rounded once: 2^-24 * sqrt(7 / 3) = 0.9e-7 for random signs, on 128 channels within a fifth."""
    tc = (8, 8, 128, 8, 16, height, 256, 2, 0, 1)
    assert runs_by_columns(*tc)
    m, _, x, w, b, g, _ = columns._arrays(tc)
    t = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    gb = ops.ops.mapped_conv_backward(t(g), t(m), None, t(x), t(w), t(b), 2, 1)[2]
    assert columns._rel(gb.cpu().numpy(), g.astype(np.float64).sum((0, 2, 3))) <= 1.1e-7


def _gradients(ops, tc, arrays, mode):
    m, _, x, w, b, g, _ = arrays
    with ops.conv_compute(mode):
        return ops.ops.mapped_conv_backward(g, m, None, x, w, b, tc[7], tc[9])


def _on_gpu(tc):
    return [None if a is None else torch.from_numpy(a).to(DEV) for a in columns._arrays(tc)]


# (..., as above) whose scatter has slices of two elements and one; slices of one, in three chunks of channels, the
# last of six; whose pixels' operands are laid out by each contraction (float32 and split), those of the weight
# gradient in two slices (split)
LARGE = [
    (3, 32, 8, 40, 80, 100, 200, 25, 0, 1),
    (2, 70, 8, 40, 80, 144, 288, 25, 0, 1),
    (32, 8, 192, 64, 128, 64, 128, 7, 0, 1),
    (2, 40, 208, 40, 80, 144, 288, 11, 0, 0),
]


@pytest.mark.parametrize("kept", [True, False], ids=["plan", "no-plan"])
@pytest.mark.parametrize("mode", ["native", "split", "bf16"])
@pytest.mark.parametrize("tc", LARGE, ids=lambda t: "x".join(map(str, t)))
def test_calls_in_slices(ops, tc, mode, kept):
    B, Cin, Cout, H, W, OH, OW, K, P, interp = tc
    assert runs_by_columns(*tc)
    arrays = m, _, x, w, b, g, bt = _on_gpu(tc)
    ops.set_conv_plan_cache(kept)
    try:
        gi, gw, gb = _gradients(ops, tc, arrays, mode)
        # a call of one element, and of one chunk of channels, whose sums are the same ones
        for at in (0, B - 1):
            one = (m, None, x[at:at + 1].contiguous(), w, b, g[at:at + 1].contiguous(), None)
            assert torch.equal(gi[at:at + 1], _gradients(ops, tc, one, mode)[0])
        if Cin == 70:
            with ops.conv_compute(mode):
                up = ops.ops.mapped_transposed_conv_forward(g, m, None, w, x.new_ones(Cin), H, W, K, interp)
            for c in (slice(0, 32), slice(32, 64), slice(64, 70)):
                part = (m, None, x[:, c].contiguous(), w[:, c].contiguous(), b, g, None)
                assert torch.equal(gi[:, c], _gradients(ops, tc, part, mode)[0])
                assert torch.equal(gi[:, c] + 1, up[:, c])
    finally:
        ops.set_conv_plan_cache(True)
    want = _gradients(ops, tc, [None if a is None else a.double() for a in arrays], "native")
    # float32 sums: eps * sqrt(n) / 2, apart by 64 channels or 32 pixels; bf16 operands: 2^-9 each
    for have, ref in zip((gi, gw, gb), want):
        assert columns._rel(have.cpu().numpy(), ref.cpu().numpy()) <= (4e-3 if mode == "bf16" else 2e-6)


@pytest.mark.parametrize("mode", ["native", "split", "bf16"])
def test_gradients_of_values_no_tap_reads_stay_out(ops, mode):
    """An infinite pixel of the image without a tap, an infinite value of the gradient and an infinite weight reach
    what is summed from them and nothing else."""
    tc = (1, 12, 40, 9, 14, 5, 7, 9, 0, 0)
    arrays = m, _, x, w, b, g, _ = _on_gpu(tc)
    m[..., 0].clamp_(0, 12)
    x[0, :, :, 13] = 0
    gi, gw, gb = _gradients(ops, tc, arrays, mode)
    x[0, :, :, 13] = float("inf")
    for have, want in zip(_gradients(ops, tc, arrays, mode), (gi, gw, gb)):
        assert torch.equal(have, want)
    x[0, :, :, 13] = 0
    kept, g[0, 7, 2, 3] = g[0, 7, 2, 3].item(), float("inf")
    hi, hw, hb = _gradients(ops, tc, arrays, mode)
    rest = [n for n in range(40) if n != 7]
    assert torch.equal(hw[rest], gw[rest]) and torch.equal(hb[rest], gb[rest])
    assert not torch.isfinite(hb[7]) and not torch.isfinite(hw[7]).all()
    at = (m[2, 3] + 0.5).floor().long()     # (the samples' pixels; no coordinate is a half)
    at = at[(at[:, 1] >= 0) & (at[:, 1] < 9)]
    reached = torch.zeros(9, 14, dtype=torch.bool, device=DEV)
    reached[at[:, 1], at[:, 0]] = True
    assert torch.equal(hi[0][:, ~reached], gi[0][:, ~reached])
    assert not torch.isfinite(hi[0][:, reached]).any()
    g[0, 7, 2, 3], w[7, 3, 2] = kept, float("inf")
    hi, hw, hb = _gradients(ops, tc, arrays, mode)
    assert torch.equal(hw, gw) and torch.equal(hb, gb)
    rest = [c for c in range(12) if c != 3]
    assert torch.equal(hi[:, rest], gi[:, rest]) and not torch.isfinite(hi[:, 3]).all()


@pytest.mark.parametrize("Cin", [8, 48, 64, 96, 97])
@pytest.mark.parametrize("Cout", [64, 66, 112])
@pytest.mark.parametrize("mode", ["native", "split", "bf16"])
def test_wide_layers_of_one_sample(ops, mode, Cout, Cin):
    """31.5, 32.5 and 55 MB of pixels: forwards (up to 48 channels, from 32 MB) and backwards (up to 96, from 54) with
    their columns in memory and without."""
    tc = (15, Cin, Cout, 12, 24, 67, 128, 1, 0, 1)
    assert runs_by_columns(*tc)
    arrays = m, _, x, w, b, g, bt = _on_gpu(tc)
    with ops.conv_compute(mode):
        have = [ops.ops.mapped_conv_forward(x, m, None, w, b, 1, 1), *_gradients(ops, tc, arrays, mode)]
    m, x, w, b, g = (a.double() for a in (m, x, w, b, g))
    want = [ops.ops.mapped_conv_forward(x, m, None, w, b, 1, 1), *ops.ops.mapped_conv_backward(g, m, None, x, w, b, 1, 1)]
    for h, ref in zip(have, want):
        assert columns._rel(h.cpu().numpy(), ref.cpu().numpy()) <= (4e-3 if mode == "bf16" else 2e-6)


@pytest.mark.parametrize("mode", ["native", "split", "bf16"])
def test_values_no_tap_reads_stay_out(ops, mode):
    """An infinite pixel without a tap, and an infinite weight of a channel beside the others."""
    tc = (1, 12, 40, 9, 14, 5, 7, 9, 0, 0)
    m, _, x, w, b, _, _ = columns._arrays(tc)
    m[..., 0] = m[..., 0].clip(0, 12)
    x[0, :, :, 13] = float("inf")
    t = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    with ops.conv_compute(mode):
        y = ops.ops.mapped_conv_forward(t(x), t(m), None, t(w), t(b), 9, 0)
        clean = x.copy()
        clean[0, :, :, 13] = 0
        want = ops.ops.mapped_conv_forward(t(clean), t(m), None, t(w), t(b), 9, 0)
        assert torch.equal(y, want)
        w[7, 3, 2] = float("inf")
        y = ops.ops.mapped_conv_forward(t(clean), t(m), None, t(w), t(b), 9, 0)
    rest = [n for n in range(40) if n != 7]
    assert torch.equal(y[:, rest], want[:, rest])
    assert not torch.isfinite(y[:, 7]).all()
