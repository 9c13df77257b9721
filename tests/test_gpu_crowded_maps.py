"""Maps that send many samples to one image element (a map that parks its invalid samples on one
pixel does): the lists of the inverted map grow as long as there are such samples, and what walks
or sorts them must neither go wrong nor take them one entry after the other.
"""
import time

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


def _crowded(rng, m, share):
    """m with a share of its samples on one spot."""
    return np.where(rng.random(m.shape[:-1] + (1,)) < share, np.float32([4.5, 3.5]), m).astype(np.float32)


def _seconds(step):
    """(first call on the map, later ones) of a step, GPU waited for."""
    times = []
    for _ in range(6):
        torch.cuda.synchronize()
        t = time.perf_counter()
        step()
        torch.cuda.synchronize()
        times.append(time.perf_counter() - t)
    return times[0], min(times[1:])


# share of 9 x 64 x 96 = 55296 samples: lists of a hundred entries, of a wave's sort (512), more,
# more than a workgroup sorts in LDS (6144), all samples
@pytest.mark.parametrize("share", [0.002, 0.008, 0.02, 0.1, 0.3, 1.0])
@pytest.mark.parametrize("Cin,Cout", [(8, 20), (72, 9)])
def test_convolutions_on_crowded_maps(ops, oracle, Cin, Cout, share):
    from _spherical_distortion_ext import _capi
    H, W, OH, OW, K = 24, 41, 64, 96, 9
    assert _capi.load().sdk_mapped_conv_by_columns(1, Cin, Cout, H, W, OH, OW, K, 0, 1,
                                                   _capi.SDK_F32, 0, 0) == 1
    rng = np.random.default_rng(int(1000 * share) + Cin)
    m = np.stack([rng.uniform(-1, W, (OH, OW, K)), rng.uniform(-1, H, (OH, OW, K))], -1)
    m = _crowded(rng, m, share)
    x = rng.standard_normal((1, Cin, H, W)).astype(np.float32)
    w = (rng.standard_normal((Cout, Cin, K)) / np.sqrt(Cin * K)).astype(np.float32)
    b, g = rng.standard_normal(Cout).astype(np.float32), rng.standard_normal((1, Cout, OH, OW)).astype(np.float32)
    bt = rng.standard_normal(Cin).astype(np.float32)
    runs = []
    for _ in range(2):       # two maps, two builds of their lists: the same sums
        tm = _t(m)
        gi, gw, _ = ops.mapped_conv_backward(_t(g), tm, None, _t(x), _t(w), _t(b), K, 1)
        yt = ops.mapped_transposed_conv_forward(_t(g), tm, None, _t(w), _t(bt), H, W, K, 1)
        runs.append((gi, gw, yt))
    assert torch.equal(runs[0][0], runs[1][0]) and torch.equal(runs[0][2], runs[1][2])
    wi, ww, _ = oracle.mapped_conv_backward(g, m, x, w, b, K, 1, None)
    assert relerr(gi.cpu().numpy(), wi) <= 1e-4 and relerr(gw.cpu().numpy(), ww) <= 1e-4
    assert relerr(yt.cpu().numpy(), oracle.mapped_transposed_conv_forward(g, m, w, bt, H, W, K, 1, None)) <= 1e-4


def test_a_crowded_map_does_not_stall_a_layer(ops):
    """64 -> 64 channels at 1 x 128 x 256, a tenth of the samples on one spot: one entry after the
    other, a step on kept lists took 17 times the even map's (an unsplit tile kernel's 1.6)."""
    m = workloads.gnomonic_kernel_map(128, 256).astype(np.float32)
    x, g = torch.randn(1, 64, 128, 256, device=DEV), torch.randn(1, 64, 128, 256, device=DEV)
    w, b = torch.randn(64, 64, 9, device=DEV) / 24, torch.randn(64, device=DEV)
    kept = []
    for share in (0.0, 0.0, 0.1):          # (the first warms up)
        tm = _t(_crowded(np.random.default_rng(1), m, share))
        kept.append(_seconds(lambda: ops.mapped_conv_backward(g, tm, None, x, w, b, 9, 1))[1])
    assert kept[2] <= 4 * kept[1]


def test_a_crowded_map_is_inverted_in_time(ops):
    """The first step on a map as above, its lists included: 17 times the even map's when one
    workgroup sorted lists of thirty thousand in memory."""
    m = workloads.gnomonic_kernel_map(128, 256).astype(np.float32)
    x, g = torch.randn(1, 64, 128, 256, device=DEV), torch.randn(1, 64, 128, 256, device=DEV)
    w, b = torch.randn(64, 64, 9, device=DEV) / 24, torch.randn(64, device=DEV)
    first = []
    for share in (0.0, 0.0, 0.1):          # (the first warms up)
        maps = [_t(_crowded(np.random.default_rng(i), m, share)) for i in range(3)]
        first.append(min(_seconds(lambda tm=tm: ops.mapped_conv_backward(g, tm, None, x, w, b, 9, 1))[0]
                         for tm in maps))
    assert first[2] <= 6 * first[1]
