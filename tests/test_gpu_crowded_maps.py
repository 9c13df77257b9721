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


@pytest.mark.parametrize("share", [0.002, 0.02, 0.1, 0.3, 1.0])
@pytest.mark.parametrize("C,P,interp", [(3, 0, 1), (11, 0, 2), (2, 3, 1), (2, 2, 0), (1, 2, 2)])
def test_average_unpooling_of_crowded_maps(ops, oracle, C, P, interp, share):
    H, W, OH, OW, K = 24, 41, 48, 70, 9
    rng = np.random.default_rng(int(1000 * share) + C)
    shape = (OH, OW, K) + ((P,) if P else ())
    m = np.stack([rng.uniform(-1, W, shape), rng.uniform(-1, H, shape)], -1)
    m = _crowded(rng, m, share)
    iw = rng.uniform(0.1, 1, shape).astype(np.float32) if P else None
    g = rng.standard_normal((1, C, OH, OW)).astype(np.float32)
    got = [ops.mapped_avg_unpool(_t(g), _t(m), _t(iw), H, W, K, interp) for _ in range(2)]
    assert torch.equal(*got)             # two maps, two builds of their lists
    f64 = lambda a: None if a is None else a.astype(np.float64)  # noqa: E731
    want = oracle.mapped_avg_unpool(f64(g), f64(m), H, W, K, interp, f64(iw))
    mag = oracle.mapped_avg_unpool(np.abs(f64(g)), f64(m), H, W, K, interp, f64(iw))
    # n float32 additions of n terms each way (n: the samples on the spot at most, merged and then
    # summed): 2 n * 2^-24 of the sum of magnitudes would bound any order; the longest chain is 256
    # entries, or a wave's share of a list, and its tree
    chain = max(256, OH * OW * K * max(P, 1) // 64 + 70)
    assert np.all(np.abs(got[0].cpu().numpy() - want) <= chain * 2.0 ** -23 * mag + 4e-6 * np.abs(g).max())


def test_a_crowded_map_does_not_stall_average_pooling(ops):
    """2 x 16 planes of 256 x 512, stride 1, a tenth of the samples on one spot: 18 ms (the even
    map's 0.1) with one entry after the other, the first step, lists included, 78 ms (0.5)."""
    m = workloads.gnomonic_kernel_map(256, 512).astype(np.float32)
    g = torch.randn(2, 16, 256, 512, device=DEV)
    first, kept = [], []
    for share in (0.0, 0.0, 0.1):          # (the first warms up)
        maps = [_t(_crowded(np.random.default_rng(i), m, share)) for i in range(3)]
        runs = [_seconds(lambda tm=tm: ops.mapped_avg_unpool(g, tm, None, 256, 512, 9, 1)) for tm in maps]
        first.append(min(r[0] for r in runs))
        kept.append(min(r[1] for r in runs))
    print("first", first, "kept", kept)
    assert kept[2] <= 25 * kept[1] and first[2] <= 40 * first[1]


@pytest.mark.parametrize("share", [0.03, 0.1, 0.6])
def test_products_gathered_on_crowded_maps(ops, oracle, share):
    """Up-sampling layers of nearest taps gather their products through the same lists."""
    H, W, OH, OW, K, Cin, Cout = 96, 129, 48, 64, 9, 12, 24
    rng = np.random.default_rng(int(100 * share))
    m = np.stack([rng.uniform(-1, W, (OH, OW, K)), rng.uniform(-1, H, (OH, OW, K))], -1)
    m = _crowded(rng, m, share)
    x = rng.standard_normal((2, Cout, OH, OW)).astype(np.float32)
    w = (rng.standard_normal((Cout, Cin, K)) / np.sqrt(Cin * K)).astype(np.float32)
    b = rng.standard_normal(Cin).astype(np.float32)
    y = [ops.mapped_transposed_conv_forward(_t(x), _t(m), None, _t(w), _t(b), H, W, K, 0) for _ in range(2)]
    assert torch.equal(*y)
    want = oracle.mapped_transposed_conv_forward(x, m, w, b, H, W, K, 0, None)
    assert relerr(y[0].cpu().numpy(), want) <= 1e-4
