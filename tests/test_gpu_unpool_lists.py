"""Average unpooling of blended and weighted samples as a gather over merged lists
(unpool_lists_kernel, csrc/mapped_gather_scatter.hip) against the oracle in float64."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from _spherical_distortion_ext import _ops
    return _ops


# (B, C, H, W, OH, OW, K, P, interp): odd planes around the planes of a thread, one pixel, maps whose
# entries merge, and one that sends every sample to one image element
@pytest.mark.parametrize("tc", [
    (1, 1, 1, 1, 1, 1, 1, 0, 1), (1, 3, 9, 14, 5, 7, 9, 0, 1), (2, 9, 17, 31, 17, 31, 9, 0, 2),
    (1, 5, 12, 20, 6, 10, 4, 3, 1), (3, 6, 12, 20, 12, 20, 7, 4, 0), (1, 33, 260, 256, 130, 128, 9, 0, 1),
    (1, 4, 6, 8, 20, 30, 9, 0, -1),
], ids=lambda t: "x".join(map(str, t)))
def test_average_unpooling_from_lists_matches_the_oracle(ops, oracle, tc):
    B, C, H, W, OH, OW, K, P, interp = tc
    rng = np.random.default_rng(sum(tc))
    shape = (OH, OW, K) + ((P,) if P else ())
    up = (1,) * (len(shape) - 2)
    oy = np.arange(OH).reshape(-1, 1, *up) * (H / OH) + rng.uniform(-1.5, 1.5, shape)
    ox = np.arange(OW).reshape(1, -1, *up) * (W / OW) + rng.uniform(-1.5, 1.5, shape)
    m = np.stack([ox, oy], -1).astype(np.float32)
    if interp < 0:
        m[:], interp = (2.25, 3.5), 1
    iw = rng.uniform(0.1, 1, shape).astype(np.float32) if P else None
    g = rng.standard_normal((B, C, OH, OW)).astype(np.float32)
    t = lambda a: None if a is None else torch.from_numpy(a).to(DEV)  # noqa: E731
    tm, tw = t(m), t(iw)
    got = ops.ops.mapped_avg_unpool(t(g), tm, tw, H, W, K, interp)
    assert torch.equal(got, ops.ops.mapped_avg_unpool(t(g), tm, tw, H, W, K, interp))
    assert torch.equal(got, ops.PYTHON_IMPL["mapped_avg_unpool"](t(g), tm, tw, H, W, K, interp))
    want = oracle.mapped_avg_unpool(g.astype(np.float64), m.astype(np.float64), H, W, K, interp,
                                    None if iw is None else iw.astype(np.float64))
    # n float32 additions of n terms: n * 2^-24 of the sum of magnitudes, n at most the samples a
    # pixel receives (5400 where all meet in one), the weights' own rounding beside it
    n = 5400 if OH > H else 64
    mag = oracle.mapped_avg_unpool(np.abs(g).astype(np.float64), m.astype(np.float64), H, W, K, interp,
                                   None if iw is None else iw.astype(np.float64))
    assert np.all(np.abs(got.cpu().numpy() - want) <= n * 2.0 ** -24 * mag + 4e-6 * np.abs(g).max())
