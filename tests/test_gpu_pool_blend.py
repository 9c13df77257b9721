"""Blended pooling by row bands (csrc/pool_blend.hip) against the oracle: values to the last bit's
neighbourhood, indices equal, at every number of planes per pass, past LDS and off the route."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from _spherical_distortion_ext import _ops
    return _ops


# (H, W, OH, OW, K, rows a tap may stray), planes for half a million results: rows of 1, of 256 pooled
# pixels and one more (off the route); a band of several rows; rows so many that four, two, one plane
# or none fit LDS
SIZES = [
    (9, 8, 40, 1, 4, 0), (7, 9, 3, 5, 9, 1), (24, 50, 12, 25, 9, 2), (10, 300, 5, 256, 9, 2),
    (10, 300, 5, 257, 9, 2), (40, 128, 20, 64, 9, 39), (80, 256, 40, 128, 9, 79),
    (200, 256, 100, 128, 4, 199),
]


@pytest.mark.parametrize("interp", [1, 2])
@pytest.mark.parametrize("tc", SIZES, ids=lambda t: "x".join(map(str, t)))
def test_blended_pooling_matches_the_oracle(ops, oracle, tc, interp):
    H, W, OH, OW, K, stray = tc
    planes = (1 << 19) // (OH * OW) + 3
    rng = np.random.default_rng(sum(tc) + interp)
    oy = np.arange(OH)[:, None, None] * (H / OH) + rng.uniform(-stray, stray, (OH, OW, K)) - 0.5
    ox = np.arange(OW)[None, :, None] * (W / OW) + rng.uniform(-2, 2, (OH, OW, K))
    m = np.stack([ox, oy], -1).astype(np.float32)
    m[0, 0, :2] = np.round(m[0, 0, :2])         # integer positions: taps of weight zero
    m[-1, -1, 0] = (-50, -50)                   # no row of the image
    x = rng.standard_normal((1, planes, H, W)).astype(np.float32)
    tx, tm = torch.from_numpy(x).to(DEV), torch.from_numpy(m).to(DEV)
    v, i = ops.ops.mapped_max_pool(tx, tm, None, K, interp)
    a = ops.ops.mapped_avg_pool(tx, tm, None, K, interp)
    wv, wi = oracle.mapped_max_pool(x, m, K, interp)
    assert np.mean(i.cpu().numpy() != wi) <= 1e-3   # (ties but for one rounding)
    # the same products and sums in the same order; K + 3 roundings where a compiler contracts
    for have, want in ((v, wv), (a, oracle.mapped_avg_pool(x, m, K, interp))):
        np.testing.assert_allclose(have.cpu().numpy(), want, rtol=1e-6, atol=(K + 3) * 2.0 ** -23)
    # bit for bit what the per-pixel kernels give (one point per sample with weight one), also
    # with values that are not finite under taps of weight zero and beside them
    x[0, 0, H // 2, W // 2], x[0, 1, 0, 0], x[0, -1, -1, -1] = np.inf, np.nan, -np.inf
    tx, one = torch.from_numpy(x).to(DEV), torch.ones(tm.shape[:-1] + (1,), device=DEV)
    v, i = ops.ops.mapped_max_pool(tx, tm, None, K, interp)
    a = ops.ops.mapped_avg_pool(tx, tm, None, K, interp)
    v1, i1 = ops.ops.mapped_max_pool(tx, tm[..., None, :].contiguous(), one, K, interp)
    a1 = ops.ops.mapped_avg_pool(tx, tm[..., None, :].contiguous(), one, K, interp)
    assert torch.equal(i, i1) and torch.equal(v, v1)
    assert torch.equal(torch.nan_to_num(a, nan=7e9), torch.nan_to_num(a1, nan=7e9))
