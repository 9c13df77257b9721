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


# (H, W, OH, OW, K, rows a tap may stray, planes per pass of the bands; None: off the route, 0: from
# global memory), planes for half a million results: rows of 1, of 256 pooled pixels and one more;
# a band of several rows; rows so many that four, two, one plane or none fit LDS
SIZES = [
    (9, 8, 40, 1, 4, 0, {4}), (7, 9, 3, 5, 9, 1, {4}), (24, 50, 12, 25, 9, 2, {4}),
    (10, 300, 5, 256, 9, 2, {4}), (10, 300, 5, 257, 9, 2, None), (40, 128, 20, 64, 9, 8, {2}),
    (40, 128, 20, 64, 4, 8, {2}), (80, 256, 40, 128, 9, 5, {2, 4}), (40, 128, 20, 64, 4, 16, {1, 2}),
    (80, 64, 40, 32, 4, 40, {1}), (40, 128, 20, 64, 9, 39, {1}), (80, 256, 40, 128, 9, 79, {0}),
    (200, 256, 100, 128, 4, 199, {0}),
]


def _planes_per_pass(m, H, W, interp):
    """What pool_blend_launch and its kernel choose for this map."""
    OH, OW = m.shape[:2]
    rows_of = lambda r: ((r * sy + 2 * sy + 2) * W + 1) * 16  # noqa: E731
    sy, lds, R = -(-H // OH), 52 * 1024, 1
    if OW > 256:
        return None
    while 2 * R * OW <= 256 and 2 * R <= OH and rows_of(2 * R) <= lds:
        R *= 2
    floats = min(rows_of(R), lds) // 4
    x, y = m[..., 0], m[..., 1]
    fx, fy = np.floor(x), np.floor(y)
    taps = []     # (row, is it read)
    for dy in (0, 1):
        for dx in (0, 1):
            w = (y - fy if dy else fy + 1 - y) * (x - fx if dx else fx + 1 - x)
            on = (w != 0) & (fy + dy >= 0) & (fy + dy < H)
            taps.append((fy + dy, on if interp == 2 else on & (fx + dx >= 0) & (fx + dx < W)))
    ways = set()
    for r in range(0, OH, R):
        rows = np.concatenate([row[r:r + R][on[r:r + R]] for row, on in taps])
        n = int(rows.max() - rows.min() + 1) * W if rows.size else 0
        ways.add(next((p for p in (4, 2, 1) if n < 65536 and (n + 1) * p <= floats), 0))
    return ways


@pytest.mark.parametrize("interp", [1, 2])
@pytest.mark.parametrize("tc", SIZES, ids=lambda t: "x".join(map(str, t[:6])))
def test_blended_pooling_matches_the_oracle(ops, oracle, tc, interp):
    H, W, OH, OW, K, stray, ways = tc
    planes = (1 << 19) // (OH * OW) + 3
    rng = np.random.default_rng(sum(tc[:6]) + interp)
    oy = np.arange(OH)[:, None, None] * (H / OH) + rng.uniform(-stray, stray, (OH, OW, K)) - 0.5
    ox = np.arange(OW)[None, :, None] * (W / OW) + rng.uniform(-2, 2, (OH, OW, K))
    m = np.stack([ox, oy], -1).astype(np.float32)
    m[0, 0, :2] = np.round(m[0, 0, :2])         # integer positions: taps of weight zero
    m[-1, -1, 0] = (-50, -50)                   # no row of the image
    assert _planes_per_pass(m, H, W, interp) == ways
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
