"""Average unpooling of blended samples with its sources in LDS (unpool_spans_kernel), on values with
one right answer: integers, samples at halves, four samples a pooled pixel.  Compared to the bit with
the oracle, as is the forward of the same maps (pool_blend.hip)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# (batch, channels, H, W, OH, OW, map): spans of 512 elements with and without a remainder, plane
# chunks that are no multiple of eight, sources of a span that fit eight, four and two planes a pass
# (rows of 150, 500 and 1200 pooled pixels), lists of more than the kept entries, and maps whose
# spans or lists send a workgroup to memory
SIZES = [
    (1, 64, 9, 14, 4, 7, "strided"), (2, 35, 61, 300, 30, 150, "strided"),
    (3, 43, 40, 1000, 20, 500, "strided"), (1, 67, 16, 2400, 8, 1200, "strided"),
    (4, 48, 48, 100, 24, 50, "repeated"), (1, 70, 64, 120, 32, 60, "scrambled"),
    (2, 40, 64, 120, 32, 60, "one spot"), (1, 64, 80, 6000, 40, 3000, "scrambled"),
    # lists of more than the kept entries in a span that goes to memory
    (1, 64, 80, 6000, 40, 3000, "repeated, scrambled"),
    # planes of a workgroup: equal shares of all that are at work at once (13 planes), whole passes of
    # eight, of sixteen, and two passes at least where spans are many
    (1, 104, 128, 256, 64, 128, "strided"), (1, 67, 160, 320, 80, 160, "strided"),
    (1, 88, 160, 320, 80, 160, "strided"), (1, 67, 256, 513, 128, 256, "strided"),
]


@pytest.mark.parametrize("interp", [1, 2])
@pytest.mark.parametrize("tc", SIZES, ids=lambda t: "x".join(map(str, t)))
def test_against_the_oracle(oracle, tc, interp):
    import _spherical_distortion_ext._ops as ops
    B, C, H, W, OH, OW, kind = tc
    rng = np.random.default_rng(sum(tc[:6]) + interp)
    y, x, k = np.meshgrid(np.arange(OH), np.arange(OW), np.arange(4), indexing="ij")
    m = np.stack([x * 2.0 + k % 2, y * 2.0 + k // 2], -1)
    m += rng.integers(-1, 2, m.shape) * 0.5
    if kind.startswith("repeated"):   # a dozen pooled pixels on each element
        m[..., 0] = m[..., 0] // 12 * 12 + rng.integers(0, 2, m.shape[:-1])
    if kind.endswith("scrambled"):
        m = rng.permutation(m.reshape(-1, 2)).reshape(m.shape)
    if kind == "one spot":      # a list of hundreds of entries
        m[rng.random((OH, OW)) < 0.3] = (7.5, 3.0)
    m = m.astype(np.float32)
    g = rng.integers(-4, 5, (B, C, OH, OW)).astype(np.float32)
    f = rng.integers(-4, 5, (B, C, H, W)).astype(np.float32)
    t = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    tm = t(m)
    have = ops.ops.mapped_avg_unpool(t(g), tm, None, H, W, 4, interp).cpu().numpy()
    assert np.array_equal(have, oracle.mapped_avg_unpool(g, m, H, W, 4, interp))
    have = ops.ops.mapped_avg_pool(t(f), tm, None, 4, interp).cpu().numpy()
    assert np.array_equal(have, oracle.mapped_avg_pool(f, m, 4, interp))
