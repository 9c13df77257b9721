"""The pair reads of the UV gather (csrc/mapped_gather_scatter.hip) at the edges of its textures, on values with one
right answer: integers, points at halves, so every product is a multiple of 1/4 and every sum a float32 number.
Compared to the bit."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    import _spherical_distortion_ext._ops as o
    return o


def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("interp", [0, 1, 2])
@pytest.mark.parametrize("size", [(1, 1), (3, 1), (1, 2), (2, 2), (4, 3), (5, 8)], ids=lambda s: "%dx%d" % s)
@pytest.mark.parametrize("planes", [1, 9, 35])
def test_uv_gather_at_the_edges(ops, oracle, planes, size, interp, dtype):
    TH, TW = size
    rng = np.random.default_rng(TH + 10 * TW + planes + interp)
    H, W, NT = 17, 33, 5
    quad = rng.integers(-1, NT + 1, (H, W))
    uv = (rng.integers(-4, 2 * np.array([TW, TH]) + 4, (H, W, 2)) / 2).astype(dtype)
    tex = rng.integers(-9, 10, (1, planes, NT, TH, TW)).astype(dtype)
    have = ops.ops.resample_from_uv_maps(_t(tex), _t(quad), _t(uv), interp).cpu().numpy()
    assert np.array_equal(have, oracle.resample_from_uv_maps(tex, quad, uv, interp))
