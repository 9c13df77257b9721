"""The texture gradient of UV resampling by texture (csrc/mapped_gather_scatter.hip,
uv_texture_scatter_kernel) on values with one right answer: integers, texture points at halves, so
every product is a multiple of 1/4 and every sum a float32 number.  Compared to the bit."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    import _spherical_distortion_ext._ops as o
    return o


# (batch, channels, textures, TH, TW, H, W): odd plane counts, one texture (its bucket shared among
# workgroups), more textures than threads of a workgroup, textures whose double sums are just in and
# just out of the LDS (8192 texels), buckets of less and more than one round of 1024 pixels (then
# taken by falling size)
SIZES = [(1, 1, 1, 1, 1, 1, 1), (2, 3, 5, 8, 9, 33, 47), (1, 13, 80, 16, 16, 60, 128),
         (1, 5, 1030, 4, 3, 40, 77), (1, 2, 3, 64, 128, 50, 90), (1, 3, 2, 91, 91, 64, 64),
         (3, 2, 1, 16, 16, 100, 120), (1, 3, 33, 5, 6, 180, 200)]
# by falling bucket size in chunks of two and of four planes, the last one ragged, and with more textures
# than threads of a workgroup; short buckets of large textures (workgroups of 512)
SIZES += [(1, 103, 20, 8, 8, 150, 160), (5, 41, 20, 8, 8, 150, 160), (1, 3, 1030, 4, 3, 1024, 1040),
          (1, 5, 320, 65, 70, 100, 110)]


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("interp", [0, 1, 2])
@pytest.mark.parametrize("tc", SIZES, ids=lambda t: "x".join(map(str, t)))
def test_texture_gradient(ops, oracle, tc, interp, dtype):
    B, C, NT, TH, TW, H, W = tc
    rng = np.random.default_rng(sum(tc) + interp)
    # runs of 1 to 70 neighbouring pixels on one point, over the rows of 16 lanes and the waves'
    # ends; some points and textures outside
    n = H * W
    length = rng.integers(1, 71, n)
    run = np.repeat(np.arange(n), length)[:n]
    quad = rng.integers(-1, NT + 1, n)[run].reshape(H, W)
    uv = (rng.integers(-4, 2 * np.array([TW, TH]) + 4, (n, 2)) / 2)[run].reshape(H, W, 2)
    uv = uv.astype(dtype)
    g = rng.integers(-3, 4, (B, C, H, W)).astype(dtype)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)  # noqa: E731
    have = ops.ops.resample_to_uv_maps(t(g), t(quad), t(uv), NT, TH, TW, interp).cpu().numpy()
    assert np.array_equal(have, oracle.resample_to_uv_maps(g, quad, uv, NT, TH, TW, interp))


def test_compiled_and_python_operators_agree(ops):
    if ops._native is None:
        pytest.skip("the compiled operator layer is not built")
    rng = np.random.default_rng(3)
    t = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    quad, uv = t(rng.integers(-1, 6, (20, 31))), t(rng.uniform(-1, 9, (20, 31, 2)))
    tex, g = t(rng.integers(-4, 5, (2, 3, 5, 8, 9)) * 1.0), t(rng.integers(-4, 5, (2, 3, 20, 31)) * 1.0)
    labels, vmap = t(rng.integers(0, 7, (2, 1, 20, 31))), t(rng.integers(0, 5, (20, 31, 2)))
    calls = {"resample_from_uv_maps": (tex, quad, uv, 1),
             "resample_to_uv_maps": (g, quad, uv, 5, 8, 9, 0),
             "voting_resample_to_map": (labels, vmap, 5, 5, 7)}
    for name, args in calls.items():
        assert getattr(ops, name) is getattr(ops.ops, name)
        assert torch.equal(getattr(ops.ops, name)(*args), ops.PYTHON_IMPL[name](*args))
        for i, a in enumerate(args):   # a tensor of another type, layout or shape: refused by both
            if not isinstance(a, torch.Tensor):
                continue
            for bad in (a.int(), a.transpose(-1, -2), a[:, :-1].contiguous(), a.cpu()):
                for fn in (getattr(ops.ops, name), ops.PYTHON_IMPL[name]):
                    if name == "resample_from_uv_maps" and i == 0 and bad.dim() == 5 and \
                            bad.is_cuda and bad.dtype == a.dtype and bad.is_contiguous():
                        continue   # (fewer channels are an ordinary call)
                    if name != "voting_resample_to_map" and i == 0 and bad.shape[2:] == a.shape[2:] \
                            and bad.is_cuda and bad.dtype == a.dtype:
                        continue
                    if name == "voting_resample_to_map" and i == 0 and bad.shape[1] == 0 and \
                            bad.is_cuda and bad.dtype == a.dtype:
                        continue
                    with pytest.raises(RuntimeError):
                        fn(*args[:i], bad, *args[i + 1:])
