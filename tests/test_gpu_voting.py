"""Voting resample: the LDS kernels of coherent maps and the histogram behind them
(csrc/voting_resample.hip) against the oracle, label by label."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _call(labels, vmap, oh, ow, nc, ws_bytes=None):
    from _spherical_distortion_ext import _capi, _ops
    t, m = torch.from_numpy(labels).to(DEV), torch.from_numpy(vmap).to(DEV)
    if ws_bytes is None:
        return _ops.voting_resample_to_map(t, m, oh, ow, nc).cpu().numpy()
    B, C, IH, IW = labels.shape
    out = torch.full((B, C, oh, ow), -1, dtype=torch.int64, device=DEV)
    ws = torch.full((ws_bytes,), 255, dtype=torch.uint8, device=DEV)
    _capi.call("sdk_voting_resample_to_map", _ops._ptr(t), _ops._ptr(m), _ops._ptr(out),
               _ops._ptr(ws), ws_bytes, B, C, IH, IW, oh, ow, nc, _ops._stream(t))
    return out.cpu().numpy()


def _coherent(ih, iw, oh, ow):
    y, x = np.mgrid[:ih, :iw]
    m = np.stack([x * ow // iw, y * oh // ih], -1).astype(np.int64)
    m[::7, ::5] = (-1, 3)                  # targets outside the output, on every side
    m[3::11, 2::13] = (ow, 0)
    m[1::9, ::17] = (0, oh + 70000)
    m[5::23, 1::19] = (ow + 5, oh - 1)     # past the edge, inside the last workgroup's square
    return m


# (batch, IH, IW, OH, OW, classes): input tiles of 16 x 16 and cell squares of 16, 8 and 4 with
# and without remainders, one pixel, one cell, each square's last number of classes and the next
SIZES = [(1, 1, 1, 1, 1, 1), (3, 33, 47, 16, 23, 13), (2, 64, 96, 32, 48, 16), (1, 50, 70, 25, 35, 17),
         (2, 48, 80, 17, 33, 64), (1, 40, 64, 20, 31, 65), (1, 32, 32, 9, 7, 256),
         (1, 32, 32, 9, 7, 257), (1, 20, 30, 60, 90, 5), (2, 48, 40, 1, 1, 256)]


def _hist(oh, ow, nc):
    return (4 * oh * ow * nc + 255) // 256 * 256


def _enough(oh, ow, nc):
    """Batch elements from which a call's histograms (4 MB) are kept in LDS."""
    return -(-(4 << 20) // _hist(oh, ow, nc))


@pytest.mark.parametrize("few", [False, True], ids=["lds", "histogram"])
@pytest.mark.parametrize("tc", SIZES, ids=lambda t: "x".join(map(str, t)))
def test_coherent_maps(oracle, tc, few):
    B, ih, iw, oh, ow, nc = tc
    B = B if few else _enough(oh, ow, nc)
    rng = np.random.default_rng(sum(tc))
    labels = rng.integers(-1, nc + 1, (B, 1, ih, iw))   # some outside [0, classes)
    vmap = _coherent(ih, iw, oh, ow)
    want = oracle.voting_resample_to_map(labels, vmap, oh, ow, nc)
    assert np.array_equal(_call(labels, vmap, oh, ow, nc), want)
    # the least workspace (histogram, no flag), and one with room for the flag but not all elements
    hist = _hist(oh, ow, nc)
    for ws in (hist, hist + 256):
        assert np.array_equal(_call(labels, vmap, oh, ow, nc, ws), want)


@pytest.mark.parametrize("nc", [4, 40])
@pytest.mark.parametrize("kind", ["scrambled", "one cell", "two halves"])
def test_maps_that_raise_the_flag(oracle, kind, nc):
    ih, iw, oh, ow = 160, 208, 40, 52
    B = _enough(oh, ow, nc)
    rng = np.random.default_rng(nc)
    labels = rng.integers(0, nc, (B, 1, ih, iw))
    vmap = _coherent(ih, iw, oh, ow)
    if kind == "scrambled":
        vmap = rng.permutation(vmap.reshape(-1, 2)).reshape(vmap.shape)
    elif kind == "one cell":
        vmap[...] = (ow - 1, oh - 1)
    else:
        vmap[:, iw // 2:] = (0, 0)
    assert np.array_equal(_call(labels, vmap, oh, ow, nc),
                          oracle.voting_resample_to_map(labels, vmap, oh, ow, nc))


@pytest.mark.parametrize("nc", [4, 40])
@pytest.mark.parametrize("kind", ["coherent", "half scrambled", "one far cell", "scrambled", "folded"])
def test_crowded_and_other_cells_side_by_side(oracle, kind, nc):
    """Cells of crowded squares are counted in memory, the others in LDS, with room for one, three and
    all of the elements' histograms, in memory that is not clear."""
    ih, iw, oh, ow = 160, 208, 40, 52
    if kind == "folded":    # squares of 16 x 16 cells that 81 tiles and more vote into, side by side
        ih, iw, oh, ow = 320, 640, 34, 68
    hist = _hist(oh, ow, nc)
    B = _enough(oh, ow, nc)
    rng = np.random.default_rng(nc)
    labels = rng.integers(-1, nc + 1, (B, 1, ih, iw))
    vmap = _coherent(ih, iw, oh, ow)
    if kind == "half scrambled":
        vmap[:80] = rng.permutation(vmap[:80].reshape(-1, 2)).reshape(80, iw, 2)
    elif kind == "one far cell":
        vmap[::16, ::16] = (1, 2)
    elif kind == "scrambled":
        vmap = rng.permutation(vmap.reshape(-1, 2)).reshape(vmap.shape)
    want = oracle.voting_resample_to_map(labels, vmap, oh, ow, nc)
    for n in (1, 3, B):   # (and 128 KB for what the LDS kernels need beside the histograms)
        assert np.array_equal(_call(labels, vmap, oh, ow, nc, n * hist + (1 << 17)), want)
    assert np.array_equal(_call(labels, vmap, oh, ow, nc), want)
