"""Backward of the convolution layers where only some gradients are wanted: what is formed is what
the full backward forms, what is not wanted stays None.  Gradient sums are added in an order that
depends on scheduling, so values are compared to rounding (1e-5)."""
import itertools

import numpy as np
import pytest
import torch

import workloads
from conftest import relerr

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("channels,transposed", [(3, False), (40, False), (40, True), (3, True)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_each_choice_of_gradients(channels, transposed, dtype):
    import spherical_distortion.nn as snn
    gen = torch.Generator(device=DEV).manual_seed(channels)
    m = torch.from_numpy(workloads.gnomonic_kernel_map(24, 48)).to(DEV, dtype)
    cls = snn.MappedTransposedConvolution if transposed else snn.MappedConvolution
    layer = cls(channels, 20, kernel_size=9).to(DEV, dtype)
    x = torch.randn(2, channels, 24, 48, generator=gen, device=DEV, dtype=dtype)
    g = torch.randn(2, 20, 24, 48, generator=gen, device=DEV, dtype=dtype)
    args = (24, 48, m) if transposed else (m,)

    def grads(want):
        leaves = [x.clone(), layer.weight, layer.bias]
        for t, on in zip(leaves, want):
            t.grad = None
            t.requires_grad_(on)
        layer(leaves[0], *args).backward(g)
        return [t.grad for t in leaves]

    full = grads((True, True, True))
    for want in itertools.product((False, True), repeat=3):
        if any(want):
            for got, ref, on in zip(grads(want), full, want):
                assert (got is not None) == on
                if on:
                    assert relerr(got.cpu().numpy(), ref.cpu().numpy()) <= 1e-5


def test_max_pool_indices_carry_no_gradient():
    import spherical_distortion.nn as snn
    m = torch.from_numpy(workloads.gnomonic_kernel_map(16, 32)).to(DEV)
    # Values above zero: a sample beside the image counts as zero, and where one wins (all others
    # of its window negative) the gradient falls beside the image too.
    x = torch.rand(1, 2, 16, 32, device=DEV).add_(0.5).requires_grad_()
    out, idx = snn.MappedMaxPool(9, snn.InterpolationType.NEAREST, return_indices=True)(x, m)
    assert idx.dtype == torch.int64 and not idx.requires_grad
    out.sum().backward()
    assert np.isclose(float(x.grad.sum()), out.numel())
