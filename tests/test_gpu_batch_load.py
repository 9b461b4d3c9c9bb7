"""What NUFFTBatch's loader keeps of an ordinary in-place copy: autograd notices
the write, sources may lie in the batch's own buffers, and list entries that a
caller replaced are written in their own layout."""

import numpy as np
import pytest
import torch

import pyfourier_amd as pf
from pyfourier_amd import demo

pytestmark = pytest.mark.gpu


def _batch(dev, nbatch=2):
    coords = [demo.golden_angle_radial_2d(7, 32), demo.golden_angle_radial_2d(7, 32)]
    return pf.plan_nufft_batch(coords, [24, 24], nbatch=nbatch, device=dev)


def _randn(rng, t):
    return torch.from_numpy(demo.complex_gaussian(rng, tuple(t.shape))).to(t.device)


def test_a_load_is_seen_by_autograd(cuda_device):
    batch = _batch(cuda_device)
    rng = np.random.default_rng(0)
    y = batch.forward([_randn(rng, v) for v in batch.images])
    w = torch.ones_like(y[0], requires_grad=True)
    loss = (w * y[0]).abs().sum()  # saves the k-space buffer for w's gradient
    batch.adjoint([_randn(rng, v) for v in batch.kspace])  # and overwrites it
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        loss.backward()


@pytest.mark.parametrize("nbatch", [2, 3])
def test_sources_in_the_buffers_themselves(cuda_device, nbatch):
    batch = _batch(cuda_device, nbatch)
    rng = np.random.default_rng(1)
    x = [_randn(rng, v) for v in batch.images]
    k = [v.clone() for v in batch.forward(x)]
    # each at its own place: the forward's results straight into the adjoint
    a = [v.clone() for v in batch.adjoint(batch.kspace)]
    b = [v.clone() for v in batch.adjoint(k)]
    assert all(torch.equal(p, q) for p, q in zip(a, b))
    # the second item's buffer for both: item by item, in order
    batch.adjoint(k)
    a = [v.clone() for v in batch.adjoint([batch.kspace[1], batch.kspace[0]])]
    b = [v.clone() for v in batch.adjoint([k[1], k[1]])]
    assert all(torch.equal(p, q) for p, q in zip(a, b))


def test_a_replaced_buffer_is_written_in_its_own_layout(cuda_device):
    coords = [demo.golden_angle_radial_2d(7, 32), demo.golden_angle_radial_2d(7, 32)]
    batch = pf.plan_nufft_batch(coords, [24, 24], nbatch=2, device=cuda_device, group=False, graph=False)
    rng = np.random.default_rng(2)
    x = [_randn(rng, v) for v in batch.images]
    batch.images[0] = torch.zeros((24, 24, 2, 1), dtype=torch.complex64, device=cuda_device).permute(2, 3, 0, 1)
    batch._load(batch.images, x)
    assert all(torch.equal(p, q) for p, q in zip(batch.images, x))
