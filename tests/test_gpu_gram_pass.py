"""The Gram's one-pass middle axis (k_gramcolq) at every line length it is
built for, as y (2-D) and z (3-D) axis, full lines (dense Gram) and pruned ones
(Toeplitz embedding), against the same operator in 64-bit torch."""

import numpy as np
import pytest
import torch

import pyfourier_amd as pf
from pyfourier_amd import demo

pytestmark = pytest.mark.gpu

PARITY = 1e-5  # the repository's complex64-against-float64 bar
SIZES = [40, 56, 72, 80, 96, 112, 120, 128, 144, 160, 168, 192, 200, 224, 240, 256, 280, 288, 320, 336, 360, 384, 400,
         448, 480, 512, 576, 640]


def rel(a, b):
    return float((a.cpu().cdouble() - b.cpu()).norm() / b.cpu().norm())


def _dense(cuda_device, shape, C, F):
    rng = np.random.default_rng(sum(shape) + C)
    d = len(shape)
    mask = torch.from_numpy((rng.random((F,) + shape) < 0.4).astype(np.float32))
    gm = pf.plan_gram(mask, shape, device=cuda_device)
    lead = (C, F) if F > 1 else (C,)
    x = torch.from_numpy(demo.complex_gaussian(rng, lead + shape)).to(cuda_device)
    y = pf.gram(x, gm, device=cuda_device)
    ax = tuple(range(-d, 0))
    m = (mask if F > 1 else mask[0]).to(cuda_device).double()
    k = torch.fft.fftshift(torch.fft.fftn(torch.fft.ifftshift(x.cdouble(), dim=ax), dim=ax), dim=ax) * m
    ref = torch.fft.fftshift(torch.fft.ifftn(torch.fft.ifftshift(k, dim=ax), dim=ax), dim=ax)
    assert rel(y, ref) < PARITY


@pytest.mark.parametrize("G", SIZES)
def test_dense_gram_lines(cuda_device, G):
    _dense(cuda_device, (G, 12), 3, 1)   # 36 values per row: a partial block of 16
    _dense(cuda_device, (G, 20), 1, 2)   # one kernel per frame
    if G <= 200:
        _dense(cuda_device, (G, 6, 8), 70, 1)  # two coil blocks


def test_dense_gram_wide_blocks(cuda_device):
    _dense(cuda_device, (80, 64, 64), 16, 1)  # 65536 lines: 32 per block


@pytest.mark.parametrize("shape", [(40, 30), (64, 25), (100, 40), (28, 20), (31, 40), (20, 18, 24), (40, 9, 10)])
@pytest.mark.parametrize("C", [1, 5])
def test_toeplitz_embedding(cuda_device, shape, C):
    rng = np.random.default_rng(sum(shape))
    d = len(shape)
    coord = rng.uniform(-np.pi, np.pi, (1, 500, d)).astype(np.float32)
    gm = pf.plan_spgram(torch.from_numpy(coord), shape, device=cuda_device)
    x = torch.from_numpy(demo.complex_gaussian(rng, (C,) + shape)).to(cuda_device)
    y = pf.sparse_gram(x, gm, device=cuda_device)
    big = tuple(2 * n for n in shape)
    box = (slice(None),) + tuple(slice(0, n) for n in shape)
    z = torch.zeros((C,) + big, dtype=torch.complex128, device=cuda_device)
    z[box] = x.cdouble()
    ax = tuple(range(1, d + 1))
    ref = torch.fft.ifftn(torch.fft.fftn(z, dim=ax) * gm.value.reshape(big).cdouble(), dim=ax)[box]
    assert rel(y, ref) < PARITY
