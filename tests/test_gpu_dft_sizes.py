"""Grid and matrix sizes with prime factors outside the radix sets: the DFT
passes on the matrix cores, as rows and columns, forward and inverse, at the
edges of the tiles that few lines take (16 lines, 16 output pairs, 4 folded
rows) and, in the volumes, 32 lines.  test_gpu_dft_shapes.py has the others."""

import numpy as np
import pytest
import torch

import pyfourier_amd as pf
from oracle import restate as R
from pyfourier_amd import demo
from pyfourier_amd._nufft import _Call

pytestmark = pytest.mark.gpu

PARITY = 1e-5  # the repository's complex64-against-float64 bar


def rel(a, b):
    a, b = np.asarray(a).ravel(), np.asarray(b).ravel()
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def _coord(ndim, rng, n=400):
    return (rng.uniform(-np.pi, np.pi, (1, n, ndim))).astype(np.float32)


def _both(cuda_device, shape, oversamp, C):
    rng = np.random.default_rng(sum(shape) + C)
    coord = _coord(len(shape), rng)
    P = R.Plan(coord, shape, width=4, oversamp=oversamp)
    plan = pf.plan_nufft(torch.from_numpy(coord), shape, width=4, oversamp=oversamp).to(cuda_device)
    assert "fft=fused" in _Call(plan, cuda_device, None, None, None).describe(C), plan.os_shape
    x = demo.complex_gaussian(rng, (C,) + tuple(shape))
    y = demo.complex_gaussian(rng, (C, 1, 400))
    yg = pf.nufft(torch.from_numpy(x).to(cuda_device), nufft_plan=plan, device=cuda_device)
    xg = pf.nufft_adj(torch.from_numpy(y).to(cuda_device), nufft_plan=plan, device=cuda_device)
    assert rel(yg.cpu().numpy(), R.nufft(x[:, None], P)) < PARITY
    assert rel(xg.cpu().numpy(), R.nufft_adj(y, P)) < PARITY


# oversampled lengths 11, 13, 17, 22, 31, 33, 61, 77, 127, 143, 263, 283, 289, 509, 1022
@pytest.mark.parametrize("n,oversamp", [(7, 1.5), (10, 1.25), (11, 1.5), (11, 2.0), (20, 1.54), (22, 1.5), (40, 1.5),
                                        (61, 1.25), (101, 1.25), (114, 1.25), (210, 1.25), (226, 1.25), (231, 1.25),
                                        (407, 1.25), (511, 2.0)])
@pytest.mark.parametrize("C", [1, 5])
def test_rows(cuda_device, n, oversamp, C):
    _both(cuda_device, (n,), oversamp, C)


@pytest.mark.parametrize("shape,oversamp", [((11, 32), 2.0), ((32, 11), 2.0), ((59, 37), 1.25), ((20, 187), 1.25),
                                            ((211, 26), 1.25), ((13, 13), 1.0 + 1.0 / 13)])
@pytest.mark.parametrize("C", [1, 2, 4, 7, 33])
def test_planes(cuda_device, shape, oversamp, C):
    _both(cuda_device, shape, oversamp, C)


@pytest.mark.parametrize("shape,oversamp", [((10, 18, 21), 1.25), ((17, 9, 11), 2.0), ((11, 16, 13), 1.5), ((32, 23, 16), 2.0)])
@pytest.mark.parametrize("C", [1, 4, 6, 32, 70])
def test_volumes(cuda_device, shape, oversamp, C):
    _both(cuda_device, shape, oversamp, C)


@pytest.mark.parametrize("shape,L", [((33, 37), 3), ((26, 32), 20), ((37, 224), 17)])
def test_field_map_segments(cuda_device, shape, L):
    """Segments on a DFT x axis, and more than a radix or register x axis
    (40 and 280 points) takes where only y needs the DFT passes."""
    rng = np.random.default_rng(L)
    C, oversamp = 3, 1.25
    coord = demo.variable_density_spiral_2d(3, 200, max(shape))
    t = np.linspace(0, 8e-3, 200).astype(np.float32)
    zmap = demo.smooth_field_map(rng, shape, 80.0)
    plan = pf.plan_nufft(torch.from_numpy(coord), shape, width=4, oversamp=oversamp, zmap=torch.from_numpy(zmap),
                         T=torch.from_numpy(t), L=L, nbins=40, L_batch_size=L).to(cuda_device)
    b0 = (plan.zmap_t_kernel.cpu().numpy().astype(np.complex128), plan.zmap_s_kernel.cpu().numpy().astype(np.complex128))
    P = R.Plan(coord, shape, width=4, oversamp=oversamp)
    x = demo.complex_gaussian(rng, (C,) + shape)
    y = demo.complex_gaussian(rng, (C,) + coord.shape[:-1])
    yg = pf.nufft(torch.from_numpy(x).to(cuda_device), nufft_plan=plan, device=cuda_device)
    xg = pf.nufft_adj(torch.from_numpy(y).to(cuda_device), nufft_plan=plan, device=cuda_device)
    assert rel(yg.cpu().numpy().reshape(C, 1, -1), R.nufft(x[:, None], P, b0=b0)) < PARITY
    assert rel(xg.cpu().numpy(), R.nufft_adj(y.reshape(C, 1, -1), P, b0=b0)[:, 0]) < PARITY


@pytest.mark.parametrize("K", [0, 3])
def test_frames_and_basis(cuda_device, K):
    rng = np.random.default_rng(K)
    F, C, shape = 4, 3, (22, 35)
    coord = demo.golden_angle_radial_2d(F * 6, 50).reshape(F, 6, 50, 2)
    P = R.Plan(coord, shape, width=4, oversamp=1.5)
    plan = pf.plan_nufft(torch.from_numpy(coord), shape, width=4, oversamp=1.5).to(cuda_device)
    basis = np.linalg.qr(demo.complex_gaussian(rng, (F, K)))[0].astype(np.complex64) if K else None
    bt = None if basis is None else torch.from_numpy(basis)
    x = demo.complex_gaussian(rng, (C, K or F) + shape)
    y = demo.complex_gaussian(rng, (C, F, 6, 50))
    yg = pf.nufft(torch.from_numpy(x).to(cuda_device), nufft_plan=plan, basis=bt, device=cuda_device)
    xg = pf.nufft_adj(torch.from_numpy(y).to(cuda_device), nufft_plan=plan, basis=bt, device=cuda_device)
    assert rel(yg.cpu().numpy().reshape(C, F, -1), R.nufft(x, P, basis=basis)) < PARITY
    assert rel(xg.cpu().numpy(), R.nufft_adj(y.reshape(C, F, -1), P, basis=basis)) < PARITY


@pytest.mark.parametrize("shape", [(11,), (509,), (13, 32), (32, 13), (46, 59), (14, 17, 11), (22, 16, 26)])
@pytest.mark.parametrize("C", [1, 5])
def test_cartesian(cuda_device, shape, C):
    rng = np.random.default_rng(len(shape) + C)
    x = torch.from_numpy(demo.complex_gaussian(rng, (C,) + shape)).to(cuda_device)
    mask = torch.from_numpy((rng.random(shape) < 0.4).astype(np.float32)).to(cuda_device)
    plan = pf.plan_fft(mask, shape)
    d, ax = len(shape), tuple(range(1, len(shape) + 1))
    for norm in (None, "ortho"):
        y = pf.fftn(d, x, plan=plan, norm=norm, device=cuda_device)
        yr = torch.fft.fftshift(torch.fft.fftn(torch.fft.ifftshift(x.cdouble(), dim=ax), dim=ax, norm=norm), dim=ax) * mask
        assert rel(y.cpu(), yr.cpu()) < PARITY
        z = pf.ifftn(d, x, plan=plan, norm=norm, device=cuda_device)
        zr = torch.fft.fftshift(torch.fft.ifftn(torch.fft.ifftshift(x.cdouble() * mask, dim=ax), dim=ax, norm=norm), dim=ax)
        assert rel(z.cpu(), zr.cpu()) < PARITY
