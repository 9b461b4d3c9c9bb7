"""The FP32 matrix-core spread (k_spread_pipe) at the edges of its forms: each
values-per-wave instance and its remainders, batches stored as one value per
grid block, grids smaller than a tile or cut by its edge, wide kernels and those
whose tap records are shorter than the four pieces a wave stages at a time, split
tiles, and frames sharing one grid through a basis of odd size."""

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


def _traj(ndim):
    if ndim == 3:
        return demo.golden_means_radial_3d(90, 33)
    if ndim == 2:
        return demo.golden_angle_radial_2d(37, 61)
    return (np.linspace(-np.pi, np.pi, 257, endpoint=False).astype(np.float32) ** 3 / np.float32(np.pi ** 2))[:, None][None]


def _check(cuda_device, ndim, shape, C, width, oversamp, chunk, routed=True):
    rng = np.random.default_rng(100 * ndim + C)
    coord = _traj(ndim)
    y = demo.complex_gaussian(rng, (C,) + coord.shape[:-1])
    plan = pf.plan_nufft(torch.from_numpy(coord), shape, width=width, oversamp=oversamp, chunk=chunk).to(cuda_device)
    what = _Call(plan, cuda_device, None, None, None).describe(C)
    assert not routed or "spread=k_spread_pipe<" in what, what
    x = pf.nufft_adj(torch.from_numpy(y).to(cuda_device), nufft_plan=plan, device=cuda_device)
    P = R.Plan(coord, shape, width=width, oversamp=oversamp)
    xr = R.nufft_adj(y.reshape(C, 1, -1), P)
    assert rel(x.cpu().numpy().reshape(xr.shape), xr) < PARITY


# 1, 2, 4, 8, 16, 32 values per wave, each with its remainders; 67 values are
# stored as 67 blocks of one value, 70 as two of 35
@pytest.mark.parametrize("C", [1, 2, 3, 4, 5, 7, 9, 15, 17, 25, 33, 67, 70])
@pytest.mark.parametrize("ndim,shape", [(1, (50,)), (2, (29, 37)), (3, (17, 21, 26))])
def test_values_per_wave(cuda_device, ndim, shape, C):
    _check(cuda_device, ndim, shape, C, 4, 1.5, 16 if C % 2 else 0)


@pytest.mark.parametrize("width", [3, 8])
@pytest.mark.parametrize("ndim,shape", [(1, (9,)), (2, (7, 11)), (2, (13, 40)), (3, (6, 9, 7)), (3, (20, 5, 12))])
def test_small_grids_and_widths(cuda_device, ndim, shape, width):
    for C in (1, 3, 8):
        # a grid axis too short for tile + width becomes one tile, which may
        # exceed every instance (the LDS-staged spread then runs)
        _check(cuda_device, ndim, shape, C, width, 2.0, 0, routed=False)


@pytest.mark.parametrize("C", [1, 8, 17])
@pytest.mark.parametrize("ndim,shape,width", [(1, (60,), 2), (1, (60,), 6), (2, (40, 44), 2), (2, (40, 44), 3),
                                              (3, (24, 20, 26), 2)])  # records of 2 and 3 pieces
def test_short_records(cuda_device, ndim, shape, width, C):
    _check(cuda_device, ndim, shape, C, width, 2.0, 0)


@pytest.mark.parametrize("C,K", [(5, 3), (1, 3), (3, 7)])
def test_shared_grid_odd_vector(cuda_device, C, K):
    """C coils x K coefficients expanded by the sort: odd values per point."""
    rng = np.random.default_rng(C * K)
    F, shape = 6, (24, 31)
    coord = demo.golden_angle_radial_2d(F * 5, 40).reshape(F, 5, 40, 2)
    basis = np.linalg.qr(demo.complex_gaussian(rng, (F, min(K, F))))[0].astype(np.complex64)
    y = demo.complex_gaussian(rng, (C, F, 5, 40))
    plan = pf.plan_nufft(torch.from_numpy(coord), shape, width=4, oversamp=1.25).to(cuda_device)
    what = _Call(plan, cuda_device, torch.from_numpy(basis), None, None).describe(C)
    assert "spread=k_sort_x+k_spread_pipe<" in what, what
    x = pf.nufft_adj(torch.from_numpy(y).to(cuda_device), nufft_plan=plan, basis=torch.from_numpy(basis),
                     device=cuda_device)
    xr = R.nufft_adj(y.reshape(C, F, -1), R.Plan(coord, shape, width=4, oversamp=1.25), basis=basis)
    assert rel(x.cpu().numpy().reshape(xr.shape), xr) < PARITY
