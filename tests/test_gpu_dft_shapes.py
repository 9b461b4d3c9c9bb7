"""The instances of the matrix-core DFT passes: 32 or 16 lines per block by 32 or
16 output pairs per wave step, whole or split over several blocks, as
pf_describe_launch reports them (dft_<axis>=<forward>/<inverse>, each lines x
pairs x blocks that split a group's outputs), against 64-bit transforms.  Few
lines always take 16 x 16; the larger instances need 512 groups."""

import ctypes

import numpy as np
import pytest
import torch

import pyfourier_amd as pf
from oracle import restate as R
from pyfourier_amd import _lib
from pyfourier_amd._nufft import _Call

pytestmark = pytest.mark.gpu

STAGE = 2e-6  # the stage tests' bound for one FP32 transform


def rel(a, b):
    return float(np.linalg.norm((a - b).ravel()) / np.linalg.norm(b.ravel()))


def _randn(rng, shape):
    return (rng.standard_normal(shape, np.float32) + 1j * rng.standard_normal(shape, np.float32)).astype(np.complex64)


def _stages(dev, shape, oversamp, C, expect, workspace=True):
    rng = np.random.default_rng(C)
    d = len(shape)
    coord = rng.uniform(-np.pi, np.pi, size=(64, d)).astype(np.float32)
    coord[0, 0] = -np.pi
    plan = pf.plan_nufft(torch.from_numpy(coord), shape, width=4, oversamp=oversamp).to(dev)
    P = R.Plan(coord, shape, width=4, oversamp=oversamp)
    call = _Call(plan, dev, None, None, None)
    what = call.describe(C)
    assert expect in what, what
    G = tuple(P.os_shape)
    Cf = 2 if d == 3 and C % 2 == 0 else max(v for v in range(1, min(C, 64) + 1) if C % v == 0)
    Ca = max(v for v in range(1, min(C, 64) + 1) if C % v == 0)
    x = _randn(rng, (C,) + tuple(shape))
    desc, L, st = call.desc(C, (None, None)), _lib.lib(), _lib.stream_of(dev)
    h, D = call.native.handle, ctypes.byref(desc)
    n = ctypes.c_size_t()
    _lib.check(L.pf_workspace_size(h, D, 1, ctypes.byref(n)))
    ws = torch.zeros(n.value, dtype=torch.uint8, device=dev) if workspace else None
    xd = torch.from_numpy(x).to(dev)
    grid = torch.full((C // Cf,) + G + (Cf,), float("nan"), dtype=torch.complex64, device=dev)
    _lib.check(L.pf_pad_fft(h, D, _lib.ptr(xd), _lib.ptr(grid), _lib.ptr(ws), st))
    ref = np.fft.ifftshift(R._to_grid(x[:, None], P, None)[:, 0], axes=tuple(range(-d, 0)))
    got = np.moveaxis(grid.cpu().numpy(), -1, 1).reshape((C,) + G)
    assert rel(got, ref) < STAGE, (shape, C)
    ga = np.ascontiguousarray(np.moveaxis(ref.reshape((C // Ca, Ca) + G), 1, -1)).astype(np.complex64)
    grid = torch.from_numpy(ga).to(dev)
    img = torch.full_like(xd, float("nan"))
    _lib.check(L.pf_ifft_crop(h, D, _lib.ptr(grid), _lib.ptr(img), 1.0, _lib.ptr(ws), st))
    back = R._from_grid(np.fft.fftshift(ref, axes=tuple(range(-d, 0)))[:, None], P, None)[:, 0] * np.prod(G)
    assert rel(img.cpu().numpy(), back) < STAGE, (shape, C)


@pytest.mark.parametrize(
    "shape,C,expect",
    [
        # one block per 16 lines and per part of the outputs
        ((90,), 3, "dft_x=16x16x1/16x16x1"),
        ((317, 5), 1, "dft_y=16x16x4/16x16x3"),
        ((5, 317), 2, "dft_x=16x16x4/16x16x3"),
        # 62 points: 32 lines x 16 pairs
        ((49,), 20032, "dft_x=32x16x1/32x16x1"),
        ((49, 20), 832, "dft_y=32x16x1/32x16x1"),
        # 113 points: 32 x 32
        ((90,), 20032, "dft_x=32x32x1/32x32x1"),
        ((90, 20), 832, "dft_y=32x32x1/32x32x1"),
        ((90, 20, 20), 64, "dft_z=32x32x1/32x32x1"),
        ((20, 90, 10), 64, "dft_y=32x32x1/32x32x1"),
        ((90, 20), 833, "dft_y=32x32x1/32x32x1"),  # 7 x 119: an odd batch, single values
        # 330 points: 32 lines forward, 16 inverse
        ((264, 10), 1664, "dft_y=32x32x1/16x16x1"),
        # 433 and 509 points: 16 lines x 32 pairs
        ((346,), 10048, "dft_x=16x32x1/16x16x1"),
        ((346, 10), 1024, "dft_y=16x32x1/16x16x1"),
        ((407,), 10048, "dft_x=16x32x1/16x32x1"),
        ((407, 10), 1024, "dft_y=16x32x1/16x32x1"),
    ],
)
def test_every_instance(cuda_device, shape, C, expect):
    print(f"dft shapes: {shape} x {C}", flush=True)
    _stages(cuda_device, shape, 1.25, C, expect)


# rows and columns of centred transforms; the same instances by the same counts
@pytest.mark.parametrize("shape,C", [((62, 62), 264), ((113, 113), 160), ((113, 113), 1), ((433, 433), 24), ((509, 30), 300)])
def test_cartesian_instances(cuda_device, shape, C):
    print(f"dft cartesian: {shape} x {C}", flush=True)
    g = torch.Generator(device=cuda_device).manual_seed(C)
    x = torch.randn((C,) + shape, dtype=torch.complex64, device=cuda_device, generator=g)
    mask = (torch.rand(shape, device=cuda_device, generator=g) < 0.4).float()
    plan, ax = pf.plan_fft(mask, shape), (1, 2)
    y = pf.fftn(2, x, plan=plan, device=cuda_device)
    z = pf.ifftn(2, x, plan=plan, device=cuda_device)
    x, mask = x.cdouble().cpu(), mask.cpu()
    yr = torch.fft.fftshift(torch.fft.fftn(torch.fft.ifftshift(x, dim=ax), dim=ax), dim=ax) * mask
    zr = torch.fft.fftshift(torch.fft.ifftn(torch.fft.ifftshift(x * mask, dim=ax), dim=ax), dim=ax)
    for a, r in ((y, yr), (z, zr)):
        a = a.cpu().reshape(r.shape)
        assert float((a - r).norm() / r.norm()) < STAGE


def test_stages_without_a_workspace(cuda_device):
    """Sizes outside the radix sets take a null FFT workspace (the in-place
    stage); the radix sizes refuse it."""
    _stages(cuda_device, (37, 29), 1.5, 3, "fft=fused", workspace=False)
    with pytest.raises(RuntimeError, match="missing FFT workspace"):
        _stages(cuda_device, (32, 32), 2.0, 3, "fft=fused", workspace=False)
