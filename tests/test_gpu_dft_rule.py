"""Which route a length outside the radix sets takes: the matrix-core DFT passes,
or rocFFT with pad and crop kernels for few transforms of more than 525 image points,
beyond 1024 points and where the x axis is longer.  Both sides of each line
against 64-bit results."""

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


def _nufft(dev, shape, oversamp, C, route):
    print(f"dft rule: {shape} sigma={oversamp} x {C} {route}", flush=True)
    rng = np.random.default_rng(sum(shape) + C)
    coord = rng.uniform(-np.pi, np.pi, (1, 300, len(shape))).astype(np.float32)
    coord[0, 0, 0] = -np.pi
    P = R.Plan(coord, shape, width=4, oversamp=oversamp)
    plan = pf.plan_nufft(torch.from_numpy(coord), shape, width=4, oversamp=oversamp).to(dev)
    what = _Call(plan, dev, None, None, None).describe(C)
    assert f"fft={route}" in what, (P.os_shape, what)
    x = demo.complex_gaussian(rng, (C,) + tuple(shape))
    y = demo.complex_gaussian(rng, (C, 1, 300))
    yg = pf.nufft(torch.from_numpy(x).to(dev), nufft_plan=plan, device=dev)
    xg = pf.nufft_adj(torch.from_numpy(y).to(dev), nufft_plan=plan, device=dev)
    assert rel(yg.cpu().numpy(), R.nufft(x[:, None], P)) < PARITY
    assert rel(xg.cpu().numpy(), R.nufft_adj(y, P)) < PARITY


@pytest.mark.parametrize(
    "shape,oversamp,few",
    [
        ((308, 10), 1.25, 1),   # 385 points: always the DFT passes
        ((314, 10), 1.25, 1),   # 393 = 3 * 131: no radix passes in rocFFT
        ((392, 10), 1.25, 1),   # 490
        ((526, 10), 1.13, 2),   # 595
        ((10, 526), 1.13, 2),
        ((352, 8), 2.0, 1),     # 704 of 352
        ((563, 8), 1.25, 16),   # 704 of 563
        ((493, 8), 1.25, 1),    # 617, prime
        ((501, 6), 2.0, 1),     # 1002 = 6 * 167 of 501
        ((550, 8), 1.25, 8),    # 688 = 16 * 43 of 550
        ((8, 6, 526), 1.13, 2),
    ],
)
def test_route_by_batch(cuda_device, shape, oversamp, few):
    if few > 1:
        _nufft(cuda_device, shape, oversamp, few - 1, "rocfft")
    _nufft(cuda_device, shape, oversamp, few, "fused")


@pytest.mark.parametrize("shape,oversamp", [((687,), 1.5), ((687, 8), 1.5), ((8, 687), 1.5), ((6, 8, 687), 1.5),
                                            ((114, 1024), 1.25)])  # 1031 points; 143 x 1280: a longer x axis
@pytest.mark.parametrize("C", [1, 17])
def test_rocfft_route(cuda_device, shape, oversamp, C):
    _nufft(cuda_device, shape, oversamp, C, "rocfft")


def _cart(dev, shape, C):
    rng = np.random.default_rng(C)
    x = torch.from_numpy(demo.complex_gaussian(rng, (C,) + shape)).to(dev)
    mask = torch.from_numpy((rng.random(shape) < 0.4).astype(np.float32)).to(dev)
    plan = pf.plan_fft(mask, shape)
    d, ax = len(shape), tuple(range(1, len(shape) + 1))
    y = pf.fftn(d, x, plan=plan, device=dev)
    z = pf.ifftn(d, x, plan=plan, device=dev)
    x, mask = x.cdouble().cpu(), mask.cpu()
    yr = torch.fft.fftshift(torch.fft.fftn(torch.fft.ifftshift(x, dim=ax), dim=ax), dim=ax) * mask
    zr = torch.fft.fftshift(torch.fft.ifftn(torch.fft.ifftshift(x * mask, dim=ax), dim=ax), dim=ax)
    assert rel(y.cpu(), yr) < PARITY and rel(z.cpu(), zr) < PARITY


@pytest.mark.parametrize("shape,C", [((546, 12), 1), ((546, 12), 2), ((14, 616), 15), ((14, 616), 16), ((1031,), 3),
                                     ((6, 1031), 2), ((1031, 6), 9)])
def test_cartesian(cuda_device, shape, C):
    print(f"dft rule: cartesian {shape} x {C}", flush=True)
    _cart(cuda_device, shape, C)


@pytest.mark.parametrize("shape,C", [((273, 10), 1), ((273, 10), 2), ((519, 6), 2)])  # embeddings 546 x 20, 1038 x 12
def test_toeplitz_embedding(cuda_device, shape, C):
    rng = np.random.default_rng(C)
    coord = rng.uniform(-np.pi, np.pi, (1, 500, 2)).astype(np.float32)
    gm = pf.plan_spgram(torch.from_numpy(coord), shape, device=cuda_device)
    x = torch.from_numpy(demo.complex_gaussian(rng, (C,) + shape)).to(cuda_device)
    y = pf.sparse_gram(x, gm, device=cuda_device).cpu()
    big = tuple(2 * n for n in shape)
    box = (slice(None),) + tuple(slice(0, n) for n in shape)
    z = torch.zeros((C,) + big, dtype=torch.complex128)
    z[box] = x.cdouble().cpu()
    ref = torch.fft.ifftn(torch.fft.fftn(z, dim=(1, 2)) * gm.value.reshape(big).cdouble().cpu(), dim=(1, 2))[box]
    assert rel(y, ref) < PARITY


@pytest.mark.parametrize("shape,oversamp,C", [((526, 10), 1.13, 1), ((563, 8), 1.25, 3)])
def test_first_call_under_capture(cuda_device, shape, oversamp, C):
    """A batch that runs rocFFT may be captured from its first call on: nothing
    is allocated there, so the DFT passes take it; after an eager call the
    captured one runs rocFFT as well."""
    print(f"dft rule: capture {shape} x {C}", flush=True)
    rng = np.random.default_rng(C)
    coord = rng.uniform(-np.pi, np.pi, (1, 300, 2)).astype(np.float32)
    coord[0, 0, 0] = -np.pi
    plan = pf.plan_nufft(torch.from_numpy(coord), shape, width=4, oversamp=oversamp).to(cuda_device)
    cart = pf.plan_fft(None, shape).to(cuda_device)
    assert "fft=rocfft" in _Call(plan, cuda_device, None, None, None).describe(C)
    x = torch.from_numpy(demo.complex_gaussian(rng, (C,) + shape)).to(cuda_device)
    y = torch.from_numpy(demo.complex_gaussian(rng, (C, 1, 300))).to(cuda_device)

    def calls():
        return (pf.nufft(x, nufft_plan=plan, device=cuda_device), pf.nufft_adj(y, nufft_plan=plan, device=cuda_device),
                pf.fftn(2, x, plan=cart, device=cuda_device))

    torch.cuda.synchronize()
    for again in range(2):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            captured = calls()
        eager = [v.clone() for v in calls()]
        for r in range(3):
            for v in captured:
                v.zero_()
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            for a, b in zip(captured, eager):
                assert rel(a.cpu(), b.cpu()) < PARITY, (again, r)
            calls()
