"""Rounding of the matrix-core DFT passes against rocFFT's single-precision
transforms, whose place they take: no larger, over the lengths they run at."""

import pytest
import torch

import pyfourier_amd as pf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,planes", [(77, 8), (196, 8), (331, 8), (484, 8), (572, 8), (660, 16), (832, 16), (880, 16), (1001, 16)])
def test_rounding_no_larger_than_rocfft(cuda_device, n, planes):
    # torch.fft on this device is rocFFT
    g = torch.Generator(device=cuda_device).manual_seed(n)
    x = torch.randn((planes, n, n), dtype=torch.complex64, device=cuda_device, generator=g)
    sh = lambda v: torch.fft.fftshift(v, dim=(1, 2))
    xs = torch.fft.ifftshift(x, dim=(1, 2))
    ref = sh(torch.fft.fft2(xs.cdouble()))
    lib = sh(torch.fft.fft2(xs)).cdouble()
    own = pf.fftn(2, x, plan=pf.plan_fft(None, (n, n)), device=cuda_device).cdouble().reshape(ref.shape)
    e_own, e_lib = (float((v - ref).norm() / ref.norm()) for v in (own, lib))
    print(f"rounding {n}: own {e_own:.3e} library {e_lib:.3e}", flush=True)
    assert e_own <= e_lib
