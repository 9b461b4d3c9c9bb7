"""Rounding of the staged derivative gather's sum over coil pairs
(k_gather_dcoord_col).

A call of 32 coils against the sum in 64 bits of 16 calls of one pair each, on
the same grids: weights, taps and a pair's own sum are then identical, and what
is left is the rounding of the 15 additions that join the pairs.  Each of them
errs by at most 2^-24 of its partial sum, uniformly distributed, and the
partial sum of k of 16 independent pairs has sqrt(k / 16) of the result's norm:
2^-24 / sqrt(3) * sqrt(sum_{k=2}^{16} k / 16) = 1.0e-7 of the result, whatever
the kernel width.  A sum that runs over all W^2 rows of all pairs instead
(4.3e-7 at W = 6, 5.6e-7 at W = 8 in an emulation of both orders) does not pass.
"""

import ctypes

import numpy as np
import pytest
import torch

import pyfourier_amd as pf
from pyfourier_amd import _lib, demo
from pyfourier_amd._nufft import _Call

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width", [4, 6, 8])
def test_pairs_are_summed_one_by_one(cuda_device, width):
    C = 32
    print(f"dcoord pairs: W={width}", flush=True)
    coord = demo.golden_means_radial_3d(96, 40)
    plan = pf.plan_nufft(torch.from_numpy(coord), 12, width=width, oversamp=2.0).to(cuda_device)
    call = _Call(plan, cuda_device, None, None, None)
    assert f"gather=k_gather_col<{width}>" in call.describe(C) and f"gather=k_gather_col<{width}>" in call.describe(2)
    M = coord.shape[0] * coord.shape[1]
    g = torch.Generator(device=cuda_device).manual_seed(width)
    grid = torch.randn((C // 2, 24, 24, 24, 2), dtype=torch.complex64, device=cuda_device, generator=g)  # pair-major
    h = torch.randn((M, C), dtype=torch.complex64, device=cuda_device, generator=g)

    def grad(c, gr, hh):
        out = torch.full((M, 3), float("nan"), device=cuda_device)
        desc = call.desc(c, (None, None))
        _lib.check(_lib.lib().pf_interp_grad(call.native.handle, ctypes.byref(desc), _lib.ptr(gr), _lib.ptr(hh), None, 0,
                                             _lib.ptr(out), _lib.stream_of(cuda_device)))
        return out.double()

    whole = grad(C, grid, h)
    parts = sum(grad(2, grid[p].contiguous(), h[:, 2 * p:2 * p + 2].contiguous()) for p in range(C // 2))
    err = float((whole - parts).norm() / parts.norm())
    assert np.isfinite(err) and err < 1.5e-7, err
