"""Calls with field-map segments or a basis at the workspace's limits: the
no-allocation entry point takes them with the coefficients applied on the fly
when the expanded samples would not fit its array, and the expanded samples of
the other entry points stay below 4 GiB."""

import ctypes

import numpy as np
import pytest
import torch

import pyfourier_amd as pf
from pyfourier_amd import _lib, demo
from pyfourier_amd._nufft import _Call

pytestmark = pytest.mark.gpu

PARITY = 1e-5  # two FP32 evaluations of one sum, each within this of the exact one


def _workspace(call, C, seg, op):
    n = ctypes.c_size_t()
    desc = call.desc(C, seg)
    _lib.check(_lib.lib().pf_workspace_size(call.native.handle, ctypes.byref(desc), op, ctypes.byref(n)))
    return n.value


@pytest.mark.parametrize("K,C,frames", [(5, 1, 8), (9, 1, 4)])
def test_noalloc_takes_odd_basis_batches_beyond_the_expanded_size(cuda_device, K, C, frames):
    # samples of 16 and 8 MiB; times K beyond 64 MiB together with the grid
    M = {5: 1 << 21, 9: 1 << 20}[K]
    print(f"noalloc: basis K={K} C={C} M={M}", flush=True)
    rng = np.random.default_rng(K)
    coord = demo.golden_angle_radial_2d(M // 1024, 1024).reshape(frames, M // 1024 // frames, 1024, 2)
    basis = rng.standard_normal((frames, K))
    plan = pf.plan_nufft(torch.from_numpy(coord.astype(np.float32)), 64, width=4, oversamp=2.0).to(cuda_device)
    call = _Call(plan, cuda_device, basis.astype(np.complex64), None, None)
    L = _lib.lib()
    npts = M // frames
    x = torch.from_numpy(demo.complex_gaussian(rng, (C, K, 64, 64))).to(cuda_device)
    y = torch.from_numpy(demo.complex_gaussian(rng, (C, frames, npts))).to(cuda_device)
    for op, src, ref in ((0, x, call.forward(x, _lib.PF_NORM_NONE)), (1, y, call.adjoint(y, _lib.PF_NORM_NONE))):
        assert _workspace(call, C, (None, None), op) > _lib.PF_NOALLOC_SCRATCH_BYTES
        out = torch.full_like(ref, float("nan"))
        desc = call.desc(C, (None, None))
        rc = L.pf_nufft_noalloc(call.native.handle, ctypes.byref(desc), op, _lib.ptr(src), _lib.ptr(out), None,
                                _lib.PF_NORM_NONE, _lib.stream_of(cuda_device))
        assert rc == 0, L.pf_last_error().decode()
        err = float((out - ref).norm() / ref.norm())
        assert err < PARITY, (op, err)


def test_expanded_samples_stay_below_4_gib(cuda_device):
    M, nt = 1 << 20, 1024
    coord = demo.golden_angle_radial_2d(M // nt, nt)
    plan = pf.plan_nufft(torch.from_numpy(coord), 32, width=4, oversamp=2.0).to(cuda_device)
    call = _Call(plan, cuda_device, None, None, None)
    for L, C, expanded in ((15, 32, True), (16, 32, False), (5, 64, True), (9, 64, False)):
        seg = (torch.zeros((L, nt), dtype=torch.complex64, device=cuda_device),
               torch.zeros((L, 32 * 32), dtype=torch.complex64, device=cuda_device))
        assert (M * L * C * 8 < 1 << 32) == expanded
        assert ("k_sort_x" in call.describe(C, seg)) == expanded, call.describe(C, seg)
        grid = L * C * 64 * 64 * 8
        assert (_workspace(call, C, seg, 1) > grid + M * L * C * 8) == expanded
