"""pf_copy_items (the batch buffers' loader): odd lengths, misaligned rows,
empty items, more items than one launch holds, and a conjugate view through
NUFFTBatch."""

import ctypes

import numpy as np
import pytest
import torch

import pyfourier_amd as pf
from pyfourier_amd import _lib, demo

pytestmark = pytest.mark.gpu


def test_copy_items_edges(cuda_device):
    rng = np.random.default_rng(0)
    sizes = [(1, 1, 1), (3, 7, 9), (2, 4096, 4096), (2, 4097, 5000), (5, 12289, 12290), (0, 4, 4), (3, 0, 4), (4, 64, 65)]
    sizes += [(1 + i % 3, 5 + i, 8 + i) for i in range(70)]
    srcs, dsts = [], []
    for i, (r, n, st) in enumerate(sizes):
        off = i % 2  # destinations on and off a 16-byte boundary
        srcs.append(torch.randn(max(1, r * n) + off, dtype=torch.complex64, device=cuda_device)[off:off + r * n])
        dsts.append(torch.full((max(1, r) * st + 1,), 7.0, dtype=torch.complex64, device=cuda_device)[off:])
    n = len(sizes)
    LL = ctypes.c_longlong * n
    VP = ctypes.c_void_p * n
    _lib.check(_lib.lib().pf_copy_items(n, VP(*[s.data_ptr() for s in srcs]), VP(*[d.data_ptr() for d in dsts]),
                                        LL(*[s[0] for s in sizes]), LL(*[s[1] for s in sizes]), LL(*[s[2] for s in sizes]),
                                        _lib.stream_of(cuda_device)))
    for (r, m, st), s, d in zip(sizes, srcs, dsts):
        ref = torch.full_like(d, 7.0)
        for k in range(r):
            ref[k * st:k * st + m] = s[k * m:(k + 1) * m]
        assert torch.equal(ref, d), (r, m, st)


def test_copy_items_refuses_bad_sizes(cuda_device):
    one = (ctypes.c_longlong * 1)(2)
    vp = (ctypes.c_void_p * 1)(16)
    bad = (ctypes.c_longlong * 1)(1)
    assert _lib.lib().pf_copy_items(1, vp, vp, one, one, bad, None) == 1  # rows would overlap: refused before any launch
    assert _lib.lib().pf_copy_items(1, None, vp, one, one, one, None) == 1


def test_batch_loads_a_conjugate_view(cuda_device):
    rng = np.random.default_rng(1)
    coords = [demo.golden_angle_radial_2d(9, 32), demo.golden_angle_radial_2d(5, 32)]
    batch = pf.plan_nufft_batch(coords, [24, 24], nbatch=3, device=cuda_device)
    x = [torch.from_numpy(demo.complex_gaussian(rng, (3, 1, 24, 24))).to(cuda_device) for _ in range(2)]
    a = [y.clone() for y in batch.forward([v.conj() for v in x])]
    b = batch.forward([v.conj().resolve_conj() for v in x])
    assert all(torch.equal(p, q) for p, q in zip(a, b))
