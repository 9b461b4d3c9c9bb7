"""Timed workloads of the NUFFT engine, called the way a reconstruction calls them.

listed() holds the workloads, draw() more of the same ranges, prepare() what a
caller has before the call (plan, data on the GPU), run() one pass through the
public operators, work() the bytes and operations a pass cannot do without and
exact() the same outputs in 64-bit torch, with none of the package's code.

Every case is a flat dict.  `kind` selects the call:

  fwd, adj, both   nufft, nufft_adj, or one after the other (density weights)
  grad             nufft with image and coordinate gradients of an L2 loss
                   (`segments` > 0: with a time-segmented field map)
  subspace         nufft + nufft_adj of a many-frame scan through a temporal basis
  gram             sparse_gram, the Toeplitz normal operator of an iteration
  batch            an uneven batch of 2-D slices, one NUFFTBatch pass
  cart             masked fftn + ifftn
"""

import math

import numpy as np
import torch

import pyfourier_amd as pf

GOLDEN = (1 + 5 ** 0.5) / 2


def listed():
    return [
        # one small slice, one coil: the latency of the smallest useful call
        dict(name="radial2d_128_1coil", kind="both", dim=2, nz=1, ny=128, nx=128, coils=1, traj="radial", views=64,
             samples=256, width=4, oversamp=2.0, segments=0),
        # the two directions of a 2-D multi-coil spiral slice at the operators' default kernel
        dict(name="spiral2d_256_16coil_fwd", kind="fwd", dim=2, nz=1, ny=256, nx=256, coils=16, traj="spiral", views=48,
             samples=4096, width=4, oversamp=1.25, segments=0),
        dict(name="spiral2d_256_16coil_adj", kind="adj", dim=2, nz=1, ny=256, nx=256, coils=16, traj="spiral", views=48,
             samples=4096, width=4, oversamp=1.25, segments=0),
        # a slice whose matrix follows a field of view, not a power of two, with an odd number of virtual coils
        dict(name="radial2d_211x187_5coil", kind="both", dim=2, nz=1, ny=211, nx=187, coils=5, traj="radial", views=300,
             samples=375, width=4, oversamp=1.25, segments=0),
        # an anisotropic volume with arbitrary matrix sizes at the default kernel
        dict(name="radial3d_90x102x110_6coil", kind="both", dim=3, nz=90, ny=102, nx=110, coils=6, traj="radial", views=3000,
             samples=220, width=4, oversamp=1.25, segments=0),
        # the benchmark's headline: a 3-D multi-coil volume at the accuracy-qualified kernel width
        dict(name="radial3d_128_32coil_w6", kind="both", dim=3, nz=128, ny=128, nx=128, coils=32, traj="radial", views=8192,
             samples=256, width=6, oversamp=2.0, segments=0),
        # a differentiable 3-D acquisition: loss, image gradient and trajectory gradient
        dict(name="radial3d_128_8coil_grad", kind="grad", dim=3, nz=128, ny=128, nx=128, coils=8, traj="radial", views=8192,
             samples=256, width=4, oversamp=2.0, segments=0),
        # the same with an off-resonance map, one 2-D slice
        dict(name="spiral2d_256_8coil_b0_grad", kind="grad", dim=2, nz=1, ny=256, nx=256, coils=8, traj="spiral", views=16,
             samples=4096, width=4, oversamp=2.0, segments=8),
        # a dynamic scan of 500 short spirals projected on 4 temporal coefficients
        dict(name="subspace2d_500frames", kind="subspace", dim=2, nz=1, ny=256, nx=256, coils=8, traj="spiral", frames=500,
             views=1, samples=2048, coeffs=4, width=4, oversamp=2.0, segments=0),
        # the normal operator applied in every iteration of a conjugate-gradient solve
        dict(name="gram2d_256_16coil", kind="gram", dim=2, nz=1, ny=256, nx=256, coils=16, traj="spiral", views=48,
             samples=4096, width=6, oversamp=1.25, segments=0),
        # slices of different matrix sizes and spoke counts in one pass
        dict(name="batch2d_32slices_8coil", kind="batch", dim=2, slices=32, n_small=128, n_mid=192, n_large=256, coils=8,
             traj="radial", min_views=16, max_views=256, samples=256, width=4, oversamp=2.0, layout_seed=7),
        # Cartesian parallel imaging: masked transform and its adjoint
        dict(name="cart2d_256_32coil", kind="cart", dim=2, nz=1, ny=256, nx=256, coils=32),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A matrix size: half of them multiples of 16 as scanners reconstruct, half whatever the field of view gives."""
    n = _log(rng, lo, hi)
    return max(lo, n // 16 * 16) if rng.random() < 0.5 else n


def draw(rng):
    top = work(listed()[5])
    while True:
        kind = rng.choice(["fwd", "adj", "both", "both", "both", "grad", "subspace", "gram", "batch", "cart"])
        coils = _log(rng, 1, 32)
        sigma = rng.choice([1.25, 1.25, 1.5, 2.0])
        c = dict(kind=kind, dim=2, nz=1, coils=coils)
        if kind == "batch":
            c.update(slices=rng.randint(4, 32), n_small=_size(rng, 96, 160), n_mid=_size(rng, 160, 224),
                     n_large=_size(rng, 224, 320), coils=_log(rng, 1, 16), traj="radial", min_views=16,
                     max_views=_log(rng, 64, 300), samples=2 * _log(rng, 96, 200), width=4, oversamp=sigma,
                     layout_seed=rng.randrange(1 << 30))
            del c["nz"]
        elif kind == "cart":
            if rng.random() < 0.3:
                c.update(dim=3, nz=_size(rng, 32, 192), ny=_size(rng, 48, 256), nx=_size(rng, 48, 256))
            else:
                c.update(ny=_size(rng, 64, 512), nx=_size(rng, 64, 512))
        else:
            three = kind in ("fwd", "adj", "both", "grad") and rng.random() < 0.5
            n = [_size(rng, 32, 144) for _ in range(3)] if three else [1] + [_size(rng, 64, 400)] * 2
            if not three and rng.random() < 0.3:
                n[1] = _size(rng, 64, 400)
            m = max(n)
            c.update(dim=3 if three else 2, nz=n[0], ny=n[1], nx=n[2], width=rng.choice([3, 4, 4, 4, 5, 6]), oversamp=sigma,
                     segments=0, samples=2 * rng.randint(m // 2, m + 20), traj="radial")
            if three:
                c.update(views=_log(rng, 200, 8192))
            else:
                c.update(views=_log(rng, 24, 500))
                if rng.random() < 0.5:
                    c.update(traj="spiral", views=rng.randint(8, 64), samples=_log(rng, 1000, 5000))
            if kind == "grad" and not three and rng.random() < 0.6:
                c.update(traj="spiral", views=rng.randint(8, 48), samples=_log(rng, 1000, 5000), segments=rng.randint(4, 8),
                         coils=_log(rng, 1, 16))
            if kind == "grad":
                c.update(coils=min(c["coils"], 16))
            if kind == "subspace":
                c.update(traj="spiral", frames=_log(rng, 40, 500), views=1, samples=_log(rng, 500, 3000),
                         coeffs=rng.randint(2, 6), coils=_log(rng, 1, 12))
            if kind == "gram":
                c.update(width=6)
        w = work(c)
        if w["bytes"] <= top["bytes"] and w["flops"] <= top["flops"]:
            return c


# ---- inputs -----------------------------------------------------------------
def _shape(c):
    return (c["nz"], c["ny"], c["nx"])[3 - c["dim"]:]


def _radial(dim, views, samples, angle):
    n = np.arange(views)
    k = np.linspace(-math.pi, math.pi, samples, endpoint=False)
    if dim == 2:
        a = n * math.pi / GOLDEN + angle
        d = np.stack([np.cos(a), np.sin(a)], -1)
    else:
        z = np.mod(n * 0.46557123, 1.0)
        a = 2 * math.pi * np.mod(n * 0.68232780, 1.0) + angle
        r = np.sqrt(1 - z * z)
        d = np.stack([r * np.cos(a), r * np.sin(a), z], -1)
    return (d[:, None, :] * k[None, :, None]).astype(np.float32)


def _spiral(views, samples, npix, angle):
    tau = np.linspace(0, 1, samples) ** 1.5
    turns = max(1.0, npix / (2.0 * views))
    a = 2 * math.pi * turns * tau[None] + (angle + 2 * math.pi * np.arange(views) / views)[:, None]
    return (math.pi * tau[None, :, None] * np.stack([np.cos(a), np.sin(a)], -1)).astype(np.float32)


def _coord(c, seed):
    """(frames, views, samples, dim) in radians, each seed at another rotation."""
    angle = 2 * math.pi * float(np.random.default_rng(seed).random())
    f = c.get("frames", 1)
    if c["traj"] == "radial":
        k = _radial(c["dim"], f * c["views"], c["samples"], angle)
    else:
        k = _spiral(f * c["views"], c["samples"], max(c["ny"], c["nx"]), angle)
    return torch.from_numpy(k.reshape(f, c["views"], c["samples"], c["dim"]))


def _weight(k):
    """Ramp density weights |k|^(dim-1), largest 1."""
    r = k.double().norm(dim=-1)
    return ((r / r.max()) ** (k.shape[-1] - 1)).float()


def _randn(gen, shape):
    return torch.randn(shape, dtype=torch.complex64, device="cuda", generator=gen)


def _image(gen, coils, planes, shape):
    """Coil images: one complex Gaussian image per plane times smooth coil profiles."""
    x = _randn(gen, (1, planes) + shape)
    if coils == 1:
        return x
    ax = [torch.linspace(-0.5, 0.5, n, device="cuda") for n in shape]
    ctr = torch.rand((coils, len(shape)), device="cuda", generator=gen) - 0.5
    r2 = sum((g.reshape((-1,) + (1,) * (len(shape) - 1 - i)) - ctr[:, i].reshape((-1,) + (1,) * len(shape))) ** 2
             for i, g in enumerate(ax))
    ph = torch.polar(torch.exp(-r2 / 0.18), 6.2 * torch.rand(coils, device="cuda", generator=gen).reshape((-1,) + (1,) * len(shape)).expand_as(r2))
    return x * ph[:, None]


def _basis(frames, coeffs):
    t2 = np.exp(np.linspace(math.log(20), math.log(300), 400))
    s = np.exp(-np.linspace(1, 300, frames)[None] / t2[:, None])
    return torch.from_numpy(np.linalg.svd(s, full_matrices=False)[2][:coeffs].T.astype(np.complex64)).cuda()


def _zmap(c, seed):
    """Smooth field map within +-100 Hz."""
    rng = np.random.default_rng(seed + 1000)
    y, x = np.meshgrid(np.linspace(-0.5, 0.5, c["ny"]), np.linspace(-0.5, 0.5, c["nx"]), indexing="ij")
    f = np.zeros_like(y)
    for s in (1, -1, 1):
        cy, cx = rng.uniform(-0.3, 0.3, 2)
        f += s * np.exp(-((y - cy) ** 2 + (x - cx) ** 2) / (2 * rng.uniform(0.1, 0.3) ** 2))
    return torch.from_numpy((f / np.abs(f).max() * 100.0).astype(np.float32))


def _times(c):
    return torch.linspace(0, 0.01, c["samples"])


def _slices(c):
    rng = np.random.default_rng(c["layout_seed"])
    n = [int(v) for v in rng.choice([c["n_small"], c["n_mid"], c["n_large"]], c["slices"])]
    return n, [int(v) for v in rng.integers(c["min_views"], c["max_views"] + 1, c["slices"])]


def _inputs(c, seed):
    """The arrays of a pass, from the seed alone (prepare and exact both start here)."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    kind = c["kind"]
    if kind == "batch":
        n, views = _slices(c)
        angle = float(np.random.default_rng(seed).random())
        coords = [torch.from_numpy(_radial(2, v, c["samples"], angle + i)) for i, v in enumerate(views)]
        return dict(shapes=n, coords=coords, images=[_randn(gen, (c["coils"], 1, m, m)) for m in n])
    shape = _shape(c)
    if kind == "cart":
        mask = (torch.rand(shape, device="cuda", generator=gen) < 0.3).float()
        return dict(image=_image(gen, c["coils"], 1, shape)[:, 0], mask=mask)
    k = _coord(c, seed)
    d = dict(coord=k, weight=_weight(k).cuda())
    if kind == "subspace":
        d["basis"] = _basis(c["frames"], c["coeffs"])
        d["image"] = _image(gen, c["coils"], c["coeffs"], shape)
    else:
        d["image"] = _image(gen, c["coils"], 1, shape)[:, 0]
    if kind in ("adj", "grad"):
        d["data"] = _randn(gen, (c["coils"],) + tuple(k.shape[1:-1]))
    if c["segments"]:
        d["zmap"] = _zmap(c, seed)
    return d


def prepare(case, seed):
    c, d = case, _inputs(case, seed)
    kind, dev = c["kind"], torch.device("cuda", torch.cuda.current_device())
    s = dict(kind=kind, dim=c["dim"], dev=dev, **d)
    if kind == "batch":
        s["plan"] = pf.plan_nufft_batch(d["coords"], d["shapes"], nbatch=c["coils"], width=c["width"], oversamp=c["oversamp"],
                                        device=dev)
    elif kind == "cart":
        s["plan"] = pf.plan_fft(d["mask"], _shape(c)).to(dev)
    elif kind == "gram":
        s["plan"] = pf.plan_spgram(d["coord"], _shape(c), weight=d["weight"], oversamp=c["oversamp"], width=c["width"], device=dev)
    else:
        opt = dict(zmap=d["zmap"], L=c["segments"], T=_times(c)) if c["segments"] else {}
        s["plan"] = pf.plan_nufft(d["coord"], _shape(c), width=c["width"], oversamp=c["oversamp"], **opt).to(dev)
    if kind == "grad":
        s["image"] = d["image"].requires_grad_()
        s["coord"] = d["coord"].to(dev).requires_grad_()
    return s


def run(state):
    s, kind, dev = state, state["kind"], state["dev"]
    if kind == "fwd":
        return pf.nufft(s["image"], nufft_plan=s["plan"], device=dev)
    if kind == "adj":
        return pf.nufft_adj(s["data"], nufft_plan=s["plan"], weight=s["weight"], device=dev)
    if kind == "both":
        y = pf.nufft(s["image"], nufft_plan=s["plan"], device=dev)
        return y, pf.nufft_adj(y, nufft_plan=s["plan"], weight=s["weight"], device=dev)
    if kind == "grad":
        s["image"].grad = s["coord"].grad = None
        r = pf.nufft(s["image"], s["coord"], nufft_plan=s["plan"], norm="ortho", device=dev) - s["data"]
        r.abs().pow(2).sum().backward()
        return r.detach(), s["image"].grad, s["coord"].grad
    if kind == "subspace":
        y = pf.nufft(s["image"], nufft_plan=s["plan"], basis=s["basis"], device=dev)
        return y, pf.nufft_adj(y, nufft_plan=s["plan"], basis=s["basis"], weight=s["weight"], device=dev)
    if kind == "gram":
        return pf.sparse_gram(s["image"], s["plan"], device=dev)
    if kind == "batch":
        y = s["plan"].forward(s["images"])
        return list(y) + list(s["plan"].adjoint())
    y = pf.fftn(s["dim"], s["image"], plan=s["plan"], device=dev)
    return y, pf.ifftn(s["dim"], y, plan=s["plan"], device=dev)


# ---- the least a pass can do ---------------------------------------------------
def _grid_len(n, sigma):
    return int(np.ceil(np.float32(sigma) * np.float32(n)))


def _fft_flops(points):
    return 5.0 * points * math.log2(max(2, points))


def work(case):
    c, kind, C = case, case["kind"], case["coils"]
    if kind == "batch":
        b = f = 0.0
        for n, v in zip(*_slices(c)):
            m = v * c["samples"]
            b += 2 * C * (n * n + m) * 8 + 8 * m
            f += 2 * C * (4 * m * c["width"] ** 2 + _fft_flops(_grid_len(n, c["oversamp"]) ** 2))
        return dict(bytes=b, flops=f)
    shape = _shape(c)
    n = math.prod(shape)
    if kind == "cart":
        return dict(bytes=2.0 * C * 2 * n * 8 + 4 * n, flops=2 * C * _fft_flops(n))
    if kind == "gram":
        g = n * 2 ** c["dim"]
        return dict(bytes=2.0 * C * n * 8 + 8 * g, flops=C * (2 * _fft_flops(g) + 6.0 * g))
    m = c.get("frames", 1) * c["views"] * c["samples"]
    k, seg = c.get("coeffs", 1), max(1, c["segments"])
    g = math.prod(_grid_len(v, c["oversamp"]) for v in shape)
    b1 = C * (k * n + m) * 8 + 4 * c["dim"] * m + (8 * seg * n if c["segments"] else 0)
    f1 = C * k * seg * (_fft_flops(g) + 4.0 * m * c["width"] ** c["dim"])
    if kind == "grad":  # forward, loss, adjoint and derivative gather
        return dict(bytes=2.0 * b1 + 16 * C * m + 4 * c["dim"] * m, flops=2 * f1 + C * seg * 4.0 * m * c["width"] ** c["dim"] * c["dim"])
    if kind == "fwd":
        return dict(bytes=float(b1), flops=f1)
    if kind == "adj":
        return dict(bytes=float(b1 + 4 * m), flops=f1)
    return dict(bytes=2.0 * b1 + 4 * m, flops=2 * f1)


# ---- the same outputs in 64 bits -----------------------------------------------
_SMALL = (1.0, 3.5156229, 3.0899424, 1.2067492, 0.2659732, 0.0360768, 0.0045813)
_LARGE = (0.39894228, 0.01328592, 0.00225319, -0.00157565, 0.00916281, -0.02057706, 0.02635537, -0.01647633, 0.00392377)


def _poly(t, coef):
    r = torch.zeros_like(t)
    for a in reversed(coef):
        r = r * t + a
    return r


def _kb(x, beta):
    """Kaiser-Bessel kernel: the published I0 polynomials (Abramowitz and Stegun 9.8.1, 9.8.2), which the operator is defined by."""
    u2 = beta * beta * (1 - x * x)
    big = u2.clamp_min(3.75 ** 2).sqrt()
    large = _poly(3.75 / big, _LARGE) * big.exp() / big.sqrt()
    return torch.where(x.abs() > 1, 0.0, torch.where(u2 < 3.75 ** 2, _poly(u2 / 3.75 ** 2, _SMALL), large))


class _Exact:
    """Separable Kaiser-Bessel gridding operator of float32 grid coordinates, computed in 64 bits.  Axes (z, y, x)."""

    def __init__(self, k, shape, width, sigma, unit=1.0 / (2 * math.pi)):
        d = len(shape)
        f = np.float32
        n_xyz = torch.tensor([float(v) for v in shape[::-1]], dtype=torch.float32)
        k = (k.reshape(-1, d).cpu() * (n_xyz * unit if unit else 1.0)).cuda()
        s = f(sigma)
        beta = float(f(math.pi) * f((((np.int16(width) / s) * (s - f(0.5))) ** 2 - f(0.8))) ** f(0.5))
        self.shape, self.width, self.G = tuple(shape), width, tuple(_grid_len(n, sigma) for n in shape)
        self.M, self.d = k.shape[0], d
        scale, self.idx, self.val, self.der, self.apod = 1.0, [], [], [], []
        e = torch.arange(width, device="cuda", dtype=torch.float64)
        for a in range(d):
            n, g = shape[a], self.G[a]
            c = (k[:, d - 1 - a] * float(f(f(g) / f(n))) + float(g // 2)).double()
            taps = torch.ceil(c - width / 2)[:, None] + e
            t = ((taps - c[:, None]) / (width / 2)).requires_grad_()
            w = _kb(t, beta)
            self.der.append(-torch.autograd.grad(w.sum(), t)[0] / (width / 2))
            self.val.append(w.detach())
            self.idx.append(torch.remainder(taps, g).long())
            scale *= float(_kb((math.ceil(-width / 2) + e) / (width / 2), beta).sum())
            i = torch.arange(n, device="cuda", dtype=torch.float64) - n // 2
            v = (beta ** 2 - (math.pi * width * i / g) ** 2).to(torch.complex128).sqrt()
            v = torch.where(v.imag.abs() > 0, 1.0, (v / torch.sinh(v) / (beta / math.sinh(beta))).real)
            self.apod.append(v)
        self.scale = scale

    def _apod(self, x):
        for a, v in enumerate(self.apod):
            x = x * v.reshape((-1,) + (1,) * (self.d - 1 - a))
        return x

    def _box(self):
        return (Ellipsis,) + tuple(slice(g // 2 - n // 2, g // 2 - n // 2 + n) for n, g in zip(self.shape, self.G))

    def _taps(self, j0, j1, axis=None):
        val = [(self.der if a == axis else self.val)[a][j0:j1] for a in range(self.d)]
        for t in np.ndindex(*(self.width,) * self.d):
            flat, w = 0, 1.0
            for a in range(self.d):
                flat = flat * self.G[a] + self.idx[a][j0:j1, t[a]]
                w = w * val[a][:, t[a]]
            yield flat, w

    def grid(self, x, norm):
        """Images (B, *N) -> grids (G, B)."""
        z = torch.zeros((x.shape[0],) + self.G, dtype=torch.complex128, device="cuda")
        z[self._box()] = self._apod(x.to(torch.complex128))
        ax = tuple(range(1, self.d + 1))
        z = torch.fft.fftshift(torch.fft.fftn(torch.fft.ifftshift(z, dim=ax), dim=ax, norm=norm), dim=ax)
        return z.reshape(x.shape[0], -1).T.contiguous()

    def image(self, g, norm):
        """Grids (G, B) -> images (B, *N)."""
        ax = tuple(range(1, self.d + 1))
        z = g.T.reshape((-1,) + self.G)
        z = torch.fft.fftshift(torch.fft.ifftn(torch.fft.ifftshift(z, dim=ax), dim=ax, norm=norm), dim=ax)
        return self._apod(z[self._box()])

    def gather(self, g, j0=0, j1=None, axis=None):
        j1 = self.M if j1 is None else j1
        y = torch.zeros((j1 - j0, g.shape[1]), dtype=torch.complex128, device="cuda")
        for flat, w in self._taps(j0, j1, axis):
            y.addcmul_(w[:, None].to(y.dtype), g[flat])
        return y / self.scale

    def spread(self, y, j0=0, j1=None):
        """Samples (M, B) -> grids (G, B)."""
        j1 = self.M if j1 is None else j1
        g = torch.zeros((math.prod(self.G), 2 * y.shape[1]), dtype=torch.float64, device="cuda")
        v = torch.view_as_real(y.contiguous()).reshape(y.shape[0], -1)
        for flat, w in self._taps(j0, j1):
            g.index_add_(0, flat, w[:, None] * v)
        return torch.view_as_complex(g.reshape(g.shape[0], -1, 2)) / self.scale

    def _step(self):
        return max(1, min(8, int(1.5e8 // max(self.M, math.prod(self.G)))))

    def forward(self, x, norm=None):
        """(C, *N) -> (C, M)."""
        return torch.cat([self.gather(self.grid(p, norm)).T for p in x.split(self._step())])

    def adjoint(self, y, norm=None):
        """(C, M) -> (C, *N)."""
        return torch.cat([self.image(self.spread(p.T.to(torch.complex128)), norm) for p in y.split(self._step())])


def _segments(zmap, t, L):
    """Histogram least-squares field-map interpolators (B (L, nt), Ct (L, *N)) of a real map in Hz, stored in complex64 as a plan keeps them."""
    z = 2 * math.pi * zmap.double()
    lo, hi = float(z.min()), float(z.max())
    h = torch.histc(z.reshape(-1), bins=40, min=lo, max=hi).double()
    e = torch.linspace(lo, hi, 41, dtype=torch.float64)
    zk = 1j * ((e[:-1] + e[1:]) / 2).to(torch.complex128)
    t = t.double()
    tl = (torch.linspace(0, L, L, dtype=torch.float64) / L * t[-1]).to(torch.complex128)
    w = h.to(torch.complex128).sqrt()
    p = torch.linalg.pinv(w[:, None] * torch.exp(-tl[:, None] * zk[None]).T) * w[None]
    b = p @ torch.exp(-zk[:, None] * t[None].to(torch.complex128))
    ct = torch.exp(-tl.reshape((-1,) + (1,) * z.dim()) * (1j * z)[None])
    return b.to(torch.complex64).cuda().to(torch.complex128), ct.to(torch.complex64).cuda().to(torch.complex128)


def exact(case, seed):
    c, d, kind = case, _inputs(case, seed), case["kind"]
    if kind == "batch":
        y, x = [], []
        for k, n, im in zip(d["coords"], d["shapes"], d["images"]):
            op = _Exact(k, (n, n), c["width"], c["oversamp"])
            v = op.forward(im[:, 0])
            y.append(v[:, None])
            x.append(op.adjoint(v)[:, None])
        return y + x
    shape = _shape(c)
    if kind == "cart":
        ax = tuple(range(1, c["dim"] + 1))
        z = torch.fft.ifftshift(d["image"].to(torch.complex128), dim=ax)
        y = torch.fft.fftshift(torch.fft.fftn(z, dim=ax), dim=ax) * d["mask"]
        return y, torch.fft.fftshift(torch.fft.ifftn(torch.fft.ifftshift(y * d["mask"], dim=ax), dim=ax), dim=ax)
    if kind == "gram":
        k = 2.0 * (d["coord"].reshape(-1, c["dim"]) * (torch.tensor([float(v) for v in shape[::-1]]) * (1.0 / (2 * math.pi))))
        big = tuple(2 * n for n in shape)
        op = _Exact(k, big, c["width"], 2.0, unit=None)
        psf = op.adjoint(d["weight"].reshape(1, -1), norm="forward")[0]
        ghat = math.prod(_grid_len(n, c["oversamp"]) for n in shape)
        t = torch.fft.fftn(torch.fft.ifftshift(psf)) / ghat
        out = []
        for x in d["image"]:
            z = torch.zeros(big, dtype=torch.complex128, device="cuda")
            box = tuple(slice(0, n) for n in shape)
            z[box] = x.to(torch.complex128)
            out.append(torch.fft.ifftn(torch.fft.fftn(z) * t)[box])
        return torch.stack(out)
    op = _Exact(d["coord"], shape, c["width"], c["oversamp"])
    ks = tuple(d["coord"].shape[1:-1])
    if kind == "fwd":
        return op.forward(d["image"]).reshape((-1,) + ks)
    if kind == "adj":
        return op.adjoint(d["data"].reshape(c["coils"], -1) * d["weight"].reshape(-1))
    if kind == "both":
        y = op.forward(d["image"])
        return y.reshape((-1,) + ks), op.adjoint(y * d["weight"].reshape(-1))
    if kind == "subspace":
        b = d["basis"].to(torch.complex128).repeat_interleave(op.M // c["frames"], 0)  # (M, K)
        C, K = c["coils"], c["coeffs"]
        y = sum(op.forward(d["image"][:, k]) * b[:, k] for k in range(K))
        yw = y * d["weight"].reshape(-1)
        x = torch.stack([op.adjoint(yw * b[:, k].conj()) for k in range(K)], 1)
        return y.reshape((C, c["frames"]) + ks), x
    # grad: r = A x - data, dL/dx = 2 A^H r, dL/dk = 2 sum_c Re(conj(r) dA/dk x)
    if c["segments"]:
        b, ct = _segments(d["zmap"], _times(c), c["segments"])
        b = b.repeat(1, c["views"])
    else:
        b, ct = [1.0], [1.0]
    r = sum(op.forward(d["image"] * ct[l], "ortho") * b[l] for l in range(len(b))) - d["data"].reshape(c["coils"], -1)
    conj = torch.conj if c["segments"] else (lambda v: v)
    gx = sum(2 * op.adjoint(r * conj(b[l]), "ortho") * conj(ct[l]) for l in range(len(b)))
    gk = torch.zeros((op.M, c["dim"]), dtype=torch.float64, device="cuda")
    for l in range(len(b)):
        for i in range(0, c["coils"], op._step()):
            g = op.grid(d["image"][i:i + op._step()] * ct[l], "ortho")
            for a in range(c["dim"]):
                dy = op.gather(g, axis=a).T * b[l]
                q = 2 * (r[i:i + op._step()].conj() * dy).real.sum(0)
                gk[:, c["dim"] - 1 - a] += q * (op.G[a] / (2 * math.pi))
    return r.reshape((-1,) + ks), gx, gk.reshape(d["coord"].shape)
