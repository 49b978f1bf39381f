"""Workloads of the framework, through its public entry points, for timing and checking.

``listed()`` holds the workloads a program using this framework meets, from a single
small transform to the 3-D normal operator at the operators' default accuracy;
``draw(rng)`` gives further ones from the same ranges, ragged sizes among them.
``prepare(case, seed)`` makes on the GPU what such a program has in hand, ``run(state)``
is one pass and returns its whole outputs, ``exact(case, seed)`` gives those outputs in
64 bits from plain torch (the Gaussian-gridding NUFFT written out tap by tap), and
``work(case)`` counts the bytes and operations the result cannot do without.

Kinds of case:

* ``nufft``: one call of an NUFFT operator: ``forward``, ``backward`` (density-weighted
  adjoint) or ``normal`` (``forward_backward``); ``nspread`` 0 is the operators' default
  accuracy (eps 1e-5), 3 the setting of the repository's benchmark;
* ``frame``: a new trajectory is set, then ``backward``: one frame of a dynamic series;
* ``sense``: the normal operator of ``joint2operators(espirit(maps), NUFFT)``;
* ``train``: one training step (forward and backward) of the differentiable NUFFT with a
  trajectory that was just updated: loss, image gradient, trajectory gradient;
* ``batch``: forward and adjoint of many uneven instances in one ``BatchPlan``;
* ``kspace``: the masked Cartesian FFT operator, ``forward`` then ``backward``;
* ``tv``: the TV prox (40 Chambolle steps), the image step of the ADMM reconstruction;
* ``fista``: a whole SENSE reconstruction, ``FIST_wrap`` on the joint operator.
"""
from __future__ import annotations

import math

import torch

GOLDEN = (1 + 5 ** 0.5) / 2


def listed():
    return [
        # one coil, one small 2-D image: the smallest call, where latency and launches count
        dict(name="radial2d_fwd_small", kind="nufft", op="forward", dim=2, n0=128, n1=128, n2=1, coils=1, traj="radial",
             spokes=128, points=256, nspread=3),
        # real-time imaging: every frame has its own golden-angle spokes, default accuracy
        dict(name="frame2d_8c", kind="frame", op="backward", dim=2, n0=192, n1=192, n2=1, coils=8, traj="radial",
             spokes=34, points=384, nspread=0),
        # the operator an iterative 2-D SENSE reconstruction calls in every iteration
        dict(name="sense2d_normal_32c", kind="sense", dim=2, n0=256, n1=256, n2=1, coils=32, traj="spiral", spokes=48,
             points=2048, nspread=3),
        # a ragged 3-D field of view (lengths with large prime factors), few coils, default accuracy
        dict(name="ragged3d_bwd_3c", kind="nufft", op="backward", dim=3, n0=91, n1=109, n2=75, coils=3, traj="ute",
             spokes=1501, points=203, nspread=0),
        # 3-D multi-coil UTE, the benchmark's geometry: each direction
        dict(name="ute3d_fwd_8c", kind="nufft", op="forward", dim=3, n0=128, n1=128, n2=128, coils=8, traj="ute",
             spokes=4096, points=256, nspread=3),
        dict(name="ute3d_bwd_8c", kind="nufft", op="backward", dim=3, n0=128, n1=128, n2=128, coils=8, traj="ute",
             spokes=4096, points=256, nspread=3),
        # the same at the operators' default accuracy: the normal operator of 3-D solvers (largest)
        dict(name="ute3d_normal_default_8c", kind="nufft", op="normal", dim=3, n0=128, n1=128, n2=128, coils=8, traj="ute",
             spokes=4096, points=256, nspread=0),
        # trajectory learning: the coordinates change every step, so every step re-bins them
        dict(name="train3d_4c", kind="train", dim=3, n0=128, n1=128, n2=128, coils=4, traj="ute", spokes=4096, points=256,
             nspread=3),
        # many patients / slices of uneven size in one set of launches
        dict(name="batch2d_16", kind="batch", dim=2, instances=16, nmin=128, nmax=320, smin=32, smax=400, cmax=32, sizes=4,
             nspread=3),
        # Cartesian masked FFT, multi-coil slice: encode and decode
        dict(name="kspace2d_32c", kind="kspace", dim=2, n0=256, n1=256, n2=1, coils=32),
        # image step of ADMM-TV on one slice
        dict(name="tv2d_256", kind="tv", dim=2, n0=256, n1=256, n2=1, niter=40),
        # whole reconstruction: 20 FISTA iterations of a 32-coil slice
        dict(name="fista2d_32c", kind="fista", dim=2, n0=256, n1=256, n2=1, coils=32, traj="spiral", spokes=48, points=2048,
             nspread=3, niter=20),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["nufft2", "nufft2", "nufft3", "nufft3", "frame", "sense", "train", "batch", "kspace", "tv", "fista"])
    ns = rng.choice([0, 3])
    if kind in ("nufft2", "frame", "sense", "fista"):
        n0, n1 = _log_int(rng, 48, 320), _log_int(rng, 48, 320)
        c = dict(kind="nufft" if kind == "nufft2" else kind, dim=2, n0=n0, n1=n1, n2=1, coils=_log_int(rng, 1, 32),
                 nspread=ns)
        if rng.random() < 0.5:
            c.update(traj="radial", spokes=_log_int(rng, 16, 400), points=2 * max(n0, n1))
        else:
            c.update(traj="spiral", spokes=_log_int(rng, 8, 48), points=_log_int(rng, 256, 2048))
        if kind == "nufft2":
            c["op"] = rng.choice(["forward", "backward", "normal"])
        elif kind == "frame":
            c["op"] = rng.choice(["forward", "backward"])
        elif kind == "fista":
            c["niter"] = rng.randint(5, 20)
        return c
    if kind in ("nufft3", "train"):
        c = dict(kind="nufft" if kind == "nufft3" else "train", dim=3, n0=_log_int(rng, 32, 128),
                 n1=_log_int(rng, 32, 128), n2=_log_int(rng, 32, 128), coils=rng.randint(1, 8 if kind == "nufft3" else 4),
                 traj="ute", spokes=_log_int(rng, 256, 4096), points=_log_int(rng, 64, 256), nspread=ns)
        if kind == "nufft3":
            c["op"] = rng.choice(["forward", "backward", "normal"])
        else:
            c["nspread"] = 3
        return c
    if kind == "batch":
        return dict(kind="batch", dim=2, instances=_log_int(rng, 2, 16), nmin=64, nmax=rng.randint(96, 320), smin=16,
                    smax=_log_int(rng, 32, 400), cmax=_log_int(rng, 1, 32), sizes=rng.randint(2, 6), nspread=3)
    if kind == "kspace":
        if rng.random() < 0.5:
            return dict(kind="kspace", dim=2, n0=_log_int(rng, 64, 512), n1=_log_int(rng, 64, 512), n2=1,
                        coils=_log_int(rng, 1, 32))
        return dict(kind="kspace", dim=3, n0=_log_int(rng, 32, 128), n1=_log_int(rng, 32, 128), n2=_log_int(rng, 32, 128),
                    coils=_log_int(rng, 1, 8))
    if rng.random() < 0.5:
        return dict(kind="tv", dim=2, n0=_log_int(rng, 64, 512), n1=_log_int(rng, 64, 512), n2=1,
                    niter=rng.choice([10, 40]))
    return dict(kind="tv", dim=3, n0=_log_int(rng, 24, 96), n1=_log_int(rng, 24, 96), n2=_log_int(rng, 24, 96),
                niter=rng.choice([10, 40]))


# ---------------------------------------------------------------------------- inputs

def _dev():
    return torch.device("cuda", torch.cuda.current_device()) if torch.cuda.is_available() else torch.device("cpu")


def _gen(seed):
    g = torch.Generator(device=_dev())
    g.manual_seed(int(seed))
    return g


def _modes(case):
    return tuple(case["n%d" % a] for a in range(case["dim"]))


def _randn(shape, g):
    return torch.complex(torch.randn(shape, generator=g, device=_dev()), torch.randn(shape, generator=g, device=_dev()))


def _trajectory(case, g):
    """d float32 arrays of radians: golden-angle radial, variable-density spiral, or
    centre-out spokes on a Fibonacci sphere, turned by an angle of the seed."""
    dev = _dev()
    ns, npt = case["spokes"], case["points"]
    turn = 2 * math.pi * torch.rand((), generator=g, device=dev, dtype=torch.float64)
    s = torch.arange(ns, device=dev, dtype=torch.float64)
    if case["traj"] == "radial":
        th = s * math.pi / GOLDEN + turn
        r = (torch.arange(npt, device=dev, dtype=torch.float64) - npt // 2) / npt
        k = [r[None] * torch.cos(th)[:, None], r[None] * torch.sin(th)[:, None]]
    elif case["traj"] == "spiral":
        t = torch.arange(npt, device=dev, dtype=torch.float64) / npt
        r = 0.5 * t ** 1.5
        th = 2 * math.pi * (case["n0"] / (2.0 * ns)) * t[None] + (2 * math.pi * s / ns)[:, None] + turn
        k = [r[None] * torch.cos(th), r[None] * torch.sin(th)]
    else:
        z = 1 - (2 * s + 1) / ns
        ph = s * math.pi * (3 - math.sqrt(5)) + turn
        rho = torch.sqrt(torch.clamp(1 - z * z, min=0))
        r = torch.arange(npt, device=dev, dtype=torch.float64) / (2 * npt)
        k = [(rho * torch.cos(ph))[:, None] * r[None], (rho * torch.sin(ph))[:, None] * r[None], z[:, None] * r[None]]
    return [(2 * math.pi * c).reshape(-1).float() for c in k]


def _density(coords, dim):
    """Ramp density weights |k|^(d-1) with a floor, as scanners' files hold them."""
    r = torch.sqrt(sum(c.double() ** 2 for c in coords)) / math.pi
    return (r ** (dim - 1)).clamp_min(1e-3).float()


def _axes(modes):
    d = len(modes)
    return [((torch.arange(m, device=_dev(), dtype=torch.float32) + 0.5) / m * 2 - 1).reshape(
        [-1 if b == a else 1 for b in range(d)]) for a, m in enumerate(modes)]


def _phantom(modes, g):
    """Ellipsoids of the seed inside the unit ball, on a bright body."""
    ax = _axes(modes)
    d = len(modes)
    img = (sum((a / 0.85) ** 2 for a in ax) <= 1).float()
    par = torch.rand((12, 2 * d + 1), generator=g, device=_dev())
    for p in par:
        cen, rad = p[:d] * 1.2 - 0.6, p[d:2 * d] * 0.25 + 0.05
        img = img + (p[-1] - 0.4) * (sum(((a - cen[i]) / rad[i]) ** 2 for i, a in enumerate(ax)) <= 1)
    return img


def _maps(modes, nc, g):
    """Smooth coil sensitivities, coil-last, sum of squares 1."""
    ax = _axes(modes)
    d = len(modes)
    par = torch.rand((nc, 2 * d + 1), generator=g, device=_dev())
    S = torch.empty(tuple(modes) + (nc,), dtype=torch.complex64, device=_dev())
    for c in range(nc):
        cen = par[c, :d] * 1.6 - 0.8
        ph = sum((par[c, d + i] * 2 - 1) * 3 * a for i, a in enumerate(ax)) + 6.28 * par[c, -1]
        S[..., c] = torch.polar(torch.exp(-sum((a - cen[i]) ** 2 for i, a in enumerate(ax)) / 0.5), ph)
    return S / torch.linalg.vector_norm(S, dim=-1, keepdim=True).clamp_min(1e-6)


def _image(case, modes, nc, g):
    return (_phantom(modes, g)[..., None] * _maps(modes, nc, g)).contiguous()


def _kdata(coords, modes, nc, g):
    """k-space samples whose magnitude falls off from the centre, as an object's does."""
    r2 = sum((c / math.pi) ** 2 for c in coords)
    return (_randn((coords[0].numel(), nc), g) / (1 + 400 * r2)[:, None]).contiguous()


def _inputs(case, seed):
    """Everything the case is computed from, made from the seed alone."""
    g = _gen(seed)
    kind = case["kind"]
    if kind == "batch":
        u = torch.rand((case["instances"], 3), generator=g, device=_dev()).tolist()
        # instance sizes belong to the case, not to the seed (an uneven but fixed workload)
        ins = []
        for i in range(case["instances"]):
            a, b, c = (i * 0.6180339887) % 1, (i * 0.7548776662 + 0.3) % 1, (i * 0.5698402910 + 0.6) % 1
            n = case["nmin"] + (case["nmax"] - case["nmin"]) * int(a * case["sizes"]) // max(1, case["sizes"] - 1)
            sub = dict(kind="nufft", dim=2, n0=n, n1=n, n2=1, coils=1 + int(c * case["cmax"]), traj="radial",
                       spokes=int(case["smin"] + b * (case["smax"] - case["smin"])), points=2 * n,
                       nspread=case["nspread"])
            sub["coords"] = _trajectory(sub, g)
            sub["image"] = _image(sub, (n, n), sub["coils"], g) * (0.5 + u[i][0])
            ins.append(sub)
        return dict(instances=ins)
    modes = _modes(case)
    if kind == "kspace":
        mask = (torch.rand(modes, generator=g, device=_dev()) < 0.4).float()
        return dict(image=_image(case, modes, case["coils"], g), mask=mask)
    if kind == "tv":
        ax = _axes(modes)
        ph = torch.polar(torch.ones(modes, device=_dev()), sum(0.3 * a for a in ax).expand(modes).contiguous())
        return dict(image=(_phantom(modes, g) * ph + 0.05 * _randn(modes, g)).contiguous())
    coords = _trajectory(case, g)
    nc = case["coils"]
    x = dict(coords=coords, dcf=_density(coords, case["dim"]))
    if kind in ("nufft", "frame"):
        if case["op"] == "backward":
            x["data"] = _kdata(coords, modes, nc, g)
        else:
            x["data"] = _image(case, modes, nc, g)
        return x
    if kind == "train":
        f = _image(case, modes, nc, g)
        x["image"] = (0.9 * f + 0.05 * _randn(f.shape, g)).contiguous()
        x["target"] = 30 * _kdata(coords, modes, nc, g)
        return x
    x["maps"] = _maps(modes, nc, g)
    if kind == "sense":
        x["data"] = _phantom(modes, g).to(torch.complex64)[..., None].contiguous()
    else:  # fista: noisy samples of a phantom, scaled as optscaling does
        ph = _phantom(modes, g)[..., None] * x["maps"]
        p = _Exact(modes, _nspread(case), coords)
        y = p.type2(ph.to(torch.complex128))
        y = y + 1e-3 * y.abs().max() * _randn(y.shape, g)
        x["data"] = (y / p.type1(y, x["dcf"]).abs().max()).to(torch.complex64).contiguous()
    return x


def _nspread(case):
    return case["nspread"] or 5  # eps 1e-5 by the reference rule


def _shown(case):
    return dict(rat=2, nspread=3) if case["nspread"] else {}


# ---------------------------------------------------------------------------- one pass

def prepare(case, seed):
    x = _inputs(case, seed)
    kind = case["kind"]
    st = dict(case=case, x=x)
    if kind == "batch":
        from mripy_amd.batch import BatchPlan
        ins = [dict(modes=(i["n0"], i["n1"]), coords=i["coords"], ncoils=i["coils"]) for i in x["instances"]]
        st["plan"] = BatchPlan(ins, rat=2, nspread=case["nspread"])
        st["images"] = [i["image"] for i in x["instances"]]
    elif kind == "kspace":
        from mripy_amd.cfft import FFT2d_kmask_hip, FFTnd_kmask_hip
        if case["dim"] == 2:
            x["mask"] = x["mask"][..., None].expand(x["image"].shape).contiguous()
        st["op"] = (FFT2d_kmask_hip if case["dim"] == 2 else FFTnd_kmask_hip)(x["mask"])
    elif kind == "train":
        from mripy_amd.autograd import NUFFT
        st["op"] = NUFFT(_modes(case), ncoils=case["coils"], rat=2, nspread=case["nspread"])
        st["coords"] = torch.stack(x["coords"])
    elif kind != "tv":
        from mripy_amd.operators import NUFFT2d_hip, NUFFT3d_hip, espirit, joint2operators
        cls = NUFFT2d_hip if case["dim"] == 2 else NUFFT3d_hip
        st["op"] = cls(_modes(case), x["dcf"], *x["coords"], **_shown(case))
        if kind in ("sense", "fista"):
            st["op"] = joint2operators(espirit(x["maps"]), st["op"])
    return st


def run(st):
    case, x = st["case"], st["x"]
    kind = case["kind"]
    if kind == "nufft" or kind == "frame":
        op = st["op"]
        if kind == "frame":
            op.set_ktraj(*x["coords"], dcf=x["dcf"])
        if case["op"] == "forward":
            return op.forward(x["data"])
        if case["op"] == "backward":
            return op.backward(x["data"])
        return op.forward_backward(x["data"])
    if kind == "sense":
        return st["op"].forward_backward(x["data"])
    if kind == "train":
        coords = st["coords"].clone().requires_grad_()  # the optimiser's updated trajectory
        f = x["image"].detach().requires_grad_()
        loss = (st["op"](f, coords) - x["target"]).abs().pow(2).sum()
        gf, gc = torch.autograd.grad(loss, (f, coords))
        return dict(loss=loss.detach(), image=gf, coords=gc)
    if kind == "batch":
        ys = st["plan"].type2(st["images"])
        return ys + st["plan"].adjoint(ys)
    if kind == "kspace":
        k = st["op"].forward(x["image"])
        return k, st["op"].backward(k)
    if kind == "tv":
        from mripy_amd.solvers import prox_tv2d_r, prox_tv3d
        return (prox_tv2d_r if case["dim"] == 2 else prox_tv3d)(x["image"], 0.2, niter=case["niter"])
    from mripy_amd.solvers import FIST_wrap
    return FIST_wrap(st["op"], None, x["data"], Nite=case["niter"], step=0.5, th=0.002)


# ---------------------------------------------------------------------------- 64 bits

class _Exact:
    """The Gaussian-gridding NUFFT in float64, tap by tap (oversampling 2): window cell
    m = 1 + floor(xi / h), taps m - ns .. m + ns - 1, weights exp(-(xi - h g)^2 / 4 tau)."""

    def __init__(self, modes, ns, coords):
        self.modes, self.ns, self.d = tuple(modes), ns, len(modes)
        self.nf = tuple(max(2 * m, 2 * ns) for m in modes)
        self.G = math.prod(self.nf)
        self.M = coords[0].numel()
        self.tau = math.pi * ns / 3.0 / modes[0] ** 2
        self.idx, self.w, self.dw = [], [], []
        for a, c in enumerate(coords):
            h = 2 * math.pi / self.nf[a]
            xi = torch.remainder(c.double(), 2 * math.pi)
            m = 1 + torch.floor(xi / h).long()
            tap = m[None] - ns + torch.arange(2 * ns, device=c.device)[:, None]
            u = xi[None] - h * tap.double()
            w = torch.exp(-u * u / (4 * self.tau))
            self.idx.append(torch.remainder(tap, self.nf[a]))
            self.w.append(w)
            self.dw.append(-w * u / (2 * self.tau))
        k = [torch.arange(m, device=_dev()) - m // 2 for m in modes]
        self.pos = [torch.remainder(v, n) for v, n in zip(k, self.nf)]
        self.deap = 1.0
        for a, v in enumerate(k):
            e = torch.exp(self.tau * v.double() ** 2)
            self.deap = self.deap * e.reshape([-1 if b == a else 1 for b in range(self.d)] + [1])
        self.deap = self.deap * (math.pi / self.tau) ** (self.d / 2)
        self.cell = None
        for a in range(self.d):
            p = self.pos[a].reshape([-1 if b == a else 1 for b in range(self.d)])
            self.cell = p if self.cell is None else self.cell * self.nf[a] + p

    def _taps(self, grad=None):
        """Per tap: flat cell index and weight (grad: the derivative along that axis)."""
        for t in range((2 * self.ns) ** self.d):
            js = [(t // (2 * self.ns) ** a) % (2 * self.ns) for a in reversed(range(self.d))]
            cell, w = 0, 1.0
            for a, j in enumerate(js):
                cell = cell * self.nf[a] + self.idx[a][j]
                w = w * (self.dw if grad == a else self.w)[a][j]
            yield cell, w

    def _grid(self, img):
        nc = img.shape[-1]
        g = torch.zeros((self.G, nc), dtype=torch.complex128, device=img.device)
        g[self.cell.reshape(-1)] = (img.to(torch.complex128) * self.deap).reshape(-1, nc)
        return torch.fft.fftn(g.reshape(self.nf + (nc,)), dim=tuple(range(self.d))).reshape(self.G, nc)

    def _gather(self, grid, grad=None):
        out = torch.zeros((self.M, grid.shape[1]), dtype=torch.complex128, device=grid.device)
        for cell, w in self._taps(grad):
            out.addcmul_(grid[cell], w[:, None].to(torch.complex128))
        return out / self.G

    def type2(self, img):
        return self._gather(self._grid(img))

    def adjoint(self, y):
        nc = y.shape[1]
        v = torch.view_as_real(y.to(torch.complex128).contiguous()).reshape(self.M, 2 * nc)
        g = torch.zeros((self.G, 2 * nc), dtype=torch.float64, device=y.device)
        for cell, w in self._taps():
            g.index_add_(0, cell, v * w[:, None])
        g = torch.view_as_complex(g.reshape(self.nf + (nc, 2)))
        g = torch.fft.ifftn(g, dim=tuple(range(self.d))).reshape(self.G, nc)
        return g[self.cell.reshape(-1)].reshape(self.modes + (nc,)) * self.deap

    def type1(self, y, dcf=None):
        return self.adjoint(y if dcf is None else y * dcf.double()[:, None]) / self.M


def exact(case, seed):
    x = _inputs(case, seed)
    kind = case["kind"]
    if kind == "batch":
        ys, ims = [], []
        for i in x["instances"]:
            p = _Exact((i["n0"], i["n1"]), case["nspread"], i["coords"])
            ys.append(p.type2(i["image"]))
            ims.append(p.adjoint(ys[-1]))
        return ys + ims
    modes = _modes(case)
    ax = tuple(range(case["dim"]))
    if kind == "kspace":
        im = x["image"].to(torch.complex128)
        m = x["mask"].double()[..., None]
        k = torch.fft.ifftshift(torch.fft.fftn(torch.fft.fftshift(im, dim=ax), dim=ax), dim=ax) * m
        return k, torch.fft.ifftshift(torch.fft.ifftn(torch.fft.fftshift(k, dim=ax), dim=ax), dim=ax)
    if kind == "tv":
        return _tv(x["image"].to(torch.complex128), 0.2, 0.1, case["niter"], case["dim"])
    p = _Exact(modes, _nspread(case), x["coords"])
    if kind in ("nufft", "frame"):
        if case["op"] == "forward":
            return p.type2(x["data"])
        if case["op"] == "backward":
            return p.type1(x["data"], x["dcf"])
        return p.type1(p.type2(x["data"]), x["dcf"])
    if kind == "train":
        grid = p._grid(x["image"])
        r = p._gather(grid) - x["target"]
        gc = torch.stack([(torch.conj(2 * r) * p._gather(grid, a)).real.sum(1) for a in range(p.d)])
        return dict(loss=(r.abs() ** 2).sum(), image=p.adjoint(2 * r), coords=gc)
    S = x["maps"].to(torch.complex128)

    def back(y):
        return (p.type1(y, x["dcf"]) * torch.conj(S)).sum(-1, keepdim=True)

    if kind == "sense":
        return back(p.type2(x["data"] * S))
    b = back(x["data"].to(torch.complex128))
    y = 0.5 * b
    acc, pre, t = torch.zeros_like(y), y, 1.0
    out = None
    for _ in range(case["niter"]):
        acc = acc - 0.5 * (back(p.type2(y * S)) - b)
        m = acc.abs()
        out = acc / (m + 1e-6) * (m - 0.002).clamp_min(0)
        tn = (1 + math.sqrt(1 + 4 * t * t)) / 2
        y = out + (t - 1) / tn * (out - pre)
        pre, t = out, tn
    return out


def _tv(y, lam, step, niter, nd):
    """Chambolle's dual steps with the reference's amplitude: complex squares, and the
    maximum with 1 taken in (real, imaginary) order."""
    G = [torch.zeros_like(y) for _ in range(nd)]

    def diff(v, a):
        d = torch.zeros_like(v)
        n = v.shape[a]
        d.narrow(a, 0, n - 1).copy_(v.narrow(a, 1, n - 1) - v.narrow(a, 0, n - 1))
        return d

    def div(g, a):
        n = g.shape[a]
        o = torch.zeros_like(g)
        o.narrow(a, 0, n - 1).sub_(g.narrow(a, 0, n - 1))
        o.narrow(a, 1, n - 1).add_(g.narrow(a, 0, n - 1))
        return o

    for _ in range(niter):
        D = sum(div(G[a], a) for a in range(nd)) - y / lam
        G = [G[a] - step * diff(D, a) for a in range(nd)]
        amp = torch.sqrt(sum(v * v for v in G))
        keep = (amp.real > 1) | ((amp.real == 1) & (amp.imag >= 0))
        amp = torch.where(keep, amp, torch.ones_like(amp))
        G = [v / amp for v in G]
    return y - lam * sum(div(G[a], a) for a in range(nd))


# ---------------------------------------------------------------------------- work

def _fft_flops(lengths):
    n = math.prod(lengths)
    return 5.0 * n * math.log2(max(2, n))


def _nufft_work(modes, M, nc, ns, passes=1):
    """One transform: image, samples, coordinates once; grid FFT, window products, deapodization."""
    d = len(modes)
    nf = [max(2 * m, 2 * ns) for m in modes]
    fl = nc * (_fft_flops(nf) + 4.0 * M * (2 * ns) ** d + 6.0 * math.prod(modes))
    return dict(bytes=8.0 * nc * (math.prod(modes) + M) + 4.0 * d * M, flops=passes * fl)


def work(case):
    kind = case["kind"]
    if kind == "batch":
        w = dict(bytes=0.0, flops=0.0)
        for i in range(case["instances"]):
            a, b, c = (i * 0.6180339887) % 1, (i * 0.7548776662 + 0.3) % 1, (i * 0.5698402910 + 0.6) % 1
            n = case["nmin"] + (case["nmax"] - case["nmin"]) * int(a * case["sizes"]) // max(1, case["sizes"] - 1)
            M = int(case["smin"] + b * (case["smax"] - case["smin"])) * 2 * n
            nc = 1 + int(c * case["cmax"])
            v = _nufft_work((n, n), M, nc, case["nspread"], 2)
            w["bytes"] += v["bytes"] + 8.0 * nc * n * n
            w["flops"] += v["flops"]
        return w
    modes = _modes(case)
    N = math.prod(modes)
    if kind == "kspace":
        nc = case["coils"]
        return dict(bytes=8.0 * N * nc * 3 + 4.0 * N, flops=2 * nc * _fft_flops(modes))
    if kind == "tv":
        # image in and out; per step and pixel: differences, updates, amplitude, quotients
        return dict(bytes=16.0 * N, flops=float(case["niter"]) * N * 24 * case["dim"])
    M, nc, ns = case["spokes"] * case["points"], case["coils"], _nspread(case)
    d = case["dim"]
    if kind in ("nufft", "frame"):
        if case["op"] == "normal":
            return dict(bytes=16.0 * N * nc + 4.0 * (d + 1) * M, flops=_nufft_work(modes, M, nc, ns, 2)["flops"])
        w = _nufft_work(modes, M, nc, ns)
        if case["op"] == "backward":
            w["bytes"] += 4.0 * M
        return w
    if kind == "train":
        w = _nufft_work(modes, M, nc, ns, 2)
        return dict(bytes=16.0 * N * nc + 8.0 * M * nc + 8.0 * d * M, flops=w["flops"] + 4.0 * d * nc * M * (2 * ns) ** d)
    it = 1 if kind == "sense" else case["niter"]
    fl = it * (_nufft_work(modes, M, nc, ns, 2)["flops"] + 16.0 * N * nc)
    extra = 16.0 * N if kind == "sense" else 8.0 * N + 8.0 * M * nc
    return dict(bytes=8.0 * N * nc + 4.0 * (d + 1) * M + extra, flops=fl)
