"""Each kernel variant at the sizes where its choice changes, against the FP64 oracle or
torch in 64 bits.  Tolerance: rel-L2 <= 1e-5 for FP32 results (the repository's bound),
FP64 results to 1e-10."""
import numpy as np
import pytest

from oracle import nufft_oracle as O

pytestmark = pytest.mark.gpu

TOL = 1e-5


def rel(a, b):
    a = np.asarray(a, np.complex128)
    b = np.asarray(b, np.complex128)
    return float(np.linalg.norm((a - b).ravel()) / np.linalg.norm(b.ravel()))


def _cnormal(rng, shape):
    return (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(np.complex64)


@pytest.mark.parametrize("modes", [(24, 20), (12, 10, 14)])
@pytest.mark.parametrize("nc", [1, 2, 3, 5, 8, 9])
def test_spread_coil_groups(modes, nc):
    print("case: adjoint", modes, nc, flush=True)
    from mripy_amd.plan import Plan
    rng = np.random.default_rng(7)
    M = 1500
    coords = [(np.pi * (2 * rng.random(M) - 1)).astype(np.float32) for _ in modes]
    y = _cnormal(rng, (M, nc))
    P = Plan(modes, ncoils=nc, rat=2, nspread=3).set_points(coords)
    p = O.Params(modes, rat=2, nspread=3)
    ref = O.type1([c.astype(np.float64) for c in coords], y.astype(np.complex128), p)
    assert rel(P.type1(y), ref) <= TOL


# (shape, rank): one long line, odd and even batches, unit axes, ragged column blocks,
# several slabs per block, the longest covered length, and lengths left to rocFFT
@pytest.mark.parametrize("shape,rank", [((2048,), 1), ((2, 3), 2), ((1, 30, 1), 3), ((45, 1, 2), 2), ((27, 50, 3), 2),
                                        ((20, 25, 21), 2), ((9, 8, 15, 2), 3), ((160, 6, 33), 2), ((4, 2048, 1), 2),
                                        ((17, 31), 2), ((1001, 3), 2), ((2021, 1), 2), ((251, 8, 3), 2), ((2049,), 1),
                                        ((12, 2050), 2), ((257, 4), 2)])
@pytest.mark.parametrize("batch_mask", [False, True])
def test_cartesian_axis_passes(shape, rank, batch_mask):
    """gn_fft_c2c with shifts and mask, both directions, out of place, in place and from a
    base that is only 8-byte aligned."""
    import torch
    from mripy_amd import _lib
    from mripy_amd.cfft import _c2c
    print("case: c2c", shape, rank, batch_mask, flush=True)
    rng = np.random.default_rng(sum(shape))
    x = _cnormal(rng, shape)
    ax = tuple(range(rank))
    mask = rng.random(shape if batch_mask else shape[:rank]).astype(np.float32)
    mb = mask if batch_mask else mask.reshape(shape[:rank] + (1,) * (len(shape) - rank))
    xs = np.fft.fftshift(x.astype(np.complex128), ax)
    fwd = np.fft.ifftshift(np.fft.fftn(xs, axes=ax), ax) * mb
    inv = np.fft.ifftshift(np.fft.ifftn(xs, axes=ax), ax)
    flags = _lib.GN_FFT_SHIFT_IN | _lib.GN_FFT_SHIFT_OUT
    buf = torch.empty(x.size + 1, dtype=torch.complex64, device="cuda")
    for t in (torch.as_tensor(x).cuda(), buf[1:].view(shape)):
        t.copy_(torch.as_tensor(x))
        assert rel(_c2c(t, rank, _lib.GN_FFT_FORWARD, flags, torch.as_tensor(mask).cuda()).cpu(), fwd) <= 2e-6
        assert rel(_c2c(t, rank, _lib.GN_FFT_INVERSE, flags).cpu(), inv) <= 2e-6
        assert rel(t.cpu(), x) == 0
    import ctypes
    shp = (ctypes.c_int64 * 3)(*(shape[:rank] + (1,) * (3 - rank)))
    batch = int(np.prod(shape[rank:])) if len(shape) > rank else 1
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.check(_lib.load().gn_fft_c2c(rank, shp, batch, _lib.GN_FFT_INVERSE, flags, None, 1, t.data_ptr(), t.data_ptr(),
                                      st))
    assert rel(t.cpu(), inv) <= 2e-6


@pytest.mark.parametrize("modes,nc", [((7, 11), 3), ((13, 49), 2), ((17, 33), 17), ((251, 20), 2), ((24, 254), 40),
                                      ((43, 34), 1), ((9, 17, 22), 3), ((17, 10, 29), 9), ((257, 12), 2)])
def test_prime_grid_lengths(modes, nc):
    """Grid lengths with primes 7 .. 251 (register butterflies, direct-sum stages, both on one
    axis, two direct sums) and 257 (rocFFT): both directions, SENSE, and the batched launch
    equal to the plain plan."""
    import torch
    from mripy_amd.batch import BatchPlan
    from mripy_amd.plan import Plan
    print("case: prime lengths", modes, nc, flush=True)
    rng = np.random.default_rng(sum(modes))
    M = 900
    coords = [(np.pi * (2 * rng.random(M) - 1)).astype(np.float32) for _ in modes]
    c64 = [c.astype(np.float64) for c in coords]
    F, y, x = _cnormal(rng, modes + (nc,)), _cnormal(rng, (M, nc)), _cnormal(rng, modes)
    P = Plan(modes, ncoils=nc, rat=2, nspread=3).set_points(coords)
    p = O.Params(modes, rat=2, nspread=3)
    assert rel(P.type2(F), O.type2(c64, F.astype(np.complex128), p)) <= TOL
    want = O.type1(c64, y.astype(np.complex128), p)
    assert rel(P.type1(y), want) <= TOL
    P.set_sense(F)
    assert rel(P.sense_type2(x), O.type2(c64, x[..., None] * F.astype(np.complex128), p)) <= TOL
    assert rel(P.sense_type1(y), (np.conj(F) * want).sum(-1)) <= TOL
    B = BatchPlan([dict(modes=modes, coords=[torch.as_tensor(c).cuda() for c in coords], ncoils=nc)] * 2)
    yt, Ft = torch.as_tensor(y).cuda(), torch.as_tensor(F).cuda()
    assert all(rel(o.cpu(), P.type2(Ft).cpu()) <= 1e-6 for o in B.type2([Ft, Ft]))
    assert all(rel(o.cpu(), P.type1(yt).cpu()) <= 1e-6 for o in B.type1([yt, yt]))


def _tv_ref(x, ndim, niter, amp):
    from oracle import solvers_oracle as R
    tv = R.TV2d_r() if ndim == 2 else R.TV3d()
    G = np.zeros(x.shape + (ndim,))
    for _ in range(niter):
        G = G - 0.1 * tv.grad(tv.Div(G) - x / 0.3)
        a = tv.amp(G) if amp == "reference" else np.sqrt((np.abs(G) ** 2).sum(-1, keepdims=True))
        G = G / np.maximum(a, np.ones(a.shape))
    return x - 0.3 * tv.Div(G)


@pytest.mark.parametrize("shape,ndim", [((2, 2), 2), ((18, 19), 2), ((33, 17, 3), 2), ((70, 2), 2), ((2, 2, 2), 3),
                                        ((8, 9, 17), 3), ((11, 3, 8, 2), 3)])
@pytest.mark.parametrize("niter", [0, 1, 7, 8, 15])
def test_tv_steps_per_launch(shape, ndim, niter):
    """Chambolle steps split over launches, at the edges of tiles and regions: against the
    FP64 oracle per trailing element, both amplitudes."""
    import torch
    from mripy_amd import solvers as S
    print("case: tv", shape, ndim, niter, flush=True)
    rng = np.random.default_rng(niter + sum(shape))
    x = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    prox = S.prox_tv2d_r if ndim == 2 else S.prox_tv3d
    for amp in ("reference", "modulus"):
        got = prox(torch.as_tensor(x).cuda(), 0.3, niter=niter, amp=amp).cpu().numpy()
        cols = x.reshape(shape[:ndim] + (-1,))
        want = np.stack([_tv_ref(cols[..., k], ndim, niter, amp) for k in range(cols.shape[-1])], -1)
        assert rel(got, want.reshape(shape)) <= 1e-10
        g32 = prox(torch.as_tensor(x.astype(np.complex64)).cuda(), 0.3, niter=niter, amp=amp)
        assert g32.dtype == torch.complex64 and rel(g32.cpu(), want.reshape(shape)) <= 1e-5


def test_tv_extreme_values():
    """Fields beyond the range of a^2 + b^2 follow the rule; infinities and NaN stay local."""
    import torch
    from mripy_amd import solvers as S
    rng = np.random.default_rng(3)
    for scale in (1e100, 1e-200):
        x = scale * (rng.standard_normal((12, 9)) + 1j * rng.standard_normal((12, 9)))
        want = _tv_ref(x, 2, 3, "reference")
        got = S.prox_tv2d_r(torch.as_tensor(x).cuda(), 0.3, niter=3).cpu().numpy()
        assert np.isfinite(want).all() and np.abs(got - want).max() <= 1e-10 * scale
    for bad in (np.nan, np.inf):
        x = rng.standard_normal((20, 40)) + 0j
        x[3, 4] = bad
        got = S.prox_tv2d_r(torch.as_tensor(x).cuda(), 0.3, niter=2).cpu().numpy()
        assert np.isfinite(got[10:, 12:]).all() and not np.isfinite(got[3, 4])


@pytest.mark.parametrize("modes,ns", [((4, 8), 3), ((21, 9), 3), ((30, 25), 5), ((4, 4, 4), 2), ((5, 9, 7), 3),
                                      ((10, 6, 13), 4)])
@pytest.mark.parametrize("nc,layout", [(1, "coil_last"), (2, "coil_major"), (4, "coil_last"), (3, "coil_major"),
                                       (17, "coil_last")])
def test_spread_tiles(modes, ns, nc, layout):
    """Axes of one tile, ragged last tiles and rows of odd length, both layouts, samples in a
    cluster (tiles of several work items) and spread out, with density weights: type 1 and
    the spread alone (every tile written)."""
    from mripy_amd.plan import Plan
    print("case: spread tiles", modes, ns, nc, layout, flush=True)
    rng = np.random.default_rng(nc + sum(modes))
    M = 700
    coords = [np.concatenate([0.02 * rng.standard_normal(400) + 0.4, np.pi * (2 * rng.random(300) - 1)]).astype(np.float32)
              for _ in modes]
    y, dcf = _cnormal(rng, (M, nc)), rng.random(M).astype(np.float32)
    P = Plan(modes, ncoils=nc, rat=2, nspread=ns, layout=layout).set_points(coords, dcf=dcf)
    p = O.Params(modes, rat=2, nspread=ns)
    c64 = [c.astype(np.float64) for c in coords]
    yl = y if layout == "coil_last" else np.ascontiguousarray(y.T)
    want = O.type1(c64, dcf[:, None].astype(np.float64) * y, p)
    got = P.type1(yl)
    assert rel(got if layout == "coil_last" else np.moveaxis(got, 0, -1), want) <= TOL
    grid = P.grid_spread(yl)
    ref = np.moveaxis(O.spread(c64, y.astype(np.complex128), p.nf, p.ns, p.tau), -1, 0)
    assert rel(grid, ref) <= TOL


@pytest.mark.parametrize("modes", [(5, 6), (64, 60), (6, 5, 7), (40, 33, 36)])
@pytest.mark.parametrize("M", [1, 64, 2047, 2049, 9000])
def test_set_points_sizes(modes, M):
    """Scan tiles, digit widths and item counts at their edges: the sample order is the stable
    order by gather tile, and both directions match the oracle.  A plan that has refused a
    non-finite coordinate takes the next points."""
    from mripy_amd.plan import Plan
    print("case: set_points", modes, M, flush=True)
    rng = np.random.default_rng(M)
    coords = [(np.pi * (2 * rng.random(M) - 1)).astype(np.float32) for _ in modes]
    c64 = [c.astype(np.float64) for c in coords]
    P = Plan(modes, ncoils=1, rat=2, nspread=3)
    bad = [c.copy() for c in coords]
    bad[1][M // 2] = np.nan
    for _ in range(2):
        with pytest.raises(ValueError):
            P.set_points(bad)
        P.set_points(coords)
        s = [(1 + np.floor(np.mod(c, 2 * np.pi) / (2 * np.pi / n)).astype(int) - 3) % n for c, n in zip(c64, P.nf)]
        key = 0
        for a, t in enumerate(P.gather_tiles):
            key = key * -(-P.nf[a] // t) + s[a] // t
        assert np.array_equal(P.sample_order(), np.argsort(key, kind="stable"))
    p = O.Params(modes, rat=2, nspread=3)
    F, y = _cnormal(rng, modes + (1,)), _cnormal(rng, (M, 1))
    assert rel(P.type2(F), O.type2(c64, F.astype(np.complex128), p)) <= TOL
    assert rel(P.type1(y), O.type1(c64, y.astype(np.complex128), p)) <= TOL


@pytest.mark.parametrize("layout", ["coil_last", "coil_major"])
@pytest.mark.parametrize("modes,nc", [((30, 40), 7), ((40, 2), 33), ((50, 3, 4), 5), ((160, 250), 16),
                                      ((160, 251), 9), ((32, 17), 64)])
def test_row_pass_blocks(modes, nc, layout):
    """Row passes of few lines (fewer coils per block) and SENSE combines whose block holds
    all coils, below and above the size that takes more threads, odd sizes.  (The window's
    width follows the first mode count, which must not be far below the others.)"""
    print("case: row passes", modes, nc, layout, flush=True)
    from mripy_amd.plan import Plan
    rng = np.random.default_rng(nc)
    M = 700
    coords = [(np.pi * (2 * rng.random(M) - 1)).astype(np.float32) for _ in modes]
    c64 = [c.astype(np.float64) for c in coords]
    S, y, x = _cnormal(rng, modes + (nc,)), _cnormal(rng, (M, nc)), _cnormal(rng, modes)
    P = Plan(modes, ncoils=nc, rat=2, nspread=3, layout=layout).set_points(coords)
    out = (lambda a: np.ascontiguousarray(np.moveaxis(a, -1, 0))) if layout == "coil_major" else (lambda a: a)
    p = O.Params(modes, rat=2, nspread=3)
    img, smp = O.type1(c64, y.astype(np.complex128), p), O.type2(c64, S.astype(np.complex128), p)
    assert rel(P.type1(out(y)), out(img)) <= TOL
    assert rel(P.type2(out(S)), out(smp)) <= TOL
    P.set_sense(out(S))
    assert rel(P.sense_type1(out(y)), (np.conj(S) * img).sum(-1)) <= TOL
    assert rel(P.sense_type2(x), out(O.type2(c64, x[..., None] * S.astype(np.complex128), p))) <= TOL


class _Diag:
    """x -> d x, with or without the forward_backward the wrappers dispatch on."""

    def __init__(self, d, fb):
        self.forward = lambda x: d * x
        self.backward = lambda x: d.conj() * x
        if fb:
            self.forward_backward = lambda x: d.conj() * (d * x)


@pytest.mark.parametrize("shape", [(1,), (255, 1), (16, 16), (17, 31, 3), (300, 219)])
@pytest.mark.parametrize("wrap", ["IST_wrap", "FIST_wrap"])
@pytest.mark.parametrize("fb", [True, False])
def test_ist_fista_update(shape, wrap, fb):
    """The update kernel against the same iteration in 64 bits (which takes the separate
    operations), for a start that has zeros; complex views and tensor thresholds keep the
    separate operations and agree.  Tolerance: ten FP32 roundings of acc per iteration,
    |acc| <= |x| + th."""
    import torch
    from mripy_amd import solvers as S
    print("case: update", shape, wrap, fb, flush=True)
    g = torch.Generator().manual_seed(3)
    b, d = (torch.randn(shape, generator=g, dtype=torch.complex64).cuda() for _ in range(2))
    b.view(-1)[1::5] = 0
    N, kw = 6, dict(Nite=6, step=0.3, th=0.05)
    want = getattr(S, wrap)(_Diag(d.to(torch.complex128), fb), b=b.to(torch.complex128), **kw)
    got = getattr(S, wrap)(_Diag(d, fb), b=b, **kw)
    lim = N * 10 * 6e-8 * float(want.norm() + 0.05 * want.numel() ** 0.5)
    assert got.dtype == torch.complex64 and float((got - want).norm()) <= lim
    th = torch.full(shape, 0.05, device="cuda")
    for v in (getattr(S, wrap)(_Diag(d, fb), b=b, Nite=N, step=0.3, th=th),
              getattr(S, wrap)(_Diag(d.conj(), fb), b=b.conj(), **kw).conj()):
        assert float((got - v).norm()) <= 2 * lim


@pytest.mark.parametrize("th", [0.5, 0.0, -1.0, 1e30])
def test_ist_fista_update_extreme_values(th):
    """Infinities, NaN, the largest and smallest values: as the separate operations."""
    import torch
    from mripy_amd import solvers as S
    inf, nan, big, tiny = float("inf"), float("nan"), 3e38, 1e-42
    v = [0.0, -0.0, 1.5, -inf, inf, nan, big, -big, tiny]
    a = torch.tensor([complex(p, q) for p in v for q in v], dtype=torch.complex64, device="cuda")
    g, xp = torch.zeros_like(a), torch.ones_like(a)
    for step, b in ((0.5, None), (0.5, a.flip(0))):
        want_acc = a - step * (g if b is None else g - b)
        want_x = S.prox_l1_soft_thresh2(want_acc, th)
        want_y = want_x + 0.25 * (want_x - xp)
        acc, x, y = S._descend(g, b, step, a.clone(), th, xp, 0.25)
        for got, want in ((acc, want_acc), (x, want_x), (y, want_y)):
            got, want = torch.view_as_real(got).cpu().numpy(), torch.view_as_real(want).cpu().numpy()
            np.testing.assert_allclose(got, want, rtol=1e-6, atol=1e-40)


def test_ist_fista_update_keeps_gradients():
    import torch
    from mripy_amd import solvers as S
    d = torch.ones(7, dtype=torch.complex64, device="cuda") * 0.5
    b = torch.ones(7, dtype=torch.complex64, device="cuda").requires_grad_()
    for wrap in ("IST_wrap", "FIST_wrap"):
        x = getattr(S, wrap)(_Diag(d, True), b=b, Nite=3, step=0.5, th=0.01)
        (grad,) = torch.autograd.grad(x.abs().sum(), b)
        assert bool((grad.abs() > 0).all())


@pytest.mark.parametrize("modes,ns", [((24, 30), 3), ((20, 17, 22), 3), ((4, 4, 4), 3), ((14, 13, 16), 5), ((5, 6), 9)])
@pytest.mark.parametrize("nc", [1, 2, 3, 4])
@pytest.mark.parametrize("layout", ["coil_last", "coil_major"])
def test_traj_grad_coil_pairs(modes, ns, nc, layout):
    """Even and odd coil counts, both layouts, and grids that a window region wraps whole."""
    print("case: trajectory gradient", modes, ns, nc, layout, flush=True)
    from mripy_amd.plan import Plan
    rng = np.random.default_rng(nc)
    M = 1100
    coords = [(np.pi * (2 * rng.random(M) - 1)).astype(np.float32) for _ in modes]
    F, w = _cnormal(rng, modes + (nc,)), _cnormal(rng, (M, nc))
    out = (lambda a: np.ascontiguousarray(np.moveaxis(a, -1, 0))) if layout == "coil_major" else (lambda a: a)
    import torch
    P = Plan(modes, ncoils=nc, rat=2, nspread=ns, layout=layout).set_points(coords)
    got = P.traj_grad(torch.as_tensor(out(F)).cuda(), torch.as_tensor(out(w)).cuda()).cpu().numpy()
    want = O.traj_grad([c.astype(np.float64) for c in coords], F, w, O.Params(modes, rat=2, nspread=ns))
    assert rel(got, want) <= TOL
