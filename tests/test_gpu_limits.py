"""Calls at the limits of what the library takes: refused with an error, or taken, as
documented."""
import numpy as np
import pytest

from oracle import nufft_oracle as O

pytestmark = pytest.mark.gpu

TOL = 1e-5  # rel-L2 of FP32 transforms against the FP64 oracle


def rel(a, b):
    a, b = np.asarray(a, np.complex128), np.asarray(b, np.complex128)
    return float(np.linalg.norm((a - b).ravel()) / np.linalg.norm(b.ravel()))


def _cnormal(rng, shape):
    return (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(np.complex64)


@pytest.mark.parametrize("M", [600000, 1048576, 1048677])
def test_pair_total_is_refused(M):
    """One-cell tiles and nspread 8: 4096 pairs per sample, so 2.5e9, 2^32 and 2^32 + 413,696
    pairs.  Each is refused before any pair is written, and the plan takes the next points."""
    print("case: pair total", M, flush=True)
    from mripy_amd.plan import Plan
    rng = np.random.default_rng(M)
    P = Plan((16, 16, 16), ncoils=1, rat=2, nspread=8, tiles=(1, 1, 1))
    coords = [(np.pi * (2 * rng.random(M) - 1)).astype(np.float32) for _ in range(3)]
    with pytest.raises(ValueError, match="pairs"):
        P.set_points(coords)
    few = [c[:300] for c in coords]
    P.set_points(few)
    y = _cnormal(rng, (300, 1))
    want = O.type1([c.astype(np.float64) for c in few], y.astype(np.complex128), O.Params((16, 16, 16), rat=2, nspread=8))
    assert rel(P.type1(y), want) <= TOL


@pytest.mark.parametrize("n,batch", [(2, 1 << 28), (2, (1 << 27) - 16)])
def test_cartesian_fft_of_many_columns(n, batch):
    """2 points x 2^28 columns: with 16 columns a block more blocks than a launch takes, and
    just as many.  Out of place and in place."""
    import ctypes
    import torch
    from mripy_amd import _lib
    from mripy_amd.cfft import _c2c
    print("case: many columns", n, batch, flush=True)
    x = torch.empty(n, batch, dtype=torch.complex64, device="cuda")
    torch.view_as_real(x).random_(-8, 8)
    want = torch.stack([x[0] + x[1], x[0] - x[1]])      # exact: small whole numbers
    assert torch.equal(_c2c(x, 1, _lib.GN_FFT_FORWARD), want)
    shp = (ctypes.c_int64 * 3)(n, 1, 1)
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.check(_lib.load().gn_fft_c2c(1, shp, batch, _lib.GN_FFT_FORWARD, 0, None, 1, x.data_ptr(), x.data_ptr(), st))
    assert torch.equal(x, want)


@pytest.mark.parametrize("niter", [0, 3])
def test_tv_prox_of_many_images(niter):
    """2^22 trailing elements of 2 x 2 pixels: a region each would be 2^32 threads.  The
    elements repeat 1024 different ones, whose prox is taken separately."""
    import torch
    from mripy_amd import solvers as S
    print("case: tv of many images", niter, flush=True)
    g = torch.Generator().manual_seed(1)
    few = torch.randn(2, 2, 1, 1024, generator=g, dtype=torch.complex128).cuda()
    x = few.expand(2, 2, 4096, 1024).contiguous()
    f = S.prox_tv2d_r(x, 0.3, niter=niter)
    want = S.prox_tv2d_r(few, 0.3, niter=niter) if niter else few
    assert float((f - want).abs().max()) <= 1e-12


def test_update_of_many_elements():
    """The IST update of 2^32 + 64 elements (more than a launch has threads) into buffers of
    the same size, every one of them checked by the least and the greatest."""
    import torch
    from mripy_amd import _lib
    n = (1 << 32) + 64
    if torch.cuda.mem_get_info()[0] < 4.5 * 8 * n:
        pytest.skip("needs 150 GB of free device memory")
    print("case: update of many elements", flush=True)
    import ctypes
    ones = torch.ones(2 * n, dtype=torch.float32, device="cuda")     # complex: 1 + 1i
    acc = torch.full((2 * n,), 3.0, dtype=torch.float32, device="cuda")
    x = torch.zeros(2 * n, dtype=torch.float32, device="cuda")
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.check(_lib.load().gn_soft_step(n, ones.data_ptr(), None, acc.data_ptr(), 2.0, 0.0, x.data_ptr(), None, 0.0, None, st))
    # acc = 3 - 2 * 1 in both parts everywhere, x = acc / (|acc| + 1e-6) * |acc|
    assert float(acc.amin()) == 1.0 and float(acc.amax()) == 1.0
    m = 2 ** 0.5
    assert abs(float(x.amin()) - m / (m + 1e-6)) <= 1e-6 and abs(float(x.amax()) - m / (m + 1e-6)) <= 1e-6
    del ones, acc, x
    torch.cuda.empty_cache()


def test_many_tile_columns():
    """One-cell tiles on two axes of 8192 cells: 2^26 tile columns, whose occupancy words one
    wave each would be 2^32 threads.  The points are taken, and a gather of ones gives each
    sample the sum of its window."""
    import torch
    from mripy_amd.plan import Plan
    print("case: many tile columns", flush=True)
    modes, M = (2, 4096, 4096), 64
    rng = np.random.default_rng(5)
    coords = [(np.pi * (2 * rng.random(M) - 1)).astype(np.float32) for _ in modes]
    P = Plan(modes, ncoils=1, rat=2, nspread=2, tiles=(4, 1, 1)).set_points(coords)
    G = float(np.prod(P.nf))
    got = P.grid_gather(torch.ones((1,) + P.nf, dtype=torch.complex64, device="cuda")).cpu().numpy()[:, 0] * G
    p = O.Params(modes, rat=2, nspread=2)
    want = np.ones(M)
    for c, n in zip(coords, P.nf):
        want = want * O.window_direct(c.astype(np.float64), n, 2, p.tau)[1].sum(1)
    assert rel(got, want) <= TOL


def test_spread_of_many_tiles():
    """2^24 spread tiles with 256 threads each (3 coils on 32768 x 65536 cells): the spread
    alone, cell by cell at every sample's window, and its norm (no other cell is set)."""
    import torch
    from mripy_amd.plan import Plan
    nf, nc, M, ns = (32768, 65536), 3, 40, 2
    if torch.cuda.mem_get_info()[0] < 4.5 * 8 * nc * nf[0] * nf[1]:
        pytest.skip("needs 230 GB of free device memory")
    print("case: many tiles", flush=True)
    rng = np.random.default_rng(2)
    coords = [(np.pi * (2 * rng.random(M) - 1)).astype(np.float32) for _ in nf]
    coords[0][:2], coords[1][:2] = (-1e-3, 1e-3), (-1e-3, 1e-3)       # the last tile and the first
    P = Plan(tuple(n // 2 for n in nf), ncoils=nc, rat=2, nspread=ns).set_points(coords)
    y = _cnormal(rng, (M, nc))
    out = P.grid_spread(torch.as_tensor(y).cuda())
    p = O.Params(P.modes, rat=2, nspread=ns)
    (i0, w0), (i1, w1) = [O.window_direct(c.astype(np.float64), n, ns, p.tau) for c, n in zip(coords, nf)]
    got = torch.stack([out[c][torch.as_tensor(i0[:, :, None]).cuda(), torch.as_tensor(i1[:, None, :]).cuda()]
                       for c in range(nc)], -1).cpu().numpy()
    want = (w0[:, :, None] * w1[:, None, :])[..., None] * y[:, None, None, :]
    assert rel(got, want) <= TOL
    norm = sum(float(torch.view_as_real(o).view(-1)[k::8].double().square().sum()) for o in out for k in range(8)) ** 0.5
    assert abs(norm - np.linalg.norm(want.ravel())) <= TOL * norm
    del out, P
    torch.cuda.empty_cache()
