"""The two ways the TV prox runs its steps (regions of cells in LDS, several steps a launch;
two kernels a step) at shapes on either side of the choice, against the iteration in 64-bit
numpy over all trailing elements at once.  Tolerances: FP64 results 1e-10, FP32 1e-6 rel-L2
(one rounding of the result)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def tv_numpy(x, ndim, niter, step=0.1, lam=0.3, amp="reference"):
    """f = x - lam Div(G) after niter projected dual steps over the first ndim axes."""
    G = [np.zeros(x.shape, np.complex128) for _ in range(ndim)]

    def div():
        out = np.zeros(x.shape, np.complex128)
        for a, g in enumerate(G):
            g = np.moveaxis(g, a, 0)
            d = np.concatenate([-g[:1], g[:-2] - g[1:-1], g[-2:-1]])
            out += np.moveaxis(d, 0, a)
        return out
    for _ in range(niter):
        D = div() - x / lam
        for a in range(ndim):
            last = np.take(D, [-1], axis=a)
            G[a] = G[a] - step * np.diff(D, axis=a, append=last)
        if amp == "reference":
            n = np.maximum(np.sqrt(sum(g * g for g in G)), 1 + 0j)
        else:
            n = np.maximum(np.sqrt(sum(np.abs(g) ** 2 for g in G)), 1)
        G = [g / n for g in G]
    return x - lam * div()


def rel(a, b):
    return float(np.linalg.norm((np.asarray(a, np.complex128) - b).ravel()) / np.linalg.norm(b.ravel()))


@pytest.mark.parametrize("shape,ndim", [((3, 3, 1100), 2), ((2, 40000), 2), ((40000, 2), 2), ((40, 40, 260), 2),
                                        ((24, 3, 700), 2), ((4, 4, 4, 130), 3), ((2, 2, 600, 3), 3), ((60, 61, 2), 3),
                                        ((17, 80, 80), 3), ((2, 3, 5), 3)])
@pytest.mark.parametrize("niter", [0, 1, 2, 8])
def test_tv_shapes(shape, ndim, niter):
    import torch
    from mripy_amd import solvers as S
    print("case: tv shape", shape, ndim, niter, flush=True)
    rng = np.random.default_rng(niter + sum(shape))
    x = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    prox = S.prox_tv2d_r if ndim == 2 else S.prox_tv3d
    for amp in ("reference", "modulus"):
        want = tv_numpy(x, ndim, niter, amp=amp)
        assert rel(prox(torch.as_tensor(x).cuda(), 0.3, niter=niter, amp=amp).cpu(), want) <= 1e-10
        got = prox(torch.as_tensor(x.astype(np.complex64)).cuda(), 0.3, niter=niter, amp=amp)
        assert got.dtype == torch.complex64
        assert rel(got.cpu(), tv_numpy(x.astype(np.complex64).astype(complex), ndim, niter, amp=amp)) <= 1e-6


@pytest.mark.parametrize("shape,ndim", [((12, 9), 2), ((40000, 2), 2), ((7, 6, 5), 3), ((60, 61, 2), 3)])
@pytest.mark.parametrize("step", [1e74, 1e75, 1e76, 1e80, 1e140])
def test_tv_projection_of_large_fields(shape, ndim, step):
    """Dual fields before, at and beyond the range of the squared square, from images of order
    1 and a large step: the projected field is of order 1 and so are its errors."""
    import torch
    from mripy_amd import solvers as S
    print("case: tv projection", shape, ndim, step, flush=True)
    rng = np.random.default_rng(sum(shape))
    x = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    want = tv_numpy(x, ndim, 1, step=step)
    prox = S.prox_tv2d_r if ndim == 2 else S.prox_tv3d
    got = prox(torch.as_tensor(x).cuda(), 0.3, step=step, niter=1).cpu().numpy()
    assert np.isfinite(want).all() and rel(want, x) > 0.1 and rel(got, want) <= 1e-10
