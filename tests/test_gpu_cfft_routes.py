"""The Cartesian FFT where the choice of its passes changes, against numpy in 64 bits:
short lines by the hundred in a block, long strided axes.  Tolerance: rel-L2 2e-6."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def check(shape, rank):
    import torch
    from mripy_amd import _lib
    from mripy_amd.cfft import _c2c
    print("case: c2c", shape, rank, flush=True)
    rng = np.random.default_rng(sum(shape))
    x = (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(np.complex64)
    ax = tuple(range(rank))
    mask = rng.random(shape[:rank]).astype(np.float32)
    flags = _lib.GN_FFT_SHIFT_IN | _lib.GN_FFT_SHIFT_OUT
    xs = np.fft.fftshift(x.astype(np.complex128), ax)
    fwd = np.fft.ifftshift(np.fft.fftn(xs, axes=ax), ax) * mask.reshape(mask.shape + (1,) * (len(shape) - rank))
    inv = np.fft.ifftshift(np.fft.ifftn(xs, axes=ax), ax)
    t = torch.as_tensor(x).cuda()
    for got, want in ((_c2c(t, rank, _lib.GN_FFT_FORWARD, flags, torch.as_tensor(mask).cuda()), fwd),
                      (_c2c(t, rank, _lib.GN_FFT_INVERSE, flags), inv)):
        assert np.linalg.norm((got.cpu().numpy() - want).ravel()) <= 2e-6 * np.linalg.norm(want.ravel())


# a block holds 2048 elements of lines of up to 64 points: columns of one slab, the whole of
# several slabs, one column short of and past a block, odd counts, enough for 512 blocks
@pytest.mark.parametrize("shape,rank", [((2, 1025), 1), ((3, 70001), 1), ((64, 33), 1), ((65, 33), 1), ((700, 3), 2),
                                        ((600, 5, 3), 2), ((90, 2, 90, 3), 3), ((2, 90, 91), 3), ((400, 90, 2), 3),
                                        ((17, 4001), 1), ((300, 34), 2), ((13, 600, 8), 2)])
def test_short_lines(shape, rank):
    check(shape, rank)


# strided axes on both sides of the lengths left to rocFFT (1860; 1100 with the prime 17), the
# same lengths contiguous, and one of each in a call
@pytest.mark.parametrize("shape,rank", [((1848, 3), 1), ((1875, 3), 1), ((5, 1875), 2), ((1088, 2), 1), ((1156, 2), 1),
                                        ((3, 1156), 2), ((1904, 4, 2), 2), ((4, 2000, 3), 2), ((1862, 1), 2)])
def test_long_axes(shape, rank):
    check(shape, rank)
