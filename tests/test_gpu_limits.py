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
