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
