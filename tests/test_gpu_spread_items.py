"""Spread work items of every length the rule gives: samples spread evenly (items longer than
a tile's pairs, none split) and in a cluster (split tiles), coil counts of each spread kernel,
few and many reduced tiles, a batch: type 1 against the FP64 oracle, rel-L2 <= 1e-5 (the
repository's bound)."""
import numpy as np
import pytest

from oracle import nufft_oracle as O

pytestmark = pytest.mark.gpu


def rel(a, b):
    a, b = np.asarray(a, np.complex128), np.asarray(b, np.complex128)
    return float(np.linalg.norm((a - b).ravel()) / np.linalg.norm(b.ravel()))


@pytest.mark.parametrize("modes,M", [((12, 12, 16), 1000), ((16, 16, 16), 9000), ((16, 16, 20), 22000), ((64, 64), 6000),
                                     ((100, 96), 30000)])
@pytest.mark.parametrize("nc", [1, 4, 8, 17])
@pytest.mark.parametrize("even", [True, False])
def test_spread_items(modes, M, nc, even):
    import torch
    from mripy_amd.batch import BatchPlan
    from mripy_amd.plan import Plan
    print("case: items", modes, M, nc, even, flush=True)
    rng = np.random.default_rng(M + nc)
    coords = [(np.pi * (2 * rng.random(M) - 1) if even else np.where(rng.random(M) < 0.7, 0.05 * rng.standard_normal(M),
               np.pi * (2 * rng.random(M) - 1))).astype(np.float32) for _ in modes]
    y = (rng.standard_normal((M, nc)) + 1j * rng.standard_normal((M, nc))).astype(np.complex64)
    P = Plan(modes, ncoils=nc, rat=2, nspread=3).set_points(coords)
    want = O.type1([c.astype(np.float64) for c in coords], y.astype(np.complex128), O.Params(modes, rat=2, nspread=3))
    got = P.type1(y)
    assert rel(got, want) <= 1e-5
    B = BatchPlan([dict(modes=modes, coords=coords, ncoils=nc)] * 3)
    yt = torch.as_tensor(y).cuda()
    assert all(rel(o.cpu(), got) <= 1e-6 for o in B.type1([yt] * 3))
