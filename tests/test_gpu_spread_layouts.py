"""Type 1 of coil-major samples, whose coils are spread in other groups and kernels, against
coil-last samples: 2-D in groups of 8 instead of 16, 3-D by k_spread_mfma from 4 coils on.
Tolerance: rel-L2 1e-6, two FP32 sums in different order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nc", [3, 8, 9, 16, 17, 31])
@pytest.mark.parametrize("ns,M", [(3, 37), (3, 9000), (8, 5000)])
def test_layouts_agree(nc, ns, M):
    import torch
    from mripy_amd.plan import Plan
    print("case: layouts", nc, ns, M, flush=True)
    g = torch.Generator().manual_seed(nc + M)
    c = [((2 * torch.rand(M, generator=g) - 1) * np.pi).cuda() for _ in range(2)]
    y = torch.randn(M, nc, generator=g, dtype=torch.complex64).cuda()
    a, b = (Plan((30, 41), ncoils=nc, rat=2, nspread=ns, layout=lay).set_points(c) for lay in ("coil_last", "coil_major"))
    want, got = a.type1(y), b.type1(y.t().contiguous()).permute(1, 2, 0)
    assert float((got - want).norm() / want.norm()) <= 1e-6


@pytest.mark.parametrize("nc", [1, 3, 4, 5])
@pytest.mark.parametrize("ns,M", [(3, 37), (3, 9000), (5, 2000)])
def test_layouts_agree_3d(nc, ns, M):
    import torch
    from mripy_amd.plan import Plan
    print("case: layouts 3-D", nc, ns, M, flush=True)
    g = torch.Generator().manual_seed(nc + M)
    c = [((2 * torch.rand(M, generator=g) - 1) * np.pi).cuda() for _ in range(3)]
    y = torch.randn(M, nc, generator=g, dtype=torch.complex64).cuda()
    a, b = (Plan((12, 15, 18), ncoils=nc, rat=2, nspread=ns, layout=lay).set_points(c) for lay in ("coil_last", "coil_major"))
    want, got = a.type1(y), b.type1(y.t().contiguous()).permute(1, 2, 3, 0)
    assert float((got - want).norm() / want.norm()) <= 1e-6
