"""Plans on either side of the choice between the pruned FFT passes and rocFFT, for grid
lengths with primes above 5: both directions and SENSE against the same plan with rocFFT.
Tolerance: rel-L2 2e-6, the two engines' FP32 errors (below 5e-7 each)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float((a - b).norm() / b.norm())


@pytest.mark.parametrize("modes,nc", [((385, 40), 2), ((392, 40), 2), ((422, 422), 2), ((446, 30), 3), ((458, 30), 3),
                                      ((519, 20), 2), ((917, 20), 2), ((956, 20), 2), ((477, 955), 1), ((228, 455), 1),
                                      ((110, 16, 16), 4), ((110, 16, 16), 5), ((251, 16, 16), 1), ((265, 16, 16), 1),
                                      ((471, 16, 16), 2), ((55, 55, 110), 1)])
def test_engines_agree(modes, nc):
    import torch
    from mripy_amd.batch import BatchPlan
    from mripy_amd.plan import Plan
    print("case: engines", modes, nc, flush=True)
    g = torch.Generator().manual_seed(sum(modes) + nc)
    M = 700
    coords = [((2 * torch.rand(M, generator=g) - 1) * np.pi).cuda() for _ in modes]
    F, y, x = [torch.randn(*s, generator=g, dtype=torch.complex64).cuda() for s in (modes + (nc,), (M, nc), modes)]
    P = Plan(modes, ncoils=nc, rat=2, nspread=3).set_points(coords)
    P.set_sense(F)

    def run():
        return [P.type2(F), P.type1(y), P.sense_type2(x), P.sense_type1(y), P.sense_type21(x)]
    auto = run()
    P.set_fft_engine("rocfft")
    for a, b in zip(auto, run()):
        assert rel(a, b) <= 2e-6
    B = BatchPlan([dict(modes=modes, coords=coords, ncoils=nc)])
    assert rel(B.type2([F])[0], auto[0]) <= 2e-6 and rel(B.type1([y])[0], auto[1]) <= 2e-6


def test_sense_combine_is_captured():
    """The first SENSE adjoint of a plan whose coils do not fit one row-pass block (two line
    buffers of 502 points x 24 coils) inside a graph: nothing is allocated, and every replay
    equals the eager result."""
    import torch
    from mripy_amd.plan import Plan
    print("case: captured combine", flush=True)
    modes, nc, M = (251, 251), 24, 300
    g = torch.Generator().manual_seed(1)
    coords = [((2 * torch.rand(M, generator=g) - 1) * np.pi).cuda() for _ in modes]
    F, y = [torch.randn(*s, generator=g, dtype=torch.complex64).cuda() for s in (modes + (nc,), (M, nc))]
    P = Plan(modes, ncoils=nc, rat=2, nspread=3).set_points(coords)
    P.set_sense(F)
    P.type1(y)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        x = P.sense_type1(y)
    want = P.sense_type1(y).clone()
    for k in range(3):
        x.zero_()
        y.mul_(2)
        graph.replay()
        torch.cuda.synchronize()
        want = want * 2
        assert torch.equal(x, want)
