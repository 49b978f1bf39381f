"""The trajectory gradient with coil pairs and with single coils in its LDS cells, at window
widths and coil counts on either side of the choice, against the FP64 oracle.  Tolerance:
rel-L2 <= 1e-5, the repository's bound for FP32 results."""
import numpy as np
import pytest

from oracle import nufft_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("modes,ns,nc", [((20, 22, 24), 3, 2), ((20, 22, 24), 4, 2), ((16, 17, 18), 5, 5), ((16, 17, 18), 6, 3),
                                         ((8, 9, 8), 8, 2), ((40, 44), 5, 3), ((40, 44), 7, 3), ((40, 44), 8, 3),
                                         ((40, 44), 8, 5), ((40, 41), 16, 2), ((40, 44), 2, 1)])
@pytest.mark.parametrize("layout", ["coil_last", "coil_major"])
def test_traj_grad_cells(modes, ns, nc, layout):
    import torch
    from mripy_amd.plan import Plan
    print("case: trajectory gradient", modes, ns, nc, layout, flush=True)
    rng = np.random.default_rng(ns + nc)
    M = 900
    coords = [np.concatenate([0.02 * rng.standard_normal(600) + 0.4, np.pi * (2 * rng.random(300) - 1)]).astype(np.float32)
              for _ in modes]
    F, w = [(rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64) for s in (modes + (nc,), (M, nc))]
    dev = (lambda a: torch.as_tensor(a if layout == "coil_last" else np.ascontiguousarray(np.moveaxis(a, -1, 0))).cuda())
    P = Plan(modes, ncoils=nc, rat=2, nspread=ns, layout=layout).set_points(coords)
    got = P.traj_grad(dev(F), dev(w)).cpu().numpy()
    want = O.traj_grad([c.astype(np.float64) for c in coords], F, w, O.Params(modes, rat=2, nspread=ns))
    assert np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want)
