"""The IST / FISTA update kernel rounds where the separate operations round."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 255, 256, 100003])
@pytest.mark.parametrize("step,th", [(0.5, 0.002), (0.3, 0.05), (1, 0.0), (-0.7, 1.0)])
@pytest.mark.parametrize("with_b", [True, False])
def test_update_is_the_separate_operations(n, step, th, with_b):
    import torch
    from mripy_amd import solvers as S
    print("case: update", n, step, th, with_b, flush=True)
    g = torch.Generator().manual_seed(n)
    grad, b, acc, xp = (torch.randn(n, generator=g, dtype=torch.complex64).cuda() for _ in range(4))
    b = b if with_b else None
    acc[::3] *= 1e-3
    want_acc = acc - step * (grad - b if with_b else grad)
    want_x = S.prox_l1_soft_thresh2(want_acc, th)
    for beta in (0.0, 0.281, 0.85):
        want_y = want_x + beta * (want_x - xp)
        got = S._descend(grad, b, step, acc.clone(), th, xp, beta)
        assert got[1] is not None
        for v, w in zip(got, (want_acc, want_x, want_y)):
            assert torch.equal(v, w)
