"""Which IST / FISTA updates may take the one-kernel path (no GPU needed for the checks)."""
import pytest
import torch

from mripy_amd import solvers as S


@pytest.mark.parametrize("owner,name", [(torch._C, "_len_torch_dispatch_stack"), (torch._C, "_len_torch_function_stack"),
                                        (torch._C, "_functorch"), (torch.autograd.forward_ad, "_current_level")])
def test_missing_torch_query_means_separate_operations(monkeypatch, owner, name):
    """A torch without one of the private queries takes the separate operations, not an error."""
    t = torch.zeros(3, dtype=torch.complex64)
    assert not S._watched()
    monkeypatch.delattr(owner, name)
    assert S._watched() and S._plain(t, t) is False
    acc, x, y = S._descend(t + 1, None, 0.5, t, 0.1)
    assert x is None and y is None and torch.equal(acc, t - 0.5)


def test_watched_by_transforms():
    seen = []

    def f(v):
        seen.append(S._watched())
        return v * 2
    torch.func.vmap(f)(torch.ones(2))
    torch.func.jvp(f, (torch.ones(2),), (torch.ones(2),))
    with torch.autograd.forward_ad.dual_level():
        f(torch.ones(2))
    assert seen == [True, True, True] and not S._watched()
