"""When projections are torch's own whatever their sizes: what is asked in front of every call, without a GPU."""
import torch

from based_amd import linear


def test_mapped_weights_are_seen():
    """Under torch.vmap the weight or the bias may be mapped and x not."""
    seen = []

    def f(w):
        seen.append(linear._watched())
        return w.sum()

    torch.vmap(f)(torch.ones(2, 3))
    with torch.no_grad():
        torch.vmap(f)(torch.ones(2, 3))
        assert seen == [True, True] and not linear._watched()
