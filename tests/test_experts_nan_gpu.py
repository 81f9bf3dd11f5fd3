"""Tokens and routers that are no numbers: every choice names an expert that there is, and only these tokens' outputs are no numbers."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def make(n, E, D, F, dtype, dev):
    g = torch.Generator().manual_seed(n + E)
    rnd = lambda *s, std=1.0: (std * torch.randn(*s, generator=g)).to(dtype).to(dev)  # noqa: E731
    return rnd(n, D), rnd(E, D, std=D ** -0.5), rnd(E, 2 * F, D, std=D ** -0.5), rnd(E, D, F, std=F ** -0.5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,E,top", [(1, 8, 2), (1, 2, 2), (3, 5, 5), (7, 64, 2), (4, 70, 4), (2, 200, 3), (16, 3, 1), (20, 8, 2), (30, 40, 3),
                                     (150, 8, 1), (600, 4, 2)])
def test_tokens_that_are_no_numbers(dev, n, E, top, dtype):
    from based_amd import ops

    h, router, w1, w2 = make(n, E, 64, 32, dtype, dev)
    clean = ops.experts(h, router, w1, w2, top)
    bad = h.clone()
    bad[n // 2, 5] = float("nan")
    y = ops.experts(bad, router, w1, w2, top)
    assert y[n // 2].isnan().all()
    rest = torch.arange(n, device=dev) != n // 2
    assert torch.equal(y[rest], clean[rest])  # (a row's sums do not depend on its place)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [1, 5, 20, 100])
def test_routers_that_are_no_numbers(dev, n, dtype):
    """An expert without a score is chosen by nobody while there are others, and a token left without a choice is no number."""
    from based_amd import ops

    h, router, w1, w2 = make(n, 6, 64, 32, dtype, dev)
    broken = router.clone()
    broken[2] = float("nan")
    others = [0, 1, 3, 4, 5]
    y, want = ops.experts(h, broken, w1, w2, 2), ops.experts(h, router[others].contiguous(), w1[others].contiguous(), w2[others].contiguous(), 2)
    assert ((y.double() - want.double()).norm() / want.double().norm()) < (1e-6 if dtype == torch.float32 else 1e-2)
    assert ops.experts(h, broken, w1, w2, 6).isnan().all()


def test_norm_in_front(dev):
    from based_amd import ops

    h, router, w1, w2 = make(3, 8, 64, 32, torch.bfloat16, dev)
    weight, res = torch.ones(64, dtype=torch.bfloat16, device=dev), torch.randn(3, 64, device=dev)
    clean = ops.experts(h, router, w1, w2, 2, norm=(res, torch.empty_like(res), weight, 1e-5, ops.NORM_RMS, 1.0))
    h[1, 9] = float("nan")
    y = ops.experts(h, router, w1, w2, 2, norm=(res, torch.empty_like(res), weight, 1e-5, ops.NORM_RMS, 1.0))
    assert y[1].isnan().all() and torch.equal(y[::2], clean[::2])
