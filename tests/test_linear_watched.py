"""When projections are torch's own whatever their sizes: what is asked in front of every call, without a GPU."""
import torch

from based_amd import linear


def watched():
    few = torch.ones(1, 8, dtype=torch.bfloat16)
    return linear._beyond(few, few) or linear._watched()


def test_mapped_weights_are_seen():
    """Under torch.vmap the weight or the bias may be mapped and x not."""
    seen = []

    def f(w):
        seen.append(watched())
        return w.sum()

    torch.vmap(f)(torch.ones(2, 3))
    with torch.no_grad():
        torch.vmap(f)(torch.ones(2, 3))
        assert seen == [True, True] and not watched()


def test_modes_and_tracing_are_seen():
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    class Seen(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class SeenToo(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with torch.no_grad():
        assert not watched()
        for mode in (Seen(), SeenToo(), torch.enable_grad(), torch.autograd.forward_ad.dual_level()):
            with mode:
                assert watched()
        traced = []
        torch.jit.trace(lambda x: traced.append(watched()) or x + 1, torch.ones(2), check_trace=False)
        assert traced == [True] and not watched()


def test_a_torch_that_cannot_be_asked(monkeypatch):
    """A build without one of the private names: everything is torch's own."""
    from types import SimpleNamespace

    whole = linear._questions()
    assert whole is not None
    names = {"_functorch": SimpleNamespace(peek_interpreter_stack=1), "_len_torch_dispatch_stack": 1, "_len_torch_function_stack": 1}
    ad = SimpleNamespace(_current_level=-1)
    assert linear._questions(SimpleNamespace(**names), ad) == (1, 1, 1)
    for gone in names:
        assert linear._questions(SimpleNamespace(**{n: v for n, v in names.items() if n != gone}), ad) is None
    assert linear._questions(SimpleNamespace(**{**names, "_functorch": SimpleNamespace()}), ad) is None
    assert linear._questions(SimpleNamespace(**names), SimpleNamespace()) is None
    with torch.no_grad():
        assert not watched()
        monkeypatch.setattr(linear, "_QUESTIONS", None)
        assert watched()
        x, w = torch.randn(3, 8), torch.randn(4, 8)
        assert torch.equal(linear.linear(x, w), torch.nn.functional.linear(x, w))


def test_scripted_exported_and_traced():
    """A projection by itself goes where torch.nn.Linear goes."""
    fc, x = linear.Linear(8, 4), torch.randn(3, 8)
    want = fc(x)
    for other in (torch.jit.script(fc), torch.jit.trace(fc, x), torch.export.export(fc, (x,)).module(), torch.compile(fc, backend="eager", fullgraph=True)):
        assert torch.equal(other(x), want)
        with torch.no_grad():
            assert torch.equal(other(x), want)


def test_parameters_that_something_stands_in_for():
    """Pruned, parametrised and replaced weights, by whatever way torch.nn.Linear finds them."""
    from torch.func import functional_call
    from torch.nn.utils import parametrize, prune

    x = torch.randn(3, 8)
    fc = linear.Linear(8, 4)
    prune.random_unstructured(fc, "weight", 0.5)
    assert torch.equal(fc(x), torch.nn.functional.linear(x, fc.weight, fc.bias)) and (fc.weight == 0).any()
    fc = linear.Linear(8, 4, bias=False)
    parametrize.register_parametrization(fc, "weight", torch.nn.ReLU())
    assert torch.equal(fc(x), x @ fc.weight.T) and (fc.weight >= 0).all()
    fc, other = linear.Linear(8, 4), torch.randn(4, 8)
    assert torch.equal(functional_call(fc, {"weight": other}, (x,)), torch.nn.functional.linear(x, other, fc.bias))
    fc.weight.data = other
    assert torch.equal(fc(x), torch.nn.functional.linear(x, other, fc.bias))
