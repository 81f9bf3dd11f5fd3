"""The projections of short prompts against torch in 64 bits: rows, features and channels around whole tiles, with bias and with the gate, rows
of wider matrices; which calls take them; and the modules, watched and unwatched."""
import pytest
import torch

from conftest import rel_l2

pytestmark = pytest.mark.gpu


def make(dev, M, N, K, bias, seed=0, wide=0):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(M, K, generator=g).bfloat16().to(dev)
    w = (torch.randn(N, K + wide, generator=g) * K ** -0.5).bfloat16().to(dev)[:, :K]
    return x, w, torch.randn(N, generator=g).bfloat16().to(dev) if bias else None


def reference(x, w, b):
    y = x.double() @ w.double().T
    return y if b is None else y + b.double()


@pytest.mark.parametrize("K", [128, 384, 1024, 2048])
@pytest.mark.parametrize("M,N,bias", [(1, 4, False), (17, 256, True), (63, 1000, False), (64, 1024, True), (65, 4100, True), (129, 68, False),
                                      (300, 3072, True), (512, 4096, False), (512, 1024, True), (1000, 512, False), (640, 4096, True)])
def test_projection(dev, M, N, K, bias):
    from based_amd import ops

    x, w, b = make(dev, M, N, K, bias, wide=8 * (M % 2))
    ref = reference(x, w, b)
    y = ops.prompt_linear(x, w, b)
    # fp32 sums rounded once: 2^-9 of a value at most, a third of that in the mean
    assert (y.double() - ref).abs().max() <= ref.abs().max() * 2 ** -8 and rel_l2(y, ref) < 2.5e-3


@pytest.mark.parametrize("M,F,K,bias", [(9, 8, 128, True), (64, 1024, 1024, False), (70, 520, 256, True), (300, 2048, 1024, False), (512, 2048, 1024, True),
                                        (513, 40, 2048, False)])
def test_gate_behind_a_projection(dev, M, F, K, bias):
    """As the projection and the gate kernel one after the other; a product that rounds to the other side of a step moves an element by 2^-7 of it."""
    from based_amd import ops

    x, w, b = make(dev, M, 2 * F, K, bias)
    y, two = ops.prompt_linear(x, w, b, gated=True), ops.swiglu(ops.prompt_linear(x, w, b))
    p = reference(x, w, b)
    ref = p[:, :F] * torch.nn.functional.silu(p[:, F:])
    assert torch.equal(y, two) and rel_l2(y, ref) < 6e-3


@pytest.mark.parametrize("M,N,K,form", [(4, 50280, 1024, 2), (8, 50280, 1024, 0), (8, 1024, 4096, 2), (9, 1024, 1024, 1), (512, 4096, 1024, 1), (513, 64, 1024, 0),
                                        (512, 4160, 1024, 0), (64, 1024, 1000, 0), (64, 1024, 2176, 0), (64, 1022, 1024, 0)])
def test_which_calls_take_them(dev, M, N, K, form):
    from based_amd import ops

    x, w, b = make(dev, M, N, K, N % 8 == 0)
    assert ops.linear_form(x, w, b) == form
    assert ops.linear_form(x.float(), w.float()) == 0 and ops.linear_form(x, w.t().contiguous().t()) == 0
    if M > 8:
        assert ops.linear_form(torch.cat([x, x], 1)[:, :K], w) == 0
    shifted = torch.empty(M * K + 1, dtype=torch.bfloat16, device=dev)[1:].view(M, K).copy_(x)  # (no whole 16-byte pieces)
    assert ops.linear_form(shifted, w, b) == 0
    assert rel_l2(ops.linear(shifted, w, b), reference(x, w, b)) < 2.5e-3
    assert rel_l2(ops.linear(x.view(1, M, K), w, b)[0], reference(x, w, b)) < 2.5e-3


@pytest.mark.parametrize("M", [4, 40])
def test_no_features(dev, M):
    from based_amd.linear import Linear

    with torch.no_grad():
        assert Linear(256, 0, device=dev, dtype=torch.bfloat16)(torch.randn(M, 256, device=dev).bfloat16()).shape == (M, 0)


def test_gates_in_whole_eights(dev):
    """Any number of rows: others are refused, as by the gate's kernel."""
    from based_amd.stack import GatedMlp

    with torch.no_grad():
        for hidden in (16, 20):
            mlp = GatedMlp(256, hidden_features=hidden, multiple_of=4, device=dev, dtype=torch.bfloat16)
            for rows in (4, 40, 600):
                x = torch.randn(1, rows, 256, device=dev).bfloat16()
                if hidden == 16:
                    assert mlp(x).shape == x.shape
                else:
                    with pytest.raises((ValueError, RuntimeError), match="width must be a multiple of 8"):
                        mlp(x)


def test_modules_that_are_watched(dev):
    """Gradients, hooks and modes see torch's own operations; the last tokens of a prompt are rows of a wider tensor."""
    from based_amd import ops
    from based_amd.linear import Linear
    from based_amd.stack import GatedMlp

    torch.manual_seed(0)
    mlp = GatedMlp(256, hidden_features=512, device=dev, dtype=torch.bfloat16)
    x = torch.randn(2, 40, 256, device=dev).bfloat16()
    with torch.no_grad():
        plain = mlp(x)
        seen = []
        handle = mlp.fc1.register_forward_hook(lambda m, a, y: seen.append(y))
        assert rel_l2(mlp(x), plain) < 1e-2 and seen[0].shape == (2, 40, 1024)
        handle.remove()
        with torch.autocast("cuda", dtype=torch.float16):
            assert mlp.fc1(x).dtype == torch.float16
        assert rel_l2(torch.vmap(mlp.fc1)(x), mlp.fc1(x)) < 1e-2
        with torch.autograd.forward_ad.dual_level():
            dual = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
            assert torch.autograd.forward_ad.unpack_dual(mlp.fc1(dual)).tangent is not None
        head = Linear(256, 1000, bias=False, device=dev, dtype=torch.bfloat16)
        last = x[:, -1:]
        assert ops.linear_form(last, head.weight) == ops.LINEAR_ROWS
        assert rel_l2(head(last), reference(last.reshape(2, 256), head.weight.detach(), None).view(2, 1, -1)) < 2.5e-3
    y = mlp.fc1(x)
    y.float().square().sum().backward()
    assert mlp.fc1.weight.grad is not None


@pytest.mark.parametrize("M", [4, 40])
def test_stacked_weights(dev, M):
    """An ensemble: torch.vmap over weights, over biases and over both, the rows the same for all; each as the library takes it alone."""
    from torch.func import functional_call

    from based_amd.linear import Linear

    torch.manual_seed(1)
    fc = Linear(256, 1024, device=dev, dtype=torch.bfloat16)
    x = torch.randn(2, M // 2, 256, device=dev).bfloat16()
    stacked = {"weight": torch.randn(3, 1024, 256, device=dev).mul(1 / 16).bfloat16(), "bias": torch.randn(3, 1024, device=dev).bfloat16()}
    with torch.no_grad():
        for names in (("weight",), ("bias",), ("weight", "bias")):
            mapped = {n: stacked[n] for n in names}
            got = torch.vmap(lambda p: functional_call(fc, p, (x,)))(mapped)
            for i in range(3):
                w, b = (mapped[n][i] if n in mapped else getattr(fc, n).detach() for n in ("weight", "bias"))
                assert rel_l2(got[i], reference(x.view(M, 256), w, b).view_as(got[i])) < 2.5e-3


def test_tensors_without_rows_of_their_own(dev):
    """A sparse weight, a nested batch and a bias of another class are torch's own."""
    from based_amd.linear import linear

    class Marked(torch.Tensor):
        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            seen.append(func)
            return super().__torch_function__(func, types, args, kwargs or {})

    x, w, b = make(dev, 40, 256, 128, True)
    plain = torch.nn.functional.linear(x, w, b)
    with torch.no_grad():
        few = w * (torch.arange(128, device=dev) % 16 == 0)
        sparse = few.float().to_sparse_csr()
        assert rel_l2(linear(x.float(), sparse), x.float() @ few.float().T) < 1e-5
        nested = torch.nested.nested_tensor([x[:12], x[12:]])
        assert torch.equal(torch.cat(list(linear(nested, w, b).unbind())), plain)
        seen = []
        assert rel_l2(linear(x, w, b.as_subclass(Marked)).as_subclass(torch.Tensor), plain) < 1e-2 and seen


@pytest.mark.parametrize("dtype,rows,width,hidden,looked_up", [
    (torch.bfloat16, 512, 256, 512, True), (torch.bfloat16, 513, 256, 512, False), (torch.float32, 40, 256, 512, False), (torch.bfloat16, 8, 200, 200, True),
    (torch.bfloat16, 9, 200, 200, False), (torch.bfloat16, 9, 2176, 128, True), (torch.bfloat16, 9, 2176, 2176, False)])
def test_what_is_not_looked_at(dev, monkeypatch, dtype, rows, width, hidden, looked_up):
    """More rows than either kernel takes, other types and channels: nothing but the library's call, of the projections and of the gate's."""
    from based_amd import ops
    from based_amd.stack import GatedMlp

    mlp = GatedMlp(width, hidden_features=hidden, multiple_of=8, device=dev, dtype=dtype)
    seen, form = [], ops.linear_form
    monkeypatch.setattr(ops, "linear_form", lambda *a: seen.append(1) or form(*a))
    with torch.no_grad():
        assert mlp(torch.randn(1, rows, width, device=dev).to(dtype)).shape == (1, rows, width)
    assert bool(seen) == looked_up


def test_module_with_a_forward_of_its_own(dev):
    """A wrapper that replaces the projection's forward (to move weights, to add a term) is called in front of the gate, too."""
    from based_amd.stack import GatedMlp

    mlp = GatedMlp(256, hidden_features=512, device=dev, dtype=torch.bfloat16)
    x = torch.randn(2, 40, 256, device=dev).bfloat16()
    inner = mlp.fc1.forward
    with torch.no_grad():
        plain = mlp(x)
        mlp.fc1.forward = lambda x: inner(x) * 0
        assert not mlp(x).any()
        del mlp.fc1.forward
        assert torch.equal(mlp(x), plain)


@torch.inference_mode()
def test_in_a_recorded_graph(dev):
    """Recorded in the mode the models record in."""
    from based_amd import ops

    x, w, b = make(dev, 200, 1024, 512, True)
    want = ops.prompt_linear(x, w, b)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            y = ops.prompt_linear(x, w, b)
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
