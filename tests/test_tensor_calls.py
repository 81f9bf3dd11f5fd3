"""csrc/tensors.cpp against what it stands for: keys of tensors' forms, and memory beside a tensor."""
import itertools
import os

import pytest
import torch

from based_amd import _lib, ops


def _tensors():
    a = torch.zeros(3, 6, 8)
    yield from (None, a, a.transpose(0, 1), a[:, :, ::2], a[..., :7], a.bfloat16(), torch.zeros(3, 6, 8, device="meta"), torch.zeros(3, 48), torch.zeros(144),
                torch.zeros(()), torch.zeros(0, 6, 8), a[:1], a[1:2].expand(3, 6, 8), torch.zeros(3, 6, 8, dtype=torch.int32))


built = pytest.mark.skipif(ops._form is ops._form_of, reason="tensors are asked from Python here")


def test_is_built(tmp_path):
    if ops._form is ops._form_of:  # (as it may be without a compiler or the headers)
        from based_amd import build

        assert not build._build_tensors(str(tmp_path / "t.so")), "tensors are asked from Python: python -m based_amd.build"
    else:
        assert os.path.exists(_lib.TENSORS_PATH)


def test_same_key_for_the_same_form_only():
    ts = list(_tensors())
    for x, y in itertools.product(ts, repeat=2):
        assert (ops._form(x) == ops._form(y)) == (ops._form_of(x) == ops._form_of(y)), (x, y)
    groups = [p for n in (0, 1, 2, 3) for p in itertools.product(ts[:6], repeat=n)]
    for x, y in itertools.product(groups, repeat=2):
        assert (ops._form(*x) == ops._form(*y)) == (ops._form_of(*x) == ops._form_of(*y))
    assert ops._form(torch.nn.Parameter(ts[1])) == ops._form(torch.zeros(3, 6, 8)) and isinstance(ops._form(*ts), tuple if ops._form is ops._form_of else bytes)


def test_other_tensors_are_left_to_python():
    class Own(torch.Tensor):
        pass

    a = torch.zeros(3, 6, 8)
    assert ops._form(a, a.as_subclass(Own)) == ops._form_of(a, a)
    assert torch.func.vmap(lambda x: x + isinstance(ops._form(x), tuple))(a).eq(1).all()
    sparse = a.to_sparse()
    assert ops._form(sparse) == ops._form_of(sparse)
    with pytest.raises(AttributeError):
        ops._form(3)
    many = [torch.zeros([1] * 40)] * 5
    assert ops._form(*many) == ops._form_of(*many)
    from torch._subclasses.fake_tensor import FakeTensorMode

    with FakeTensorMode() as mode:
        fake = mode.from_tensor(a)
        assert ops._form(fake) == ops._form_of(fake) and type(ops._empty(a, torch.float32, 2)) is type(fake)


def test_memory_beside_a_tensor():
    a = torch.zeros(3, 6, dtype=torch.bfloat16)
    for like, sizes in ((a, (2, 3, 4)), (a, (0, 5)), (a, ()), (a.to("meta"), (7,)), (torch.nn.Parameter(a.float()), (2, 1)), (a, (1,) * 12)):
        for dtype in (torch.float32, torch.bfloat16, torch.uint8):
            x, y = ops._empty(like, dtype, *sizes), ops._empty_of(like, dtype, *sizes)
            assert (x.shape, x.stride(), x.dtype, x.device, x.requires_grad) == (y.shape, y.stride(), y.dtype, y.device, False)
    with torch.inference_mode():
        assert ops._empty(a, torch.float32, 2).is_inference()
    for bad in ((-1,), (1 << 70,), ("2",), (1 << 61,), (True, 2)):
        with pytest.raises((RuntimeError, TypeError, OverflowError)):
            ops._empty(a, torch.float32, *bad)


@built
def test_a_library_of_another_torch_is_left_alone(monkeypatch):
    monkeypatch.setattr(torch, "__version__", "0.0.1+x")
    with pytest.warns(UserWarning, match="built against torch"):
        assert _lib.tensor_calls(1, 2) == (1, 2)
    monkeypatch.setattr(_lib, "TENSORS_PATH", os.devnull + "-none")
    assert _lib.tensor_calls(1, 2) == (1, 2)
