"""The fp32 form of the Taylor linear attention prefill against the definition in 64 bits: lengths around the 16-token tiles and
64-token chunks, head dims around the 16-channel tiles, sequences in one piece and in segments, layouts of every alignment, and values
that are no numbers."""
import pytest
import torch

from conftest import rel_l2
from oracle import based_oracle as O

pytestmark = pytest.mark.gpu
# Products and sums are fp32 (2^-24 = 6e-8 each).  A token's denominator and the terms of its output are positive and signed sums of
# some thousand of them in blocks of 64, errors of random signs: below 32 roundings in the 2-norm.
TOL = 2e-6


def make(seed, B, H, L, dv, dtype=torch.float32):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(B, H, L, n, generator=g).to(dtype) for n in (16, 16, dv)]


def check(dev, q, k, v, tol=TOL, split=None):
    from based_amd import ops

    ref = O.linear_attn_quadratic(q.double(), k.double(), v.double())
    kv_ref, ks_ref = O.linear_attn_prefill_state(k.double(), v.double())
    y, kv, ks = ops.linear_attn_prefill(q.to(dev), k.to(dev), v.to(dev), return_state=True, split=split)
    assert rel_l2(y, ref) < tol and rel_l2(kv, kv_ref) < TOL and rel_l2(ks, ks_ref) < TOL
    assert bool((ks[..., 0] == q.shape[2]).all())
    return y, kv, ks


@pytest.mark.parametrize("L", [1, 15, 16, 17, 63, 64, 65, 127, 129, 640, 1000])
@pytest.mark.parametrize("split", [None, False])
def test_lengths(dev, L, split):
    check(dev, *make(L, 2, 3, L, 64), split=split)


@pytest.mark.parametrize("dv", [1, 15, 16, 17, 64, 72, 112, 300])
def test_head_dims(dev, dv):
    check(dev, *make(dv, 1, 2, 150, dv))


@pytest.mark.parametrize("B,H,L", [(1, 1, 2048), (1, 16, 1024), (4, 16, 200), (8, 16, 130), (16, 16, 70)])
def test_segments_agree_with_one_piece(dev, B, H, L):
    """From 64 wavefronts (sixteen segments) to as many as fill the GPU (none)."""
    from based_amd import ops

    q, k, v = (x.to(dev) for x in make(5, B, H, L, 64))
    a, b = ops.linear_attn_prefill(q, k, v, return_state=True), ops.linear_attn_prefill(q, k, v, return_state=True, split=False)
    for x, y in zip(a, b):
        assert rel_l2(x, y) < TOL
    assert rel_l2(ops.linear_attn_prefill(q, k, v)[0], b[0]) < TOL


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("off,pad", [(0, 0), (1, 0), (0, 3), (2, 1)])
def test_layouts(dev, dtype, off, pad):
    """Rows that start anywhere: the general form of the loads gives what the wide one gives (bf16: a head dim the bf16 kernels refuse)."""
    B, H, L, dv = 2, 3, 100, 24 if dtype == torch.bfloat16 else 64
    q, k, v = make(7, B, H, L, dv, dtype)
    wide = torch.zeros(B, L, off + H * (32 + dv) + pad, dtype=dtype, device=dev)
    views, at = [], off
    for x in (q, k, v):
        n = H * x.shape[-1]
        wide[..., at:at + n] = x.to(dev).transpose(1, 2).reshape(B, L, n)
        views.append(wide[..., at:at + n].view(B, L, H, x.shape[-1]).transpose(1, 2))
        at += n
    ref = O.linear_attn_quadratic(q.double(), k.double(), v.double())
    from based_amd import ops

    y, kv, _ = ops.linear_attn_prefill(*views, return_state=True)
    assert rel_l2(y, ref) < (TOL if dtype == torch.float32 else 3e-3)   # (one rounding to bf16: at most 2^-9, 1.7e-3 in the 2-norm)
    assert rel_l2(kv, O.linear_attn_prefill_state(k.double(), v.double())[0]) < TOL


@pytest.mark.parametrize("which", ["q", "k", "v"])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
@pytest.mark.parametrize("t", [0, 5, 70, 131])
def test_no_numbers_stay_behind_their_token(dev, which, value, t):
    """A token that is no number changes no output before it (a query: none but its own)."""
    from based_amd import ops

    q, k, v = make(9, 1, 2, 150, 32)
    clean = ops.linear_attn_prefill(q.to(dev), k.to(dev), v.to(dev))[0]
    x = {"q": q, "k": k, "v": v}
    x[which][:, :, t, 3] = value
    y = ops.linear_attn_prefill(*(x[n].to(dev) for n in "qkv"))[0]
    assert torch.equal(y[:, :, :t], clean[:, :, :t]) or rel_l2(y[:, :, :t], clean[:, :, :t]) < 2e-7
    assert not bool(torch.isfinite(y[:, :, t]).all())
    if which == "q":
        assert torch.equal(y[:, :, t + 1:], clean[:, :, t + 1:])


@pytest.mark.parametrize("split", [None, False])
@pytest.mark.parametrize("value", [float("inf"), float("-inf")])
def test_infinite_values_stay_infinite(dev, value, split):
    """Every weight is positive: behind an infinite value its channel is that infinity, also where the sum over features has no other
    sign (queries and keys above zero)."""
    from based_amd import ops

    q, k, v = make(13, 1, 2, 200, 20)
    v[:, :, 5, 3] = value
    y = ops.linear_attn_prefill(*(x.to(dev) for x in (q.abs(), k.abs(), v)), split=split)[0]
    assert bool((y[:, :, 5:, 3] == value).all())
    y[:, :, 5:, 3] = 0
    assert bool(torch.isfinite(y).all())


def test_as_many_heads_as_a_launch_takes(dev):
    """2^23 heads of two groups of channel tiles: a single token is its own output."""
    from based_amd import ops

    B, H, dv = 1 << 19, 16, 65
    q = torch.randn(B, H, 1, 16, device=dev)
    v = torch.randn(B, H, 1, dv, device=dev)
    y = ops.linear_attn_prefill(q, q, v)[0]
    for part in (slice(0, 64), slice(B // 2 - 32, B // 2 + 32), slice(B - 64, B)):
        assert rel_l2(y[part], v[part]) < TOL


def test_refused_as_before(dev):
    from based_amd import ops

    q, k, v = (x.to(dev) for x in make(1, 1, 2, 200, 64))
    with pytest.raises(ValueError, match="can be split"):
        ops.linear_attn_prefill(q, k, v, split=2)
    with pytest.raises(ValueError):
        ops.linear_attn_prefill(q, k, torch.zeros(1, 2, 200, 1040, device=dev))
