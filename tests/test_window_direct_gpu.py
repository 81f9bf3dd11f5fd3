"""Window attention over bf16 prompts of 64-channel heads (keys and values straight into LDS) and of others
against 64 bits: portions, windows and heads around tiles of 64 keys and 128 rows, either sign of the scale, and scores that climb."""
import math

import pytest
import torch

from oracle import sozilix_oracle as O

pytestmark = pytest.mark.gpu


def run(dev, q, k, v, window, scale, start, shift=0):
    from based_amd import ops

    B, L, H, d = q.shape
    G = k.shape[2]
    wide = torch.full((B, L + 3, G, 2 * d + 8 * shift), float("nan"), dtype=torch.bfloat16, device=dev)  # (rows of a wider cache)
    cache = wide[..., :2 * d] if shift == 0 else torch.as_strided(wide, (B, L + 3, G, 2 * d), (wide.stride(0), wide.stride(1), 2 * d, 1))
    out = torch.empty(B, L, H * d, dtype=torch.bfloat16, device=dev)
    for lo, hi in ((0, start), (start, L)):
        if hi > lo:
            s = slice(lo, hi)
            ops.window_attn_prefill(*(t[:, s].to(dev).flatten(2) for t in (q, k, v)), cache, H, G, window, scale, lo, out=out[:, s])
    return out.double().cpu().view(B, L, H, d)


def error(out, q, k, v, window, scale):
    ref = torch.stack([O.window_softmax(a.double(), b.double(), c.double(), scale, window) for a, b, c in zip(q, k, v)])
    return float(((out - ref).norm(dim=-1) / ref.norm(dim=-1)).max())


@pytest.mark.parametrize("H,G,L,start,window", [(1, 1, 1, 0, 1), (4, 1, 31, 0, 129), (3, 1, 43, 0, 20), (16, 4, 65, 0, 64), (16, 4, 97, 33, 33), (5, 1, 128, 0, 1),
                                                (2, 2, 129, 64, 63), (16, 2, 200, 0, 65), (16, 16, 257, 0, 129), (12, 4, 321, 100, 128), (7, 1, 130, 1, 500),
                                                (8, 8, 640, 0, 513), (2, 1, 700, 690, 129)])
@pytest.mark.parametrize("scale", [0.125, -0.3])
def test_portions_windows_and_heads(dev, H, G, L, start, window, scale):
    g = torch.Generator().manual_seed(L + window)
    q, k, v = (torch.randn(2, L, n, 64, generator=g).bfloat16() for n in (H, G, G))
    # bf16 weights and outputs: 2^-9 each, of rows whose values partly cancel
    assert error(run(dev, q, k, v, window, scale, start, L % 2), q, k, v, window, scale) < 2e-2


@pytest.mark.parametrize("step", [0.02, 0.2, 3.0, -0.2])
def test_scores_that_climb(dev, step):
    """Scores that grow (or fall) by `step` powers of two from key to key: a new largest one in every tile, or none."""
    L, window = 300, 129
    g = torch.Generator().manual_seed(1)
    q, k, v = (0.05 * torch.randn(1, L, 2, 64, generator=g) for _ in range(3))
    q[..., 0] = 1.0
    k[..., 0] = (step / 1.4426950408889634) * torch.arange(L)[None, :, None]
    q, k, v = (t.bfloat16() for t in (q, k, 20 * v))
    assert error(run(dev, q, k, v, window, 1.0, 0), q, k, v, window, 1.0) < 2e-2


@pytest.mark.parametrize("d", [48, 64, 96])
def test_weights_are_summed_in_32_bits(dev, d):
    """One key of weight one and of the only value, the others all of a weight 0.96 * 2^-8 above 0.5, of which bf16 leaves 0.5: their sum has the
    whole of it where it is of 32-bit weights.  Means over channels and tokens, of outputs rounded by 2^-9 at most."""
    L, window = 100, 129
    weight = 0.5 * (1 + 0.96 * 2.0 ** -8)
    q, k, v = (torch.zeros(1, L, 1, d, dtype=torch.bfloat16) for _ in range(3))
    q[..., 0], k[:, 0, :, 0] = 1.0, 1.0
    v[:, 0] = 1.0 + torch.rand(1, 1, d, generator=torch.Generator().manual_seed(2)).bfloat16()
    out = run(dev, q, k, v, window, -math.log(weight), 0)[0, 20:, 0]
    ref = O.window_softmax(q[0].double(), k[0].double(), v[0].double(), -math.log(weight), window)[20:, 0]
    # (with weights of 0.5 the outputs 1 / (1 + n w) are 0.9 to 1.0 of 3.7e-3 too large)
    assert abs(float((out / ref - 1).mean())) < 5e-4


@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("H,G,B,L,start,window,rot,half", [
    (16, 4, 1, 3, 0, 129, 32, True), (16, 4, 2, 64, 1, 65, 64, False), (16, 4, 1, 777, 0, 129, 32, True), (16, 4, 1, 300, 77, 130, 32, True),
    (12, 4, 3, 130, 0, 20, 8, False), (136, 1, 1, 33, 20, 64, 16, True), (16, 16, 2, 257, 0, 129, 0, False), (5, 1, 1, 140, 13, 500, 48, True),
    (16, 2, 32, 128, 0, 513, 32, True), (16, 2, 33, 128, 0, 513, 32, True), (16, 4, 3, 1024, 0, 129, 32, True), (16, 4, 7, 512, 0, 129, 32, False)])
def test_cache_that_the_attention_fills(dev, H, G, B, L, start, window, rot, half, norm):
    """Rows of the cache behind a portion, and what a second portion makes of them: written by the attention itself, or in front of it where the
    portion's own keys lie in the output's rows; both sides of the rule that tells them."""
    from based_amd import ops
    from based_amd.mixers.window_attention import _ExactRotary

    g = torch.Generator().manual_seed(L + B)
    n, d = L + start, 64
    kw = dict(rope=_ExactRotary(rot, base=100.0, interleaved=not half).tables(n, dev) if rot else None, value_norm_eps=1e-5 if norm else None)
    x = torch.randn(B, n, H * d + 2 * G * d, generator=g).bfloat16().to(dev)
    q, k, v = x[..., :H * d], x[..., H * d:(H + G) * d], x[..., (H + G) * d:]

    def run(inside):
        cache = torch.full((B, n + 2, G, 2 * d), float("nan"), dtype=torch.bfloat16, device=dev)
        room = x.clone()
        kk, vv = (room[..., H * d:(H + G) * d], room[..., (H + G) * d:]) if inside else (k, v)
        out = room[..., :H * d]
        for lo, hi in ((0, start), (start, n)):
            if hi > lo:
                s = slice(lo, hi)
                ops.window_attn_prefill(q[:, s], kk[:, s], vv[:, s], cache, H, G, window, d ** -0.5, lo, out=out[:, s], **kw)
        return out.double(), cache

    out, cache = run(False)
    ref, rows = run(True)
    # a rotation's two products and a norm's sum are added in one order or the other: now and then the other of two neighbours in bf16
    assert float((cache[:, :n].double() - rows[:, :n].double()).norm() / rows[:, :n].double().norm()) < 2 ** -12
    assert cache[:, n:].isnan().all() and rows[:, n:].isnan().all()
    assert float((out - ref).norm() / ref.norm()) < 2 ** -10
    want = v.view(B, n, G, d).double()
    if norm:
        want = want / (want.square().mean(-1, keepdim=True) + 1e-5).sqrt()
    # eight significant bits: an element is rounded by at most 2^-8 of itself
    assert float(((cache[:, :n, :, d:].double() - want).norm(dim=-1) / want.norm(dim=-1)).max()) < 2 ** -8


@pytest.mark.parametrize("H,G,B,L,window,rot,half,norm", [
    (16, 16, 28, 52, 129, 64, False, True), (16, 4, 32, 64, 129, 64, False, False), (16, 16, 28, 52, 129, 64, True, True), (16, 4, 3, 200, 65, 32, True, False)])
def test_keys_are_turned_to_the_same_numbers(dev, H, G, B, L, window, rot, half, norm):
    """Cache and outputs of a portion whose keys and values the attention leaves in the cache, and of the same one with a launch for that in front."""
    from based_amd import ops
    from based_amd.mixers.window_attention import _ExactRotary

    d, g = 64, torch.Generator().manual_seed(L)
    kw = dict(rope=_ExactRotary(rot, base=100.0, interleaved=not half).tables(L, dev), value_norm_eps=1e-5 if norm else None)
    x = torch.randn(B, L, H * d + 2 * G * d, generator=g).bfloat16().to(dev)
    got = []
    for inside in (False, True):  # (a launch where keys and values lie in the output's rows)
        cache, room = torch.zeros(B, L, G, 2 * d, dtype=torch.bfloat16, device=dev), x.clone()
        own = room if inside else x
        k, v = own[..., H * d:(H + G) * d], own[..., (H + G) * d:]
        ops.window_attn_prefill(x[..., :H * d], k, v, cache, H, G, window, d ** -0.5, 0, out=room[..., :H * d], **kw)
        got.append((room[..., :H * d].clone(), cache))
    assert torch.equal(got[0][1], got[1][1]) and bool(got[0][1].any())
    assert torch.equal(got[0][0], got[1][0])
